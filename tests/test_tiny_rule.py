"""Which frames of few triangles take one launch (euc_amd/csrc/internal.hpp,
tiny_frame): on the CPU, its answers where both sides were measured, at sizes whose
products pass 64 bits, and that fewer triangles or a smaller target never refuse
what more admit; on the GPU, frames on both sides of the line and of tall targets,
bit-exact, each on the side that the rule says."""
import os
import subprocess

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import AaMode, BandPolicy, CullMode, DepthMode, PipelineDesc, Shader, Xform
from tests.parity import assert_bit_exact, run_pair

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include "internal.hpp"
int main(int argc, char **argv) {
    for (int i = 1; i + 2 < argc; i += 3)
        printf("%d", (int)euchip::tiny_frame(strtoull(argv[i], 0, 10), strtoul(argv[i + 1], 0, 10), strtoul(argv[i + 2], 0, 10)));
    printf("\n");
}
"""

# (triangles, columns, rows): one launch at least as fast with the triangles filling
# the target and well faster with them filling a part of it, or slower by far
FASTER = [(64, 64, 64), (64, 160, 90), (32, 320, 180), (64, 320, 180), (12, 800, 600), (24, 960, 540), (12, 1280, 720),
          (12, 1600, 1200), (2, 1600, 900), (2, 1920, 1080), (4, 1600, 900), (2, 1000, 1000)]
SLOWER = [(65, 64, 64), (64, 480, 1440), (64, 640, 1920), (64, 960, 540), (32, 960, 2880), (12, 1280, 3840), (12, 1600, 4800),
          (24, 1600, 900), (2, 3840, 2160), (1, 3840, 3840), (64, 3840, 3840), (12, 1920, 1920)]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    src, exe = d / "rule.cpp", d / "rule"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                           os.path.join(ROOT, "euc_amd", "csrc"), str(src), "-o", str(exe)])

    def ask(frames):
        r = subprocess.run([str(exe), *[str(x) for f in frames for x in f]], capture_output=True, text=True, check=True)
        return [c == "1" for c in r.stdout.strip()]
    return ask


def test_measured(rule):
    assert rule(FASTER) == [True] * len(FASTER)
    assert rule(SLOWER) == [False] * len(SLOWER)


def test_largest_sizes(rule):
    big = (1 << 24) - 1
    assert rule([(n, w, h) for n in (1, 64) for w, h in [(big, 1), (big, big), (1 << 20, 1 << 20), (3000, big)]]) == [False] * 8


def test_monotone(rule):
    sizes = [1, 7, 64, 300, 640, 1000, 1600, 2000, 2560, 4000, 9000]
    for n in (1, 2, 12, 32, 33, 64):
        grid = np.array(rule([(n, w, h) for w in sizes for h in sizes])).reshape(len(sizes), -1)
        assert not (grid[1:] & ~grid[:-1]).any() and not (grid[:, 1:] & ~grid[:, :-1]).any()
        more = np.array(rule([(n + 1, w, h) for w in sizes for h in sizes])).reshape(grid.shape)
        assert not (more & ~grid).any()


def soup(seed, n):
    rng = np.random.default_rng(seed)
    pos = np.empty((3 * n, 4), np.float32)
    pos[:, :2] = rng.uniform(-1.3, 1.3, (3 * n, 2))
    pos[:, 2] = rng.uniform(-0.1, 1.1, 3 * n)
    pos[:, 3] = rng.uniform(0.6, 1.4, 3 * n)
    return S.Mesh(pos=pos, count=3 * n, rgba8=rng.integers(0, 2 ** 32, 3 * n, dtype=np.uint64).astype(np.uint32),
                  col=rng.uniform(0.0, 1.0, (3 * n, 4)).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("n,w,h", [(64, 96, 12000), (3, 7, 9001), (32, 640, 900), (33, 640, 640), (64, 640, 573), (64, 640, 574),
                                   (12, 1600, 1233), (12, 1600, 1234), (1, 2048, 1573), (2, 2049, 100), (2, 1999, 40)])
@pytest.mark.parametrize("dm,aa", [(DepthMode.LESS_WRITE, 0), (DepthMode.NONE, 1), (DepthMode.GREATER_PASS, 0)])
def test_both_sides(rule, n, w, h, dm, aa):
    from euc_amd.renderer import Context
    d = PipelineDesc.make(Shader.COLOR if aa else Shader.FLAT, Xform.CLIP, depth_mode=dm, cull=CullMode.NONE,
                          aa_mode=AaMode.Msaa(aa) if aa else AaMode.NONE, band_policy=BandPolicy.SEQ)
    ctx = Context(0)
    try:
        ctx.set_profiling(True)
        r = run_pair(ctx, d, S.uniforms(), soup(w + n, n), w, h, color_init=2, depth_init=0.5)
        assert_bit_exact(r, f"{n} triangles, {w}x{h}")
        assert set(ctx.kernel_stats()) == ({"tiny"} if rule([(n, w, h)])[0] else {"setup", "raster"})
    finally:
        ctx.close()
