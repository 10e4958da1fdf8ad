"""Lines frames of more lines, vertices and pixels than one launch takes threads
for (2^32): on the CPU, the launches that euc_amd/csrc/internal.hpp makes of them
cover every line and vertex once; on the GPU, 2^28 lines and more against the
oracle."""
import os
import subprocess

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, DepthMode, PipelineDesc, Primitives, Shader, Xform
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "internal.hpp"
using namespace euchip;
static int check(uint64_t lines, uint64_t vertices) {
    uint64_t next = 0, shaded = 0;
    int bad = 0, launches = 0;
    line_launches((uint32_t)lines, vertices, [&](const LineLaunch &l) {
        const uint64_t groups = (uint64_t)l.line_groups + l.vertex_groups;
        if (groups == 0 || groups * 256 >= 1ull << 32) bad++;
        if (l.line_groups && l.first != next) bad++;
        next += (uint64_t)l.line_groups * kLinesPerBlock;
        if (l.vertex_groups && shaded) bad++;
        shaded += (uint64_t)l.vertex_groups * 256;
        launches++;
    });
    if (next < lines || next >= lines + kLinesPerBlock || shaded < vertices || shaded >= vertices + 256) bad++;
    if (lines <= 1u << 27 && vertices < 1ull << 31 && launches != 1) bad++;
    if (bad) printf("%llu lines, %llu vertices\n", (unsigned long long)lines, (unsigned long long)vertices);
    return bad;
}
int main() {
    int bad = 0;
    for (int b = 0; b < 31; b++)
        for (int64_t e = -17; e <= 17; e++)
            for (int c = 0; c < 33; c++)
                for (int64_t f = -257; f <= 257; f += 257) {
                    const int64_t n = (1ll << b) + e, v = c == 0 ? 0 : (1ll << (c - 1)) + f;
                    if (n >= 1 && n < 1ll << 31 && v >= 0 && v < (1ll << 32) - 256) bad += check(n, v);
                }
    bad += check((1u << 31) - 1u, (1ull << 32) - 257u);
    for (uint64_t n : {1ull, 255ull, 256ull, 257ull, (1ull << 31) - 1, 1ull << 31, (1ull << 31) + 1, 1ull << 33, (3ull << 32) + 5}) {
        uint64_t done = 0;  // a fill's parts
        for (uint64_t m = n; m;) {
            const uint64_t g = launch_groups(m, 256), part = m < g * 256 ? m : g * 256;
            if (g * 256 >= 1ull << 32 || !part) { bad++; break; }
            done += part, m -= part;
        }
        bad += done != n;
    }
    return bad != 0;
}
"""


def test_launches(tmp_path):
    src, exe = tmp_path / "launches.cpp", tmp_path / "launches"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                           os.path.join(ROOT, "euc_amd", "csrc"), str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:500]


@pytest.mark.gpu
@pytest.mark.parametrize("instances,shader", [(511, Shader.FLAT), (512, Shader.COLOR), (513, Shader.FLAT)])
def test_many_lines(instances, shader):
    """Instances of 2^19 lines each, all in the same place: the target is that of one instance."""
    from euc_amd.renderer import Context
    w, h, n = 640, 480, 1 << 19
    rng = np.random.default_rng(instances)
    pos = np.ones((2048, 2, 4), np.float32)
    pos[:, 0, :2] = rng.uniform(-1.0, 1.0, (2048, 2))
    pos[:, 1, :2] = pos[:, 0, :2] + rng.normal(0.0, 0.2, (2048, 2))
    pos[:, :, 2] = rng.uniform(0.0, 1.0, (2048, 2))
    pos[300:, :, :2] += np.float32(4.0)  # most lines miss the target
    idx = np.arange(2 * n, dtype=np.uint32)
    idx[600:] = 600 + idx[600:] % (4096 - 600)
    kind = {"rgba8": rng.integers(0, 2 ** 32, 4096, dtype=np.uint64).astype(np.uint32)} if shader == Shader.FLAT else \
        {"col": rng.uniform(0.0, 1.0, (4096, 4)).astype(np.float32)}

    def mesh(k):
        return S.Mesh(pos=pos.reshape(-1, 4), idx=idx, count=2 * n, n_instances=k, **kind)
    d = PipelineDesc.make(shader, Xform.CLIP, depth_mode=DepthMode.LESS_WRITE, band_policy=BandPolicy.SEQ,
                          primitives=Primitives.LINE_LIST)
    oc, od = np.full((h, w), 9, np.uint32), np.full((h, w), 1.0, np.float32)
    rc, frags = O.render(d, S.uniforms(), mesh(1), oc, od)
    assert rc == 0 and frags > 1000
    ctx = Context(0)
    try:
        gm, c, z = ctx.mesh(mesh(instances)), ctx.color_target(w, h), ctx.depth_target(w, h)
        for _ in range(2):
            ctx.render(d, S.uniforms(), gm, c, z, clear_color=9, clear_depth=1.0)
            assert np.array_equal(c.download(), oc)
            assert np.array_equal(z.download().view(np.uint32), od.view(np.uint32))
    finally:
        ctx.close()
