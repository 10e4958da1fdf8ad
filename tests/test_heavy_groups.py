"""The workgroups of a frame that take its heavy tiles (euc_amd/csrc/internal.hpp,
heavy_group_count) each read a place of the heavy-tile list at once: on the CPU,
for list sizes around the multiples of 8 and the smallest ones and for triangle
counts on both sides of each, never more workgroups than places; on the GPU, a
list that is nearly full, against the oracle."""
import os
import subprocess

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, CullMode, DepthMode, PipelineDesc, Shader, Xform
from tests.parity import assert_bit_exact, run_pair

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "internal.hpp"
int main() {
    int bad = 0;
    for (uint64_t cap = 0; cap < 0xFFFFFFF0ull; cap += cap < 1100 ? 1 : cap)
        for (uint64_t tris = 1; tris < 1ull << 32; tris += tris < 70000 ? 61 : tris) {
            const uint32_t g = euchip::heavy_group_count((uint32_t)cap, (uint32_t)tris);
            if (g <= cap && g % 8u == 0u && g <= 512u && (g >= 8u || cap < 8u)) continue;
            if (!bad++) printf("%llu places, %llu triangles: %u\n", (unsigned long long)cap, (unsigned long long)tris, g);
        }
    return bad != 0;
}
"""


def test_heavy_group_count(tmp_path):
    src, exe = tmp_path / "groups.cpp", tmp_path / "groups"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                           os.path.join(ROOT, "euc_amd", "csrc"), str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:500]


@pytest.mark.gpu
def test_full_list():
    """A context's first frame: 256 places for the heavy tiles, 247 tiles that nearly all
    are heavy, triangles for more workgroups than places."""
    from euc_amd.renderer import Context
    rng = np.random.default_rng(5)
    n = 60000
    pos = np.ones((n, 3, 4), np.float32)
    pos[:, :, :2] = rng.uniform(-1.0, 1.0, (n, 1, 2)) + rng.uniform(-0.02, 0.02, (n, 3, 2))
    pos[:, :, 2] = rng.uniform(0.05, 0.95, (n, 1))
    mesh = S.Mesh(pos=pos.reshape(-1, 4), count=3 * n, rgba8=rng.integers(0, 2 ** 32, 3 * n, dtype=np.uint64).astype(np.uint32))
    d = PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.NONE,
                          band_policy=BandPolicy.SEQ)
    ctx = Context(0)
    try:
        for frame in range(2):
            r = run_pair(ctx, d, S.uniforms(), mesh, 13 * 32, 19 * 8, color_init=frame)
            assert r["frags"] > 50000
            assert_bit_exact(r, f"frame {frame}")
    finally:
        ctx.close()
