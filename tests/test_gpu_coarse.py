"""Coarse shading's shared samples (pipeline.rs:541-570): pixels of a 2 x 2 block
take their four samples together where one triangle won them.  Bands of odd
heights (blocks cut by a band or by a tile's first row), odd target sizes, every
tile shape, triangles of less than a pixel up to the whole target.  Every frame
equals the oracle's, bit-exact."""
import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import AaMode, BandPolicy, CullMode, DepthMode, PipelineDesc, Shader, Xform
from euc_amd.renderer import Request
from tests.parity import assert_bit_exact, assert_same, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,nu,level,band", [
    (1013, 161, 60, 1, BandPolicy.PAR),   # bands of 39 rows
    (1013, 161, 9, 1, BandPolicy.SEQ),
    (611, 333, 200, 1, BandPolicy.PAR),   # triangles of about a pixel
    (1777, 99, 24, 2, BandPolicy.PAR),    # bands of 45 rows, cells of 4 x 4
    (333, 250, 40, 6, BandPolicy.SEQ),    # one cell per tile
    (33, 9, 16, 1, BandPolicy.SEQ),
])
@pytest.mark.parametrize("shader", [Shader.PHONG, Shader.GOURAUD, Shader.FLAT])
def test_shared_samples(gpu_ctx, w, h, nu, level, band, shader):
    sc = S.torus_scene(0xC0A + nu, w, h, nu, max(3, nu // 2), 4)
    m = sc.mesh
    m.rgba8 = np.arange(1, m.n_vertices + 1, dtype=np.uint32) * np.uint32(2654435761)
    d = PipelineDesc.make(shader, Xform.MVP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.NONE,
                          aa_mode=AaMode.Msaa(level), band_policy=band, threads=64)
    r = run_pair(gpu_ctx, d, sc.uniforms, m, w, h, color_init=5)
    assert r["frags"] > 20
    assert_bit_exact(r, f"{w}x{h} level {level}")
    c, z = gpu_ctx.color_target(w, h), gpu_ctx.depth_target(w, h)
    b = gpu_ctx.batch().set(d, [Request(gpu_ctx.mesh(m), c, z, sc.uniforms)], clear_color=5, clear_depth=1.0)
    for tile_w in (8, 16, 32):
        b.set_tile_width(tile_w)
        b.run()
        assert_same(c.download(), z.download(), r["o_color"], r["o_depth"], f"{w}x{h} level {level} tile {tile_w}")
    b.close()
