"""Setup's binning: the (tile, triangle) pairs of a workgroup spread over its
lanes in rounds of 1024.  Frames whose workgroups have no pair, one round, many
rounds, more distinct tiles than the hash table holds and triangles of more
tiles than a round takes, with meshes around the workgroup sizes (64 and 256
triangles).  Every frame equals the oracle's, bit-exact."""
import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, CullMode, DepthMode, PipelineDesc, Shader, Xform
from euc_amd.renderer import Request
from tests.parity import assert_bit_exact, assert_same, run_pair

pytestmark = pytest.mark.gpu

DESC = PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.NONE,
                         band_policy=BandPolicy.SEQ)


def triangles(seed, groups):
    """groups: (count, size) of triangles scattered over the target, mixed in a seeded order."""
    rng = np.random.default_rng(seed)
    n = sum(c for c, _ in groups)
    size = np.concatenate([np.full(c, s) for c, s in groups])[rng.permutation(n)]
    pos = np.empty((n, 3, 4), np.float32)
    pos[:, :, :2] = rng.uniform(-1.0, 1.0, (n, 1, 2)) + rng.uniform(-1.0, 1.0, (n, 3, 2)) * size[:, None, None]
    pos[:, :, 2] = rng.uniform(0.05, 0.95, (n, 3))
    pos[:, :, 3] = 1.0
    rgba8 = rng.integers(0, 2 ** 32, 3 * n, dtype=np.uint64).astype(np.uint32)
    return S.Mesh(pos=pos.reshape(-1, 4), count=3 * n, rgba8=rgba8)


@pytest.mark.parametrize("w,h,groups", [
    (64, 16, [(63, 0.5)]), (64, 16, [(64, 0.5)]), (64, 16, [(65, 0.5)]),   # 4 tiles
    (200, 90, [(257, 0.3)]),                    # a workgroup and a triangle, one round each
    (640, 480, [(1500, 0.3)]),                  # dozens of tiles per triangle: several rounds
    (1280, 720, [(4000, 0.02), (300, 0.9)]),    # small and large mixed
    (64, 64, [(32768, 0.1)]), (64, 64, [(32769, 0.1)]),  # the limit of the small workgroups
    (2048, 2048, [(17000, 0.004), (3, 3.0)]),   # triangles of thousands of tiles among tiny ones
    (3000, 40, [(6000, 0.05), (40, 2.0)]),      # wide: nearly all tiles in a row
])
def test_pair_rounds(gpu_ctx, w, h, groups):
    mesh = triangles(w + h, groups)
    assert mesh.n_triangles > ((w + 31) // 32) * ((h + 7) // 8)  # binned, not the big-triangle mode
    r = run_pair(gpu_ctx, DESC, S.uniforms(), mesh, w, h, color_init=9)
    assert r["frags"] > 100
    assert_bit_exact(r, f"{w}x{h} {groups}")
    c, d = gpu_ctx.color_target(w, h), gpu_ctx.depth_target(w, h)
    b = gpu_ctx.batch().set(DESC, [Request(gpu_ctx.mesh(mesh), c, d, S.uniforms())], clear_color=9, clear_depth=1.0)
    for tile_w in (8, 32):
        b.set_tile_width(tile_w)
        b.run()
        assert_same(c.download(), d.download(), r["o_color"], r["o_depth"], f"batch {w}x{h} tile {tile_w}")
    b.close()
