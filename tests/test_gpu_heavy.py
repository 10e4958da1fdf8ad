"""Which workgroup takes which tile: frames whose heavy tiles (128 entries and
more) are none, some, all of the tiles, or more than the launch has workgroups,
and big-triangle frames without row checkpoints that have heavy tiles as well.
Every frame equals the oracle's, bit-exact."""
import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, CullMode, DepthMode, PipelineDesc, Shader, Xform
from tests.parity import assert_bit_exact, run_pair

pytestmark = pytest.mark.gpu

DESC = PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.NONE,
                         band_policy=BandPolicy.SEQ)


def scattered(seed, n, extent, size, n_large=0):
    """n triangles of clip-space `size` spread evenly over [-extent, extent]^2, then n_large ones over the whole target."""
    rng = np.random.default_rng(seed)
    pos = np.empty((n + n_large, 3, 4), np.float32)
    pos[:n, :, :2] = rng.uniform(-extent, extent, (n, 1, 2)) + rng.uniform(-size, size, (n, 3, 2))
    pos[n:, :, :2] = rng.uniform(-1.0, 1.0, (n_large, 3, 2))
    pos[:, :, 2] = rng.uniform(0.05, 0.95, (n + n_large, 1))
    pos[:, :, 3] = 1.0
    rgba8 = rng.integers(0, 2 ** 32, 3 * (n + n_large), dtype=np.uint64).astype(np.uint32)
    return S.Mesh(pos=pos.reshape(-1, 4), count=3 * (n + n_large), rgba8=rgba8)


@pytest.mark.parametrize("w,h,n,extent,size,n_large", [
    (33, 9, 3000, 1.0, 0.2, 0),            # 4 tiles, all heavy, 8 workgroups
    (250, 190, 6000, 0.3, 0.02, 0),        # some heavy
    (640, 480, 3000, 1.0, 0.004, 0),       # none heavy, some empty
    (1024, 800, 600000, 1.0, 0.004, 0),    # 3200 tiles, most heavy: more than the workgroups
    (3000, 1800, 20000, 1.0, 0.01, 0),     # 21,150 tiles: several per workgroup
    (2048, 2048, 1000, 0.01, 0.01, 8),     # big-triangle frame without checkpoints, a few heavy tiles
])
def test_heavy_tiles(gpu_ctx, w, h, n, extent, size, n_large):
    mesh = scattered(w + n, n, extent, size, n_large)
    gm = gpu_ctx.mesh(mesh)
    for rep in range(2):  # the second frame takes the counters that the first one left
        r = run_pair(gpu_ctx, DESC, S.uniforms(), mesh, w, h, color_init=3 + rep, gmesh=gm)
        assert r["frags"] > 100
        assert_bit_exact(r, f"{w}x{h}, {n} + {n_large} triangles, frame {rep}")
