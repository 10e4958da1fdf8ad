"""Frames with more heavy tiles than workgroups of their own for them: meshes of
more triangles than tiles (binned frames) whose triangles are large, so that nearly
every tile is heavy.  The frame equals the oracle's, and takes no longer than the
same request as a batch of one, which has no pass of heavy tiles, by a factor that
lies far from both sides (0.5 to 0.8 of it; 2.4 to 5.4 with all tiles left to a few
workgroups)."""
import time

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, CullMode, DepthMode, PipelineDesc, Shader, Xform
from euc_amd.renderer import Request
from tests.parity import assert_bit_exact, run_pair

pytestmark = pytest.mark.gpu

DESC = PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.NONE,
                         band_policy=BandPolicy.SEQ)


def large(seed, n, half):
    rng = np.random.default_rng(seed)
    pos = np.ones((n, 3, 4), np.float32)
    pos[:, :, :2] = rng.uniform(-0.8, 0.8, (n, 1, 2)) + rng.uniform(-half, half, (n, 3, 2))
    pos[:, :, 2] = rng.uniform(0.0, 1.0, (n, 3))
    rgba8 = rng.integers(0, 2 ** 32, 3 * n, dtype=np.uint64).astype(np.uint32)
    return S.Mesh(pos=pos.reshape(-1, 4), count=3 * n, rgba8=rgba8)


@pytest.mark.parametrize("w,h,n,half", [(640, 480, 3000, 0.6), (333, 211, 1500, 0.5), (1024, 1024, 6000, 0.2)])
def test_more_heavy_tiles_than_workgroups(gpu_ctx, w, h, n, half):
    mesh = large(n, n, half)
    gm = gpu_ctx.mesh(mesh)
    for rep in range(2):
        r = run_pair(gpu_ctx, DESC, S.uniforms(), mesh, w, h, color_init=rep, gmesh=gm)
        assert_bit_exact(r, f"{w}x{h}, frame {rep}")
    assert r["frags"] > 10 ** 5
    c, z = gpu_ctx.color_target(w, h), gpu_ctx.depth_target(w, h)
    b = gpu_ctx.batch().set(DESC, [Request(gm, c, z, S.uniforms())], clear_color=0, clear_depth=1.0)

    def batch():
        b.launch()
        b.wait()

    def best(f):
        times = []
        for _ in range(8):
            t = time.perf_counter()
            f()
            times.append(time.perf_counter() - t)
        return min(times)

    frame = best(lambda: gpu_ctx.render(DESC, S.uniforms(), gm, c, z, clear_color=0, clear_depth=1.0))
    whole = best(batch)
    print(f"frame {frame * 1e6:.0f} us, batch of one {whole * 1e6:.0f} us")
    assert frame < 1.6 * whole
    b.close()


def heavy_tiles(mesh, w, h):
    """Tiles (32 x 8) that 128 triangles and more reach by their bounding boxes."""
    px = (mesh.pos.reshape(-1, 3, 4)[:, :, :2].astype(np.float64) * [0.5, -0.5] + 0.5) * [w, h]
    lo, hi = np.clip(np.floor(px.min(1)), 0, [w, h]).astype(int), np.clip(np.floor(px.max(1) + 1), 0, [w, h]).astype(int)
    n = np.zeros((-(-h // 8), -(-w // 32)), int)
    for (x0, y0), (x1, y1) in zip(lo, hi):
        if x0 < x1 and y0 < y1:
            n[y0 // 8:(y1 - 1) // 8 + 1, x0 // 32:(x1 - 1) // 32 + 1] += 1
    return int((n >= 128).sum())


@pytest.mark.parametrize("w,h,n,region,kind", [
    (640, 480, 8000, (0.30, 0.12), "own"),         # a workgroup for each heavy tile
    (1280, 960, 8000, (0.22, 0.10), "two"),        # up to two for a workgroup
    (3000, 1800, 24000, (0.19, 0.08), "two"),      # and more tiles than workgroups
    (320, 240, 8000, (0.90, 0.40), "busy"),        # more than an eighth of the tiles
    (1280, 960, 60000, (0.45, 0.35), "busy"),      # more than an eighth, and than the workgroups
])
def test_who_takes_heavy_tiles(gpu_ctx, w, h, n, region, kind):
    rng = np.random.default_rng(n + w)
    pos = np.ones((n, 3, 4), np.float32)
    size = np.array([12.0 / w, 12.0 / h])  # 6 pixels each way: none is dropped as too small
    pos[:, :, :2] = rng.uniform(-1.0, 1.0, (n, 1, 2)) * region + rng.uniform(-1.0, 1.0, (n, 3, 2)) * size
    pos[:, :, 2] = rng.uniform(0.05, 0.95, (n, 1))
    mesh = S.Mesh(pos=pos.reshape(-1, 4), count=3 * n, rgba8=rng.integers(0, 2 ** 32, 3 * n, dtype=np.uint64).astype(np.uint32))
    groups, tiles, heavy = min(512, n // 128 // 8 * 8 + 8), -(-w // 32) * -(-h // 8), heavy_tiles(mesh, w, h)
    assert n > tiles or kind == "two"
    assert kind == ("own" if heavy <= groups else "two" if heavy <= min(2 * groups, tiles // 8) else "busy"), (heavy, groups, tiles)
    gm = gpu_ctx.mesh(mesh)
    for rep in range(2):
        r = run_pair(gpu_ctx, DESC, S.uniforms(), mesh, w, h, color_init=rep, gmesh=gm)
        assert_bit_exact(r, f"{kind}, frame {rep}")
    assert r["frags"] > 1000


@pytest.mark.parametrize("region,kind", [((0.30, 0.06), "busy"), ((0.16, 0.045), "two"), ((0.06, 0.03), "own")])
def test_big_triangle_frames(gpu_ctx, region, kind):
    """The same where a frame also has large triangles that are on no tile's list (no row checkpoints)."""
    w = h = 2048
    n, n_large = 16000, 6
    rng = np.random.default_rng(6)
    pos = np.ones((n + n_large, 3, 4), np.float32)
    pos[:n, :, :2] = rng.uniform(-1.0, 1.0, (n, 1, 2)) * region + rng.uniform(-1.0, 1.0, (n, 3, 2)) * [0.016, 0.012]
    pos[n:, :, :2] = rng.uniform(-1.0, 1.0, (n_large, 3, 2))
    pos[:, :, 2] = rng.uniform(0.05, 0.95, (n + n_large, 1))
    mesh = S.Mesh(pos=pos.reshape(-1, 4), count=3 * (n + n_large),
                  rgba8=rng.integers(0, 2 ** 32, 3 * (n + n_large), dtype=np.uint64).astype(np.uint32))
    small = S.Mesh(pos=pos[:n].reshape(-1, 4), count=3 * n)
    groups, tiles, heavy = n // 128 // 8 * 8 + 8, 64 * 256, heavy_tiles(small, w, h)
    assert n + n_large <= tiles and tiles * n > 8 << 20  # big-triangle mode, without checkpoints
    assert kind == ("own" if heavy <= groups else "two" if heavy <= 2 * groups else "busy"), (heavy, groups)
    gm = gpu_ctx.mesh(mesh)
    for rep in range(2):
        r = run_pair(gpu_ctx, DESC, S.uniforms(), mesh, w, h, color_init=rep, gmesh=gm)
        assert_bit_exact(r, f"{kind}, frame {rep}")
    assert r["frags"] > 10000
