"""Frames of few triangles (one launch, everything in LDS) against the oracle,
bit-exact, on both sides of the rule that picks them: every shader, sampler
wrapping, depth mode, MSAA level, geometry stage, band policy, loaded and cleared
targets, instances with a trailing partial triangle, clip coordinates with w <= 0
and non-finite ones, one triangle up to the limit and past it."""
import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import (AaMode, BandPolicy, CoordinateMode, CullMode, DepthMode, Geometry, PipelineDesc,
                              PixelFormat, Sampler, Shader, Xform)
from tests.parity import assert_bit_exact, run_pair

pytestmark = pytest.mark.gpu

DEPTHS = [DepthMode.LESS_WRITE, DepthMode.GREATER_WRITE, DepthMode.NONE, DepthMode.LESS_PASS, DepthMode(2, True)]


def cube(instances=1):
    pos, nrm, idx = S.box(1)
    uv = (pos[:, :2] * 1.5 + 0.2).astype(np.float32)
    col = np.abs(np.concatenate([pos, np.ones_like(pos[:, :1])], 1)).astype(np.float32)
    models = np.stack([S.f32(S.translation(0.9 * i - 0.6, 0.3 * i, 3.0 + 0.4 * i) @ S.rotation(0.5 + i, 0.8, 0.2)).reshape(16)
                       for i in range(instances)])
    rgba8 = np.arange(1, len(pos) + 1, dtype=np.uint32) * np.uint32(0x9E3779B1)
    return S.Mesh(pos=pos, nrm=nrm, uv=uv, col=col, rgba8=rgba8, idx=idx, count=int(idx.size), n_instances=instances,
                  models=models)


@pytest.mark.parametrize("shader", list(Shader))
@pytest.mark.parametrize("k", range(5))
def test_cube(gpu_ctx, shader, k):
    w, h = [(161, 97), (640, 480), (33, 9), (999, 300), (320, 240)][k]
    rng = np.random.default_rng(k)
    lvp = S.f32(S.perspective_fov_lh_zo(0.9, 64, 64, 0.1, 50.0) @ S.look_at_lh((3, 4, -2), (0, 0, 3), (0, 1, 0)))
    u = S.uniforms(view_proj=S.f32(S.perspective_fov_lh_zo(1.2, w, h, 0.1, 50.0)), light_pos=(3, 4, -2), light_vp=lvp)
    d = PipelineDesc.make(shader, Xform.MVP, depth_mode=DEPTHS[k], cull=[CullMode.BACK, CullMode.NONE, CullMode.FRONT][k % 3],
                          aa_mode=AaMode.Msaa(k) if k > 1 else AaMode.NONE, band_policy=BandPolicy(k % 2),
                          geometry=[Geometry.IDENTITY, Geometry.REVERSED, Geometry.BOTH_SIDES][k % 3],
                          sampler=list(Sampler)[(2 * k + int(shader)) % 9], pixel_format=PixelFormat(k % 2), threads=64)
    tex = rng.integers(0, 2 ** 32, (19, 23), dtype=np.uint64).astype(np.uint32)
    sh = rng.uniform(0.5, 1.0, (40, 30)).astype(np.float32)
    loaded = k in (1, 3)
    r = run_pair(gpu_ctx, d, u, cube(1 + k % 3), w, h, texture=tex, shadow=sh,
                 color_init=rng.integers(0, 2 ** 32, (h, w), dtype=np.uint64).astype(np.uint32) if loaded else 11,
                 depth_init=rng.uniform(0.9, 1.0, (h, w)).astype(np.float32) if loaded else [1.0, 1.0, 0.5, 1.0, 0.98][k])
    assert_bit_exact(r, f"{shader} {k}")


def soup(seed, n, special=False):
    rng = np.random.default_rng(seed)
    pos = np.empty((3 * n, 4), np.float32)
    pos[:, :2] = rng.uniform(-1.5, 1.5, (3 * n, 2))
    pos[:, 2] = rng.uniform(-0.2, 1.2, 3 * n)
    pos[:, 3] = rng.uniform(0.5, 1.5, 3 * n)
    if special:
        pos[rng.random(3 * n) < 0.1, 3] = -0.7
        pos[rng.random(3 * n) < 0.05, 3] = 0.0
        pos[rng.random(3 * n) < 0.05, 0] = np.nan
        pos[rng.random(3 * n) < 0.05, 1] = np.inf
        pos[rng.random(3 * n) < 0.05, 2] = np.nan
    rgba8 = rng.integers(0, 2 ** 32, 3 * n, dtype=np.uint64).astype(np.uint32)
    return S.Mesh(pos=pos, count=3 * n, rgba8=rgba8)


@pytest.mark.parametrize("w,h,n", [(640, 480, 1), (640, 480, 63), (640, 480, 64), (640, 480, 65), (1600, 40, 12),
                                   (1601, 40, 2), (1600, 300, 13), (31, 7, 64), (1283, 771, 7)])
@pytest.mark.parametrize("special", [False, True])
def test_limits(gpu_ctx, w, h, n, special):
    mesh = soup(w + n, n, special)
    for dm in DEPTHS:
        d = PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=dm, cull=CullMode.NONE, band_policy=BandPolicy.SEQ,
                              coordinate_mode=CoordinateMode.OPENGL if special else CoordinateMode.VULKAN)
        r = run_pair(gpu_ctx, d, S.uniforms(), mesh, w, h, color_init=2, depth_init=0.6)
        assert_bit_exact(r, f"{w}x{h} {n} {dm}")


def test_partial_triangles_and_async(gpu_ctx):
    """count % 3 = 1: triangles straddle instances; tiny and binned frames alternate without a wait."""
    m = cube(3)
    m.count = 35
    u = S.uniforms(view_proj=S.f32(S.perspective_fov_lh_zo(1.2, 300, 200, 0.1, 50.0)))
    d = PipelineDesc.make(Shader.PHONG, Xform.MVP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.NONE, band_policy=BandPolicy.SEQ)
    r = run_pair(gpu_ctx, d, u, m, 300, 200, color_init=3)
    assert r["frags"] > 1000
    assert_bit_exact(r, "partial triangles")
    sc = S.torus_scene(5, 300, 200, 60, 30, 2)
    rt = run_pair(gpu_ctx, d, sc.uniforms, sc.mesh, 300, 200, color_init=3)
    assert_bit_exact(rt, "torus")
    gm, gt = gpu_ctx.mesh(m), gpu_ctx.mesh(sc.mesh)
    outs = []
    for k in range(9):
        c, z = gpu_ctx.color_target(300, 200), gpu_ctx.depth_target(300, 200)
        gpu_ctx.render(d, sc.uniforms if k % 3 else u, gt if k % 3 else gm, c, z, clear_color=3, clear_depth=1.0, sync=False)
        outs.append((c, z, rt if k % 3 else r))
    gpu_ctx.synchronize()
    for k, (c, z, want) in enumerate(outs):
        assert np.array_equal(c.download(), want["o_color"]), k
        assert np.array_equal(z.download().view(np.uint32), want["o_depth"].view(np.uint32)), k


def test_budget_refuses_as_before():
    """A budget that cannot hold the scratch of a binned frame refuses a frame of few triangles too."""
    from euc_amd._lib import EuchipError
    from euc_amd.renderer import Context
    ctx = Context(0)
    try:
        m = cube()
        u = S.uniforms(view_proj=S.f32(S.perspective_fov_lh_zo(1.2, 160, 90, 0.1, 50.0)))
        d = PipelineDesc.make(Shader.PHONG, Xform.MVP, depth_mode=DepthMode.LESS_WRITE, cull=CullMode.BACK,
                              band_policy=BandPolicy.SEQ)
        gm, c, z = ctx.mesh(m), ctx.color_target(160, 90), ctx.depth_target(160, 90)
        ctx.set_budget(ctx.bytes_in_use())
        with pytest.raises(EuchipError) as e:
            ctx.render(d, u, gm, c, z, clear_color=3, clear_depth=1.0)
        assert e.value.name == "OVER_BUDGET"
        ctx.set_budget(ctx.bytes_in_use() + (1 << 30))
        r = run_pair(ctx, d, u, m, 160, 90, color_init=3)
        assert_bit_exact(r, "within the budget")
    finally:
        ctx.close()
