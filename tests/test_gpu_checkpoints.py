"""Frames of few triangles through the row checkpoints: the depth modes, MSAA and
occlusion bounds of test_gpu_bigtri.py, whose meshes of up to 64 triangles take one
launch by default, in a context with a budget, which keeps to the frames with
scratch memory, and with more triangles than one launch takes.  Each checks that no
frame took the one launch."""
import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import DepthMode
from tests import test_gpu_bigtri as B
from tests.parity import assert_bit_exact, run_pair

pytestmark = pytest.mark.gpu

MODES = [DepthMode.LESS_WRITE, DepthMode.GREATER_WRITE, DepthMode.LESS_PASS, DepthMode.NONE, DepthMode(2, True)]


@pytest.fixture(params=["budget", "none"])
def ctx(request):
    from euc_amd.renderer import Context
    c = Context(0)
    if request.param == "budget":
        c.set_budget(1 << 36)
    c.few = request.param == "budget"  # frames of few triangles are checkpoint frames here
    c.set_profiling(True)
    yield c
    names = set(c.kernel_stats())
    c.close()
    assert names == {"setup", "raster"}, names


def more(ctx, mesh, n):
    """The mesh, or its triangles over and over up to n where few would take one launch."""
    if ctx.few:
        return mesh
    k = -(-3 * n // mesh.count)
    return S.Mesh(pos=np.tile(mesh.pos, (k, 1))[:3 * n], count=3 * n, rgba8=np.tile(mesh.rgba8, k)[:3 * n] + np.arange(3 * n, dtype=np.uint32) // 3)


@pytest.mark.parametrize("dm", MODES)
def test_depth_modes(ctx, dm):
    init = 0.5 if dm.test in (2, 3) else 1.0
    mesh = more(ctx, B.corner_triangles(11, 40), 97)
    assert B.checkpoint_on(mesh.count // 3, 700, 500)
    r = run_pair(ctx, B.flat(dm=dm), S.uniforms(), mesh, 700, 500, depth_init=init)
    assert r["frags"] > 10 ** 5 or dm.test == 2
    assert_bit_exact(r, f"corner triangles {dm}")


@pytest.mark.parametrize("dm", MODES[:2])
@pytest.mark.parametrize("slope", [False, True])
def test_near_ties(ctx, dm, slope):
    mesh = more(ctx, B.tie_triangles(31 + slope, 48, slope=slope), 130)
    init = 0.0 if dm.test == 3 else 1.0
    r = run_pair(ctx, B.flat(dm=dm), S.uniforms(), mesh, 700, 500, depth_init=init)
    assert r["frags"] > 5 * 10 ** 5
    assert_bit_exact(r, f"ulp-close corner triangles {dm} slope={slope}")


@pytest.mark.parametrize("dm", MODES[:2])
def test_clip_and_large_weights(ctx, dm):
    rng = np.random.default_rng(41)
    m = B.corner_triangles(41, 40)
    pos = m.pos.copy()
    pos[:, 2] = rng.uniform(-0.4, 1.4, len(pos)).astype(np.float32)
    far = rng.random(40) < 0.5
    pos.reshape(40, 3, 4)[far, :, :2] *= np.float32(40.0)
    mesh = more(ctx, S.Mesh(pos=pos, count=m.count, rgba8=m.rgba8), 80)
    r = run_pair(ctx, B.flat(dm=dm), S.uniforms(), mesh, 640, 480, depth_init=0.0 if dm.test == 3 else 1.0)
    assert r["frags"] > 10 ** 5
    assert_bit_exact(r, "clipped and far corner triangles")
