"""The lines' walk and the keys between frames, against the oracle, bit-exact:
lines of one pixel, of about the length at which the whole wave takes a line, far
longer, and with ends thousands of pixels outside (64-bit steps), line counts
around a workgroup's 16; and frames of other depth modes, sizes and loaded
targets after one another on one context, which find the keys of the last frame
zeroed."""
import ctypes as C

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, DepthMode, PipelineDesc, Primitives, Shader, Xform
from euc_amd.renderer import Context
from oracle import oracle as O
from tests.parity import assert_bit_exact, run_pair

pytestmark = pytest.mark.gpu


def lines(seed, n, length, w, extent=1.0):
    """n lines of about `length` pixels at a target of width w."""
    rng = np.random.default_rng(seed)
    pos = np.ones((n, 2, 4), np.float32)
    pos[:, 0, :2] = rng.uniform(-extent, extent, (n, 2))
    pos[:, 1, :2] = pos[:, 0, :2] + rng.normal(0.0, 2.0 * length / w, (n, 2))
    pos[:, :, 2] = rng.uniform(0.0, 1.0, (n, 2))
    rgba8 = rng.integers(0, 2 ** 32, 2 * n, dtype=np.uint64).astype(np.uint32)
    return S.Mesh(pos=pos.reshape(-1, 4), count=2 * n, rgba8=rgba8)


def desc(dm, band=BandPolicy.SEQ):
    return PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=dm, band_policy=band, primitives=Primitives.LINE_LIST)


@pytest.mark.parametrize("n,length,extent", [(1, 20, 0.5), (15, 1, 1.0), (17, 255, 0.8), (64, 260, 1.0), (300, 900, 1.5),
                                             (40, 60000, 30.0), (4000, 12, 1.0)])
def test_line_lengths(gpu_ctx, n, length, extent):
    w, h = 1500, 700
    mesh = lines(n + length, n, length, w, extent)
    r = run_pair(gpu_ctx, desc(DepthMode.LESS_WRITE), S.uniforms(), mesh, w, h)
    assert_bit_exact(r, f"{n} lines of {length}")


def test_keys_between_frames():
    ctx = Context(0)
    try:
        rng = np.random.default_rng(3)
        for k, (dm, w, h, load) in enumerate([
                (DepthMode.LESS_WRITE, 300, 200, False), (DepthMode.GREATER_WRITE, 300, 200, True),
                (DepthMode.NONE, 640, 480, False), (DepthMode.LESS_PASS, 200, 333, True),
                (DepthMode.LESS_WRITE, 640, 480, True), (DepthMode.NONE, 64, 48, True),
                (DepthMode.GREATER_PASS, 900, 600, True), (DepthMode.LESS_WRITE, 300, 200, False)]):
            mesh = lines(50 + k, 500, 60, w)
            z = rng.uniform(0.2, 0.8, (h, w)).astype(np.float32) if load else 1.0
            c = rng.integers(0, 2 ** 32, (h, w), dtype=np.uint64).astype(np.uint32) if load else 7
            r = run_pair(ctx, desc(dm), S.uniforms(), mesh, w, h, color_init=c, depth_init=z)
            assert r["frags"] > 50
            assert_bit_exact(r, f"frame {k} {dm}")
    finally:
        ctx.close()


def test_keys_replaced_within_a_budget():
    """Larger keys that fit the budget only once the old ones are freed (the new
    storage may then have the old address) start at zero as well."""
    ctx = Context(0)
    try:
        gm = ctx.mesh(lines(7, 300, 40, 640))
        sizes = [(100, 80), (320, 240), (640, 480)]
        targets = [(ctx.color_target(*s), ctx.depth_target(*s)) for s in sizes]
        for k, ((w, h), (c, z)) in enumerate(zip(sizes, targets)):
            if k:
                old = sizes[k - 1][0] * sizes[k - 1][1]
                ctx.set_budget(ctx.bytes_in_use() + 8 * (max(w * h, old + old // 2) - old))
            ctx.render(desc(DepthMode.LESS_WRITE), S.uniforms(), gm, c, z, clear_color=9, clear_depth=1.0)
            oc, od = np.full((h, w), 9, np.uint32), np.full((h, w), 1.0, np.float32)
            rc, frags = O.render(desc(DepthMode.LESS_WRITE), S.uniforms(), lines(7, 300, 40, 640), oc, od)
            assert rc == 0 and frags > 50
            assert np.array_equal(c.download(), oc), k
            assert np.array_equal(z.download().view(np.uint32), od.view(np.uint32)), k
    finally:
        ctx.close()


def test_first_frame_captured():
    """A context's first lines frame recorded into a graph: the eager frames before
    and between its replays, and each replay, find the keys zeroed."""
    hip = C.CDLL("libamdhip64.so.7")
    w, h = 640, 480
    ctx = Context(0)
    old = ctx.color_target(w, 2 * h)  # its storage, all ones, may become the keys
    old.clear(0xFFFFFFFF)
    ctx.synchronize()
    old.close()
    try:
        mesh = lines(8, 400, 50, w)
        gm, stream = ctx.mesh(mesh), C.c_void_p(ctx.stream())
        d = desc(DepthMode.LESS_WRITE)
        oc, od = np.full((h, w), 9, np.uint32), np.full((h, w), 1.0, np.float32)
        rc, frags = O.render(d, S.uniforms(), mesh, oc, od)
        assert rc == 0 and frags > 50
        (gc, gz), (ec, ez) = [(ctx.color_target(w, h), ctx.depth_target(w, h)) for _ in range(2)]

        def render(c, z):
            ctx.render(d, S.uniforms(), gm, c, z, clear_color=9, clear_depth=1.0, sync=False)

        def check(c, z, what):
            ctx.synchronize()
            assert np.array_equal(c.download(), oc), what
            assert np.array_equal(z.download().view(np.uint32), od.view(np.uint32)), what

        graph, ex = C.c_void_p(), C.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed: the frame allocates
        render(gc, gz)
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
        for k in range(3):
            render(ec, ez)
            check(ec, ez, f"eager {k}")
            ec.clear(0)
            gc.clear(0)
            gz.clear(0)
            assert hip.hipGraphLaunch(ex, stream) == 0
            check(gc, gz, f"replay {k}")
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
    finally:
        ctx.close()
