"""Lines frames on both sides of the count up to which a line has a wave to itself
(2048): bit-exact with the oracle, cleared and loaded targets, lines shorter and
longer than a wave's 64 steps, with shaded vertices.  And the time of few long
lines over loaded depth, by a factor between both sides (1.4 times that of short
lines with a wave each, 3.2 with the whole wave walking four lines in turn)."""
import time

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import BandPolicy, DepthMode, PipelineDesc, Primitives, Shader, Xform
from tests.parity import assert_bit_exact, run_pair

pytestmark = pytest.mark.gpu


def lines(seed, n, length, w, h):
    rng = np.random.default_rng(seed)
    pos = np.ones((n, 2, 4), np.float32)
    a = rng.uniform(0.0, 2.0 * np.pi, n)
    pos[:, 0, :2] = rng.uniform(-1.0, 1.0, (n, 2))
    pos[:, 1, 0] = pos[:, 0, 0] + np.cos(a) * length * 2.0 / w
    pos[:, 1, 1] = pos[:, 0, 1] + np.sin(a) * length * 2.0 / h
    pos[:, :, 2] = rng.uniform(0.0, 1.0, (n, 2))
    return S.Mesh(pos=pos.reshape(-1, 4), count=2 * n, rgba8=rng.integers(0, 2 ** 32, 2 * n, dtype=np.uint64).astype(np.uint32),
                  col=rng.uniform(0.0, 1.0, (2 * n, 4)).astype(np.float32))


def desc(shader, dm):
    return PipelineDesc.make(shader, Xform.CLIP, depth_mode=dm, band_policy=BandPolicy.SEQ, primitives=Primitives.LINE_LIST)


@pytest.mark.parametrize("n", [1, 3, 5, 2047, 2048, 2049])
@pytest.mark.parametrize("length", [1, 64, 700])
@pytest.mark.parametrize("shader,dm", [(Shader.FLAT, DepthMode.LESS_WRITE), (Shader.COLOR, DepthMode.LESS_PASS),
                                       (Shader.COLOR, DepthMode.GREATER_WRITE), (Shader.FLAT, DepthMode.NONE)])
def test_counts(gpu_ctx, n, length, shader, dm):
    w, h = 500, 301
    rng = np.random.default_rng(n)
    loaded = dm in (DepthMode.LESS_PASS, DepthMode.GREATER_WRITE)
    r = run_pair(gpu_ctx, desc(shader, dm), S.uniforms(), lines(n + length, n, length, w, h), w, h,
                 color_init=rng.integers(0, 2 ** 32, (h, w), dtype=np.uint64).astype(np.uint32) if loaded else 5,
                 depth_init=rng.uniform(0.2, 0.8, (h, w)).astype(np.float32) if loaded else 1.0)
    assert_bit_exact(r, f"{n} lines of {length}")


def test_few_long_lines(gpu_ctx):
    w, h = 1920, 1080
    c, z = gpu_ctx.color_target(w, h), gpu_ctx.depth_target(w, h)
    z.clear(1.0)
    best = {}
    for length in (5, 900):
        gm = gpu_ctx.mesh(lines(3, 300, length, w, h))
        for _ in range(6):
            t = time.perf_counter()
            for _ in range(50):
                gpu_ctx.render(desc(Shader.FLAT, DepthMode.LESS_PASS), S.uniforms(), gm, c, z, sync=False)
            gpu_ctx.synchronize()
            best[length] = min(best.get(length, 1.0), (time.perf_counter() - t) / 50)
    print(f"{best[5] * 1e6:.1f} us, {best[900] * 1e6:.1f} us")
    assert best[900] < 2.2 * best[5]
