"""The names that kernel statistics come under: each one the runtime records is
explained in include/euchip.h (CPU), and each kind of frame has its own (GPU)."""
import os
import re

import numpy as np
import pytest

from euc_amd import scenes as S
from euc_amd.pipeline import DepthMode, PipelineDesc, Primitives, Shader, Xform

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def read(*path):
    with open(os.path.join(ROOT, *path)) as f:
        return f.read()


def test_names_documented():
    names = set(re.findall(r'timed(?:_on)?\(ctx,[^"()]*"(\w+)"', read("euc_amd", "csrc", "runtime.cpp")))
    assert {"setup", "raster", "lines", "clear", "batch_setup", "batch_raster"} <= names
    before = read("include", "euchip.h").split("typedef struct euchip_kernel_stat")[0]
    comment = before[before.rindex("/*"):]
    assert not [n for n in names if f'"{n}"' not in comment]


@pytest.mark.gpu
def test_names_per_frame():
    from euc_amd.renderer import Context
    ctx = Context(0)
    try:
        sc = S.torus_scene(1, 320, 240, 24, 12, 1)
        d = PipelineDesc.make(Shader.PHONG, Xform.MVP, depth_mode=DepthMode.LESS_WRITE)
        dl = PipelineDesc.make(Shader.PHONG, Xform.MVP, depth_mode=DepthMode.LESS_WRITE, primitives=Primitives.LINE_TRIANGLE_LIST)
        few = S.Mesh(pos=sc.mesh.pos, nrm=sc.mesh.nrm, idx=sc.mesh.idx[:36], count=36)
        c, z = ctx.color_target(320, 240), ctx.depth_target(320, 240)
        ctx.set_profiling(True)
        for desc, mesh, names in [(d, sc.mesh, {"setup", "raster"}), (d, few, {"tiny"}), (dl, sc.mesh, {"lines"})]:
            ctx.reset_stats()
            ctx.render(desc, sc.uniforms, ctx.mesh(mesh), c, z, clear_color=0, clear_depth=1.0)
            assert set(ctx.kernel_stats()) == names
        ctx.reset_stats()
        c.clear(np.uint32(5))
        ctx.synchronize()
        assert set(ctx.kernel_stats()) == {"clear"}
    finally:
        ctx.close()
