"""The renders that this framework's performance is judged by.

Each case is one pass of a program over its public entry points
(`Context.render`, `Batch`): a frame, a frame of several passes or draws, or a
batch of requests.  A case names its `kind` and its sizes:

  cube     12 textured triangles without a depth test, one blocking render
  icon     one small Phong object into a small square target, one blocking render
  soup     random clip-space triangles, flat colours (large triangles)
  torus    Phong or Gouraud tori (small triangles)
  draws    many objects, one render() each, into one pair of targets
  shadow   depth-only pass, then Phong with a shadow lookup into a BGRA target
  terrain  depth-only pass, then a textured, shadowed, multisampled heightfield
  wire     the edges of a torus as lines
  icons    a batch of small objects, replayed from a graph
  views    a batch of textured views of resident meshes, set anew each pass

Targets are tensors wrapped as device buffers, so results stay on the device as
a program that displays or encodes them there would have it.  Frames are
enqueued without waiting (`sync=False`) as in an animation loop, except where
the kind says "blocking".
"""
from __future__ import annotations

import math

import numpy as np
import torch

from euc_amd import scenes as S
from euc_amd._lib import FORMAT_F32, FORMAT_RGBA8
from euc_amd.pipeline import (AaMode, BandPolicy, CullMode, DepthMode, PipelineDesc, PixelFormat, PixelMode, Primitives,
                              Sampler, Shader, Xform)
from euc_amd.renderer import Buffer2d, Context, Request

SAMPLERS = {"linear": Sampler.LINEAR, "linear_tiled": Sampler.LINEAR_TILED, "nearest_clamped": Sampler.NEAREST_CLAMPED}
ICON_CLEAR = 0xFF202020


def listed():
    return [
        # The smallest frame a program draws: examples/texture_mapping.rs, a dozen
        # textured triangles; latency and launches are what it waits for.
        {"name": "cube_800x600", "kind": "cube", "width": 800, "height": 600, "texture": 256, "sampler": "linear"},
        # One thumbnail on its own, as a program without a batch renders it.
        {"name": "icon_96", "kind": "icon", "side": 96, "triangles": 2000},
        # Large overlapping triangles (user interfaces, backdrops, stress tests).
        {"name": "soup_640x480", "kind": "soup", "width": 640, "height": 480, "triangles": 1024},
        # A scene of objects, one draw call each, over the depth the earlier ones left;
        # the window has an odd size.
        {"name": "draws_1003x701", "kind": "draws", "width": 1003, "height": 701, "objects": 16, "triangles": 3000},
        # The flagship frame: dense smooth meshes, per-pixel lighting, full HD.
        {"name": "torus_phong_1080p", "kind": "torus", "width": 1920, "height": 1080, "segments": 256, "rings": 128,
         "instances": 4, "shader": "phong"},
        # Per-vertex lighting of coarser meshes at a laptop's resolution.
        {"name": "torus_gouraud_1366x768", "kind": "torus", "width": 1366, "height": 768, "segments": 97, "rings": 51,
         "instances": 3, "shader": "gouraud"},
        # The largest frame: a million triangles in ultra HD.
        {"name": "torus_phong_2160p", "kind": "torus", "width": 3840, "height": 2160, "segments": 256, "rings": 128,
         "instances": 16, "shader": "phong"},
        # The reference's own benchmark frame (benches/teapot.rs) at one of its sizes: a
        # few thousand triangles with a point light's shadow map.
        {"name": "shadow_1024x800", "kind": "shadow", "width": 1024, "height": 800, "segments": 80, "rings": 40,
         "shadow": 512},
        # An outdoor scene: every pixel shaded, texture, shadow map, coarse-sample antialiasing.
        {"name": "terrain_1080p", "kind": "terrain", "width": 1920, "height": 1080, "grid": 317, "texture": 1024,
         "shadow": 2048, "msaa": 1},
        # A wireframe view (examples/wireframes.rs).
        {"name": "wire_1280x720", "kind": "wire", "width": 1280, "height": 720, "segments": 64, "rings": 32},
        # A thumbnail service: a fixed set of objects rendered in one replay.
        {"name": "icons_1024", "kind": "icons", "requests": 1024},
        # A render service's batch: cameras, sizes and textures differ per request and
        # per batch, meshes are resident.
        {"name": "views_64", "kind": "views", "requests": 64, "triangles": 200000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cube", "icon", "soup", "draws", "torus", "torus", "shadow", "terrain", "wire", "icons", "views"])
    if kind == "cube":
        w = _log(rng, 320, 1600)
        return {"kind": kind, "width": w, "height": max(240, w * 3 // 4 - rng.randrange(9)),
                "texture": rng.choice([64, 256, 333, 1024]), "sampler": rng.choice(sorted(SAMPLERS))}
    if kind == "icon":
        return {"kind": kind, "side": _log(rng, 32, 256), "triangles": _log(rng, 200, 20000)}
    if kind == "soup":
        w = _log(rng, 320, 1024)
        return {"kind": kind, "width": w, "height": w * 3 // 4 + rng.randrange(9), "triangles": _log(rng, 128, 1024)}
    if kind == "draws":
        w = _log(rng, 320, 1600)
        return {"kind": kind, "width": w, "height": w * 9 // 16 + rng.randrange(9), "objects": _log(rng, 4, 24),
                "triangles": _log(rng, 200, 20000)}
    if kind == "torus":
        w = _log(rng, 320, 3840)
        n = _log(rng, 24, 256)
        return {"kind": kind, "width": w, "height": w * 9 // 16 + rng.randrange(-7, 1), "segments": n,
                "rings": max(8, n // 2 - rng.randrange(5)), "instances": rng.randrange(1, 10),
                "shader": rng.choice(["phong", "gouraud"])}
    if kind == "shadow":
        w = _log(rng, 320, 2048)
        n = _log(rng, 24, 160)
        return {"kind": kind, "width": w, "height": w * 25 // 32 + rng.randrange(5), "segments": n, "rings": max(8, n // 2),
                "shadow": _log(rng, 200, 1024)}
    if kind == "terrain":
        w = _log(rng, 480, 1920)
        return {"kind": kind, "width": w, "height": w * 9 // 16 - rng.randrange(5), "grid": _log(rng, 40, 317),
                "texture": rng.choice([128, 500, 1024]), "shadow": _log(rng, 300, 2048), "msaa": rng.choice([0, 1, 1, 2])}
    if kind == "wire":
        w = _log(rng, 320, 1920)
        n = _log(rng, 16, 128)
        return {"kind": kind, "width": w, "height": w * 9 // 16 + rng.randrange(5), "segments": n, "rings": max(8, n // 2)}
    if kind == "icons":
        return {"kind": kind, "requests": _log(rng, 32, 1024)}
    return {"kind": kind, "requests": _log(rng, 6, 64), "triangles": _log(rng, 5000, 200000)}


# --------------------------------------------------------------------------- #
# Scenes: what a pass draws, on the host.  A scene is a list of passes (or
# requests): dicts of mesh, uniforms, desc, size and texture.
# --------------------------------------------------------------------------- #

def _item(mesh, u, desc, w, h, texture=None, color=0):
    return {"mesh": mesh, "u": u, "desc": desc, "w": w, "h": h, "texture": texture, "color": color}


def _torus_mesh(c, instances, seed):
    return S.torus_scene(seed, c["width"], c["height"], c["segments"], c["rings"], instances)


def _scene(c, seed):
    kind = c["kind"]
    write = DepthMode.LESS_WRITE
    shadow_desc = PipelineDesc.make(Shader.DEPTH_ONLY, Xform.MVP, pixel_mode=PixelMode.PASS, depth_mode=write,
                                    cull=CullMode.NONE, band_policy=BandPolicy.SEQ)
    if kind == "cube":
        tex = S.noise_texture(seed, c["texture"])
        sc = S.texture_cube_scene(tex, seed % 4000, c["width"], c["height"])
        d = PipelineDesc.make(Shader.TEXTURED, Xform.MVP, sampler=SAMPLERS[c["sampler"]])
        return [_item(sc.mesh, sc.uniforms, d, sc.width, sc.height, tex, 180)]
    if kind == "icon":
        sc = S.icon_request(seed, c["triangles"], c["triangles"], c["side"], c["side"])
        d = PipelineDesc.make(Shader.PHONG, Xform.MVP, depth_mode=write, band_policy=BandPolicy.SEQ)
        return [_item(sc.mesh, sc.uniforms, d, sc.width, sc.height, None, ICON_CLEAR)]
    if kind == "soup":
        sc = S.plain_scene(seed, c["triangles"], c["width"], c["height"])
        return [_item(sc.mesh, sc.uniforms, PipelineDesc.make(Shader.FLAT, Xform.CLIP, depth_mode=write), sc.width, sc.height)]
    if kind == "torus":
        sc = _torus_mesh(c, c["instances"], seed)
        d = PipelineDesc.make(Shader.PHONG if c["shader"] == "phong" else Shader.GOURAUD, Xform.MVP, depth_mode=write)
        return [_item(sc.mesh, sc.uniforms, d, sc.width, sc.height)]
    if kind == "draws":
        d = PipelineDesc.make(Shader.GOURAUD, Xform.MVP, depth_mode=write)
        vp = S.perspective_fov_lh_zo(1.1, c["width"], c["height"], 0.1, 100.0)
        u = S.uniforms(view_proj=S.f32(vp), lights=[((-0.3, -0.6, -0.7), 1.0), ((0.7, 0.3, -0.4), 0.5)])
        r = S.rand_f32(seed, 6 * c["objects"]).astype(np.float64).reshape(-1, 6)
        out = []
        for k in range(c["objects"]):
            m = S.icon_request(seed + 1 + k, c["triangles"], c["triangles"]).mesh
            m.models = S.f32(S.translation((r[k, 0] - 0.5) * 7.0, (r[k, 1] - 0.5) * 4.0, 4.0 + 3.0 * r[k, 2]) @
                             S.rotation(*(r[k, 3:] * 2 * np.pi))).reshape(1, 16)
            out.append(_item(m, u, d, c["width"], c["height"]))
        return out
    if kind == "shadow":
        sc = _torus_mesh(c, 1, seed)
        m = sc.mesh
        light = np.array([-8.0, 5.0, -5.0])
        m.models = S.f32(S.translation(0.0, 0.0, 2.4) @ S.rotation(*(S.rand_f32(seed, 3).astype(np.float64) * 6.28))).reshape(1, 16)
        lvp = S.f32(S.perspective_fov_lh_zo(0.45, c["shadow"], c["shadow"], 0.1, 100.0) @
                    S.look_at_lh(light, (0.0, 0.0, 2.4), (0.0, 1.0, 0.0)))
        vp = S.f32(S.perspective_fov_lh_zo(1.0, c["width"], c["height"], 0.01, 100.0))
        u = S.uniforms(view_proj=vp, light_pos=tuple(light), light_vp=lvp)
        d = PipelineDesc.make(Shader.PHONG_SHADOW, Xform.MVP, depth_mode=write, pixel_format=PixelFormat.BGRA8)
        return [_item(m, S.uniforms(view_proj=lvp), shadow_desc, c["shadow"], c["shadow"]),
                _item(m, u, d, c["width"], c["height"])]
    if kind == "terrain":
        sc = S.heightfield_scene(seed, c["width"], c["height"], c["grid"], c["texture"], c["shadow"])
        d = PipelineDesc.make(Shader.TEX_SHADOW, Xform.MVP, depth_mode=write,
                              aa_mode=AaMode.Msaa(c["msaa"]) if c["msaa"] else AaMode.NONE)
        return [_item(sc.mesh, sc.extra["shadow_uniforms"], shadow_desc, c["shadow"], c["shadow"]),
                _item(sc.mesh, sc.uniforms, d, sc.width, sc.height, sc.texture)]
    if kind == "wire":
        sc = _torus_mesh(c, 1, seed)
        m = sc.mesh
        m.models = S.f32(S.translation(0.0, 0.0, 2.2) @ S.rotation(*(S.rand_f32(seed, 3).astype(np.float64) * 6.28))).reshape(1, 16)
        m.col = np.repeat(np.array([[1.0, 0.25, 0.25, 1.0]], np.float32), m.n_vertices, 0)
        d = PipelineDesc.make(Shader.COLOR, Xform.MVP, depth_mode=write, primitives=Primitives.LINE_TRIANGLE_LIST)
        return [_item(m, sc.uniforms, d, sc.width, sc.height)]
    if kind == "icons":
        d = PipelineDesc.make(Shader.PHONG, Xform.MVP, depth_mode=write, band_policy=BandPolicy.SEQ)
        sides = 32 + (S.rand_f32(0x51DE, c["requests"]) * 225).astype(int)  # the service's target sizes
        scs = [S.icon_request(seed * 4099 + i, min_side=int(s), max_side=int(s)) for i, s in enumerate(sides)]
        return [_item(sc.mesh, sc.uniforms, d, sc.width, sc.height, None, ICON_CLEAR) for sc in scs]
    assert kind == "views", kind
    d = PipelineDesc.make(Shader.TEXTURED, Xform.MVP, depth_mode=write, band_policy=BandPolicy.SEQ)
    meshes, texs = S.serving_assets(seed, 6, 4, 1000, c["triangles"], (256, 512, 1024, 2048))
    out = []
    for i in range(c["requests"]):
        side = S.serving_request(i, 1, 1)[3]
        mi, ti, u, _ = S.serving_request(seed * 7919 + i, len(meshes), len(texs))
        out.append(_item(meshes[mi], u, d, side, side, texs[ti]))
    return out


# --------------------------------------------------------------------------- #
# Prepare and run
# --------------------------------------------------------------------------- #

_context = None


def context() -> Context:
    """A program's one context."""
    global _context
    if _context is None:
        _context = Context(torch.cuda.current_device())
    return _context


def _targets(ctx, sizes):
    """(colour tensor, depth tensor, [(colour buffer, depth buffer)]): targets of
    the given sizes, one after the other in one tensor each."""
    n = sum(w * h for w, h in sizes)
    color = torch.full((n,), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    depth = torch.full((n,), 0.5, dtype=torch.float32, device="cuda")
    bufs, at = [], 0
    for w, h in sizes:
        bufs.append((Buffer2d(ctx, FORMAT_RGBA8, w, h, color.data_ptr() + 4 * at),
                     Buffer2d(ctx, FORMAT_F32, w, h, depth.data_ptr() + 4 * at)))
        at += w * h
    if len(sizes) == 1:
        w, h = sizes[0]
        color, depth = color.view(h, w), depth.view(h, w)
    return color, depth, bufs


def prepare(case, seed):
    ctx = context()
    kind = case["kind"]
    items = _scene(case, seed)
    meshes, textures = {}, {}
    for it in items:  # meshes and textures that several requests share are uploaded once
        if id(it["mesh"]) not in meshes:
            meshes[id(it["mesh"])] = ctx.mesh(it["mesh"])
        t = it["texture"]
        if t is not None and id(t) not in textures:
            textures[id(t)] = ctx.texture(t)
    state = {"kind": kind, "ctx": ctx, "items": [
        dict(it, mesh=meshes[id(it["mesh"])], texture=None if it["texture"] is None else textures[id(it["texture"])])
        for it in items]}
    if kind in ("shadow", "terrain"):
        s = items[0]
        state["map"] = torch.full((s["h"], s["w"]), 0.5, dtype=torch.float32, device="cuda")
        state["map_buffer"] = Buffer2d(ctx, FORMAT_F32, s["w"], s["h"], state["map"].data_ptr())
        items = items[1:]
    sizes = [(it["w"], it["h"]) for it in (items if kind in ("icons", "views") else items[:1])]
    state["color"], state["depth"], state["buffers"] = _targets(ctx, sizes)
    if kind in ("icons", "views"):
        state["requests"] = [Request(it["mesh"], c, d, it["u"], texture=it["texture"])
                             for it, (c, d) in zip(state["items"], state["buffers"])]
        state["batch"] = ctx.batch()
        if kind == "icons":
            state["batch"].set(items[0]["desc"], state["requests"], clear_color=ICON_CLEAR, clear_depth=1.0)
    torch.cuda.synchronize()  # the tensors are filled on torch's stream, the context has its own
    return state


def run(state):
    ctx, kind, items = state["ctx"], state["kind"], state["items"]
    if kind == "icons":
        state["batch"].launch(graph=True)
        state["batch"].wait()
    elif kind == "views":
        b = state["batch"]
        b.set(items[0]["desc"], state["requests"], clear_color=0, clear_depth=1.0)
        b.launch()
        b.wait()
    elif kind in ("shadow", "terrain"):
        s, m = items
        (color, depth), = state["buffers"]
        ctx.render(s["desc"], s["u"], s["mesh"], None, state["map_buffer"], clear_depth=1.0, sync=False)
        ctx.render(m["desc"], m["u"], m["mesh"], color, depth, texture=m["texture"], shadow=state["map_buffer"],
                   clear_color=0, clear_depth=1.0, sync=False)
        return {"map": state["map"], "color": state["color"], "depth": state["depth"]}
    elif kind == "draws":
        (color, depth), = state["buffers"]
        for k, it in enumerate(items):  # the first draw clears, the others add to what is there
            ctx.render(it["desc"], it["u"], it["mesh"], color, depth, clear_color=None if k else 0,
                       clear_depth=None if k else 1.0, sync=False)
    else:
        it, = items
        (color, depth), = state["buffers"]
        if kind == "cube":
            ctx.render(it["desc"], it["u"], it["mesh"], color, None, texture=it["texture"], clear_color=it["color"])
            return {"color": state["color"]}
        ctx.render(it["desc"], it["u"], it["mesh"], color, depth, clear_color=it["color"], clear_depth=1.0,
                   sync=kind == "icon")
    return {"color": state["color"], "depth": state["depth"]}


def work(case):
    """Bytes of a pass: meshes and textures read once per use, targets written once."""
    items = _scene(case, 1)
    reads, seen = 0, set()
    for it in items:
        m, t = it["mesh"], it["texture"]
        if id(m) not in seen:
            seen.add(id(m))
            reads += m.input_bytes()
        if t is not None and id(t) not in seen:
            seen.add(id(t))
            reads += t.nbytes
    kind = case["kind"]
    if kind in ("shadow", "terrain"):
        s, m = items
        return {"bytes": reads + 2 * 4 * s["w"] * s["h"] + 8 * m["w"] * m["h"], "flops": 0}
    if kind in ("icons", "views"):
        return {"bytes": reads + sum(8 * it["w"] * it["h"] for it in items), "flops": 0}
    return {"bytes": reads + (4 if kind == "cube" else 8) * items[0]["w"] * items[0]["h"], "flops": 0}


# --------------------------------------------------------------------------- #
# Depth in 64 bits: the nearest surface at every pixel's corner, triangle by
# triangle, with no pixel order, spans or rounding of its own.  Colours are bytes.
# --------------------------------------------------------------------------- #

def _depth64(it, depth):
    """Nearest depth of the item's triangles, minimum with `depth` (float64, (h, w))."""
    m, d, w, h = it["mesh"], it["desc"], it["w"], it["h"]
    f64 = dict(dtype=torch.float64, device="cuda")
    pos = torch.tensor(m.pos, **f64)
    idx = torch.arange(m.count, device="cuda") if m.idx is None else torch.tensor(m.idx.astype(np.int64), device="cuda")
    if d.xform == Xform.CLIP:
        clip = pos[None]
    else:
        vp = torch.tensor(it["u"][:16].reshape(4, 4), **f64)
        models = torch.tensor(m.models, **f64).view(-1, 4, 4)
        clip = torch.cat([pos, torch.ones_like(pos[:, :1])], 1) @ (vp @ models).transpose(1, 2).contiguous()
    ndc = clip[..., :3] / clip[..., 3:]
    tri = ndc[:, idx].reshape(-1, 3, 3)
    x = (tri[..., 0] * 0.5 + 0.5) * w
    y = (tri[..., 1] * -0.5 + 0.5) * h
    z = tri[..., 2]
    det = (x[:, 1] - x[:, 0]) * (y[:, 2] - y[:, 0]) - (y[:, 1] - y[:, 0]) * (x[:, 2] - x[:, 0])
    x0, x1 = x.amin(1).ceil().clamp(0, w), x.amax(1).floor().add(1).clamp(0, w)
    y0, y1 = y.amin(1).ceil().clamp(0, h), y.amax(1).floor().add(1).clamp(0, h)
    keep = (det != 0) & (x1 > x0) & (y1 > y0)
    if d.cull == CullMode.BACK:
        keep &= det < 0  # the screen's y axis points down
    elif d.cull == CullMode.FRONT:
        keep &= det > 0
    x, y, z, det = x[keep], y[keep], z[keep], det[keep]
    x0, y0 = x0[keep].long(), y0[keep].long()
    bw, bh = x1[keep].long() - x0, y1[keep].long() - y0
    ends = torch.cumsum(bw * bh, 0).cpu().numpy()
    flat, at, base = depth.view(-1), 0, 0
    while at < len(ends):
        to = max(at + 1, int(np.searchsorted(ends, base + (1 << 24), side="right")))
        n = (bw * bh)[at:to]
        t = torch.repeat_interleave(torch.arange(at, to, device="cuda"), n)
        k = torch.arange(t.numel(), device="cuda") - (torch.cumsum(n, 0) - n)[t - at]
        px, py = x0[t] + k % bw[t], y0[t] + k // bw[t]
        e = []
        for i in range(3):
            j, l = (i + 1) % 3, (i + 2) % 3
            e.append(((x[t, j] - px) * (y[t, l] - py) - (y[t, j] - py) * (x[t, l] - px)) / det[t])
        zz = e[0] * z[t, 0] + e[1] * z[t, 1] + e[2] * z[t, 2]
        ok = (e[0] >= 0) & (e[1] >= 0) & (e[2] >= 0) & (zz >= 0) & (zz <= 1)
        flat.scatter_reduce_(0, (py * w + px)[ok], zz[ok], "amin")
        base, at = int(ends[to - 1]), to
    return depth


def exact(case, seed):
    kind = case["kind"]
    if kind in ("cube", "wire"):  # bytes alone; a line's pixels come from an integer walk of rounded ends
        return None
    items = _scene(case, seed)

    def fresh(it):
        return torch.ones((it["h"], it["w"]), dtype=torch.float64, device="cuda")

    if kind in ("shadow", "terrain"):
        return {"map": _depth64(items[0], fresh(items[0])), "color": None, "depth": _depth64(items[1], fresh(items[1]))}
    if kind in ("icons", "views"):
        return {"color": None, "depth": torch.cat([_depth64(it, fresh(it)).view(-1) for it in items])}
    depth = fresh(items[0])
    for it in items:
        _depth64(it, depth)
    return {"color": None, "depth": depth}
