"""The work users of this renderer have it do, as measurable cases.

A case is one pass of a program that keeps its meshes, textures, targets and
programs on the device: it draws through the public classes of
`softglrender_amd.renderer` and reads the images (or weights, or errors) it
needs back, as a headless renderer, a data generator or a trainer does.

Kinds:
  mesh      one displaced sphere, lit (Blinn-Phong, PBR + IBL or the learned shader), with or without a shadow
            pass, a floor that receives the shadow, a translucent sphere over it, 4x multisampling, a depth image
  viewer    an interactive viewer's frame: many small meshes, floor, skybox, axis lines and an FXAA pass
  wire      wireframe, vertex points and thick lines over a shaded mesh
  stress    random small triangles and screen-covering ones with vertex colours
  views     a captured batch of independent views, every image read back
  ibl       irradiance and prefiltered specular maps from an environment cube
  train     steps of the learned shader's training from given weights and records
  evaluate  the learned shader's error and gradient over a set of records
"""
from __future__ import annotations

import functools
import math
import struct

import numpy as np
import torch

from softglrender_amd import scenes
from softglrender_amd import stream as S
from softglrender_amd.renderer import (ClearStates, RendererHIP, SamplerDesc, ShaderResources, TextureDesc,
                                       VertexArray)

# ----------------------------------------------------------------------------- the cases


def listed():
    return [
        # a thumbnail or a test image: the smallest call, colour and depth wanted
        dict(name="thumbnail", kind="mesh", width=160, height=120, msaa=False, freq=6, shading="blinn", tex=64, layout=0,
             shadow=0, floor=False, translucent=False, depth=True),
        # a VGA frame of a small textured model without multisampling, colour and depth wanted (RGB-D data)
        dict(name="sphere_vga", kind="mesh", width=640, height=480, msaa=False, freq=14, shading="blinn", tex=512,
             layout=0, shadow=0, floor=False, translucent=False, depth=True),
        # an interactive viewer's window: many draws a frame, each too small to fill the device
        dict(name="viewer_window", kind="viewer", width=1366, height=768, nodes=16, freq=24, tex=256, sky=256, fxaa=True),
        # a preview of the full frame below: the same passes on a tenth of everything
        dict(name="pbr_preview", kind="mesh", width=480, height=270, msaa=True, freq=60, shading="pbr", tex=512, layout=2,
             shadow=512, floor=True, translucent=True, depth=False),
        # a full HD frame of a dense model: shadow pass, floor, PBR with image-based light, translucency, 4x
        # multisampling (the benchmark's frame, with the floor that makes the shadow map matter)
        dict(name="pbr_full_hd", kind="mesh", width=1920, height=1080, msaa=True, freq=224, shading="pbr", tex=2048,
             layout=2, shadow=2048, floor=True, translucent=True, depth=False),
        # a point-cloud-like soup of tiny triangles behind big ones at 4K: binning, depth culling and bandwidth
        dict(name="soup_4k", kind="stress", width=3840, height=2160, msaa=True, n=2_000_000, big=2000),
        # data generation: many views of several meshes in one captured batch, every image wanted
        dict(name="views_48", kind="views", views=48, scenes=16, size=512, tri_hi=100_000, tex=512),
        # an environment map becomes usable: 36 small cube-face passes with long shaders
        dict(name="ibl_512", kind="ibl", src=512, irr=32, pref=128),
        # the learned shader trained on captured fragments (forward, backward, update)
        dict(name="train_64_steps", kind="train", records=262_144, batch=16_384, steps=64),
        # the learned shader judged on held-out fragments, and its gradient over them
        dict(name="evaluate_300k", kind="evaluate", records=300_007),
        # the learned shader in a frame
        dict(name="learned_full_hd", kind="mesh", width=1920, height=1080, msaa=True, freq=160, shading="neural", tex=1024,
             layout=1, shadow=0, floor=False, translucent=False, depth=False),
        # an inspection view: wireframe, points and thick lines, odd sizes
        dict(name="wireframe", kind="wire", width=1001, height=563, msaa=False, freq=40, line_width=2.0, point_size=3.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mesh", "mesh", "mesh", "viewer", "wire", "stress", "views", "ibl", "train", "evaluate"])
    width = _log(rng, 64, 1920)
    height = max(33, int(width * rng.uniform(0.5, 1.0)))
    if kind == "mesh":
        msaa = rng.random() < 0.5
        shading = rng.choice(["blinn", "pbr", "pbr", "neural"])
        learned = shading == "neural"
        return dict(kind="mesh", width=width, height=min(height, 1080), msaa=msaa, freq=_log(rng, 6, 220), shading=shading,
                    tex=_log(rng, 64, 2048), layout=rng.randrange(3),
                    shadow=0 if learned or rng.random() < 0.5 else _log(rng, 128, 2048),
                    floor=not learned and rng.random() < 0.5, translucent=not learned and rng.random() < 0.5,
                    depth=not msaa and rng.random() < 0.5)
    if kind == "viewer":
        return dict(kind="viewer", width=max(width, 320), height=max(height, 200), nodes=rng.randrange(4, 25),
                    freq=_log(rng, 4, 40), tex=_log(rng, 32, 512), sky=_log(rng, 32, 256), fxaa=rng.random() < 0.5)
    if kind == "wire":
        return dict(kind="wire", width=width, height=height, msaa=rng.random() < 0.5, freq=_log(rng, 6, 60),
                    line_width=rng.choice([1.0, 1.0, 2.0, 3.0]), point_size=rng.choice([1.0, 2.0, 3.0, 5.0]))
    if kind == "stress":
        w = _log(rng, 256, 3840)
        return dict(kind="stress", width=w, height=max(33, int(w * rng.uniform(0.4, 0.56))), msaa=rng.random() < 0.7,
                    n=_log(rng, 10_000, 2_000_000), big=rng.choice([0, 1, 13, 200, 2000]))
    if kind == "views":
        return dict(kind="views", views=rng.randrange(3, 49), scenes=rng.randrange(1, 17), size=_log(rng, 48, 512),
                    tri_hi=_log(rng, 2_000, 100_000), tex=_log(rng, 64, 512))
    if kind == "ibl":
        src = 1 << rng.randrange(5, 10)
        return dict(kind="ibl", src=src, irr=_log(rng, 8, min(32, src)), pref=1 << rng.randrange(4, 8))
    if kind == "train":
        batch = _log(rng, 512, 16_384)
        return dict(kind="train", records=_log(rng, 4_096, 262_144), batch=batch, steps=_log(rng, 4, 64))
    return dict(kind="evaluate", records=_log(rng, 500, 300_000))


# ----------------------------------------------------------------------------- inputs from a seed


@functools.lru_cache(maxsize=64)
def _unit_sphere(freq):
    v, idx = scenes.icosphere(freq, 1.0)
    return v, np.ascontiguousarray(idx)


def _blob(freq, rng, amount=0.1, radius=1.0):
    """A sphere displaced by smooth waves, with its area-weighted normals (64-byte vertices)."""
    v, idx = _unit_sphere(freq)
    v = v.copy()
    p = v[:, 0:3].astype(np.float64)
    d = np.zeros(len(p))
    for k in range(6):
        w = rng.normal(size=3) * (1.5 + 1.5 * k)
        d += np.sin(p @ w + rng.uniform(0, 2 * np.pi)) / (1.0 + k)
    p *= (radius * (1.0 + amount * 0.5 * d))[:, None]
    a, b, c = p[idx[:, 0]], p[idx[:, 1]], p[idx[:, 2]]
    fn = np.cross(b - a, c - a)
    n = np.stack([np.bincount(idx.reshape(-1), np.repeat(fn[:, k], 3), len(p)) for k in range(3)], -1)
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    v[:, 0:3], v[:, 8:11] = p, n
    return v, idx


def _noise(size, rng):
    """(size, size, 3) value noise in [0, 1], four octaves."""
    acc = np.zeros((3, size, size), np.float32)
    for o in range(4):
        g = 4 * 2 ** o + 1
        lat = torch.from_numpy(rng.random((1, 3, g, g)).astype(np.float32))
        up = torch.nn.functional.interpolate(lat, size=(size, size), mode="bilinear", align_corners=True)
        acc += up[0].numpy() * np.float32(0.5 ** o / 1.875)
    return np.moveaxis(acc, 0, -1)


def _u8(x):
    return np.clip(x * 255.0 + 0.5, 0, 255).astype(np.uint8)


def _rgba(rgb):
    out = np.full(rgb.shape[:2] + (4,), 255, np.uint8)
    out[..., :3] = rgb
    return out


def _pbr_images(size, rng):
    albedo = _rgba(_u8(0.15 + 0.8 * _noise(size, rng)))
    n = _noise(size, rng)
    t = (n[..., :2] - 0.5) * 0.8
    inv = 1.0 / np.sqrt(1.0 + t[..., 0] ** 2 + t[..., 1] ** 2)
    normal = _rgba(_u8(np.stack([t[..., 0] * inv, t[..., 1] * inv, inv], -1) * 0.5 + 0.5))
    m = _noise(size, rng)
    metal = np.where(m[..., 1] > 0.55, np.float32(0.95), np.float32(0.05))
    mr = _rgba(_u8(np.stack([np.zeros_like(metal), 0.2 + 0.7 * m[..., 0], metal], -1)))
    return albedo, normal, mr


def _eye(rng, radius):
    """A camera on a sphere, never close to the poles."""
    phi, y = rng.uniform(0, 2 * np.pi), rng.uniform(-0.5, 0.6)
    c = math.sqrt(1.0 - y * y)
    return (radius * c * math.cos(phi), radius * y, radius * c * math.sin(phi))


def _translate(x, y, z):
    m = np.eye(4)
    m[:3, 3] = (x, y, z)
    return m


# ----------------------------------------------------------------------------- a small program on the renderer


class Program:
    """What a program keeps between frames: a renderer, its resources and the calls of one frame."""

    def __init__(self):
        self.r = RendererHIP(0)
        self.r.create()
        self.frame = []
        self.reads = []
        self.programs = {}

    def texture(self, image=None, width=0, height=0, fmt=S.FMT_RGBA8, usage=S.USAGE_SAMPLER | S.USAGE_UPLOAD, mip=False,
                msaa=False, cube=None, is_cube=False, layout=0, filt=None, wrap=S.WRAP_REPEAT):
        if image is not None:
            height, width = image.shape[:2]
        if cube is not None:
            height, width = cube[0].shape[:2]
        t = self.r.createTexture(TextureDesc(width=width, height=height, type=S.TEX_CUBE if is_cube or cube else S.TEX_2D,
                                             format=fmt, usage=usage, useMipmaps=mip, multiSample=msaa, layout=layout))
        lin = S.FILTER_LINEAR if filt is None else filt
        t.setSamplerDesc(SamplerDesc(S.FILTER_LINEAR_MIPMAP_LINEAR if mip else lin, lin, wrap, wrap, wrap, S.BORDER_BLACK))
        if image is not None:
            t.setImageData([image])
        elif cube is not None:
            t.setImageData(cube)
        else:
            t.initImageData()
        return t

    def mesh(self, verts, idx):
        return self.r.createVertexArrayObject(VertexArray(verts.shape[1] * 4, verts, idx))

    def target(self, color=None, depth=None, face=0, level=0):
        f = self.r.createFrameBuffer(True)
        if color is not None:
            f.setColorAttachment(color, level, face)
        if depth is not None:
            f.setDepthAttachment(depth)
        return f

    def begin(self, fbo, width, height, color=(0.02, 0.02, 0.05, 1.0), depth=1.0, clear_color=True, clear_depth=True):
        cs = ClearStates(clear_depth, clear_color, color, depth)
        self.frame.append((self.r.beginRenderPass, (fbo, cs)))
        self.frame.append((self.r.setViewPort, (0, 0, width, height)))

    def end(self):
        self.frame.append((self.r.endRenderPass, ()))

    def draw(self, vao, shading, defines, states, model, scene=bytes(S.SCENE_BYTES), material=bytes(S.MATERIAL_BYTES),
             samplers=None):
        key = (shading, defines)
        if key not in self.programs:
            p = self.r.createShaderProgram()
            p.addDefines([n for n, bit in (("ALBEDO_MAP", S.DEF_ALBEDO), ("NORMAL_MAP", S.DEF_NORMAL),
                                           ("METALROUGHNESS_MAP", S.DEF_METALROUGH)) if defines & bit])
            if not p.setShading(shading):
                raise RuntimeError(f"shading model {shading}")
            self.programs[key] = p
        res = ShaderResources()
        for n, b in (("UniformsModel", model), ("UniformsScene", scene), ("UniformsMaterial", material)):
            ub = self.r.createUniformBlock(n, len(b))
            ub.setData(b)
            res.blocks[n] = ub
        for n, t in (samplers or {}).items():
            s = self.r.createUniformSampler(n, TextureDesc())
            s.setTexture(t)
            res.samplers[n] = s
        self.frame += [(self.r.setVertexArrayObject, (vao,)), (self.r.setShaderProgram, (self.programs[key],)),
                       (self.r.setShaderResources, (res,)),
                       (self.r.setPipelineStates, (self.r.createPipelineStates(states),)), (self.r.draw, ())]

    def read(self, tex, layer=0, level=0):
        self.reads.append((tex, layer, level))

    def run(self):
        for fn, args in self.frame:
            fn(*args)
        return [t.readImage(layer, level) for t, layer, level in self.reads]


def _states(func=S.DEPTH_LESS, cull=True, blend=False):
    rs = S.RenderStates(blend=blend, depth_test=True, depth_mask=not blend, depth_func=func, cull_face=cull)
    rs.set_blend_factor(S.BF_SRC_ALPHA, S.BF_ONE_MINUS_SRC_ALPHA)
    return rs


def _floor(half, y):
    """A floor of two triangles, 64-byte vertices, facing up."""
    v = np.zeros((4, 16), np.float32)
    v[:, 0:3] = [[-half, y, half], [half, y, half], [half, y, -half], [-half, y, -half]]
    v[:, 4:6] = [[0, 0], [4, 0], [4, 4], [0, 4]]
    v[:, 8:11] = (0, 1, 0)
    v[:, 12:15] = (1, 0, 0)
    return v, np.array([[0, 1, 2], [0, 2, 3]], np.int32)


def _ibl_textures(p, seed):
    irr, pref = scenes.ibl_maps(seed)
    ti = p.texture(cube=irr, wrap=S.WRAP_CLAMP_TO_EDGE)
    tp = p.texture(cube=pref[0], mip=True, wrap=S.WRAP_CLAMP_TO_EDGE)
    for lev in range(1, len(pref)):
        for face in range(6):
            tp.setLevelData(face, lev, pref[lev][face])
    return ti, tp


def _weights(rng):
    """A 24-64-64-3 network with the outputs around mid-grey."""
    w = [rng.uniform(-1, 1, (64, 24)) * math.sqrt(6 / 24), rng.uniform(-0.1, 0.1, 64),
         rng.uniform(-1, 1, (64, 64)) * math.sqrt(6 / 64), rng.uniform(-0.1, 0.1, 64),
         rng.uniform(-1, 1, (3, 64)) * math.sqrt(6 / 64) * 0.3, np.full(3, 0.5)]
    return np.concatenate([np.ravel(x) for x in w]).astype(np.float32)


def _prepare_mesh(c, rng):
    p = Program()
    w, h = c["width"], c["height"]
    verts, idx = _blob(c["freq"], rng)
    vao = p.mesh(verts, idx)
    albedo, normal, mr = _pbr_images(c["tex"], rng)
    ta = p.texture(albedo, mip=True, layout=c["layout"])
    color = p.texture(width=w, height=h, usage=S.USAGE_COLOR | S.USAGE_SAMPLER, msaa=c["msaa"], wrap=S.WRAP_CLAMP_TO_EDGE)
    depth = p.texture(width=w, height=h, fmt=S.FMT_FLOAT32, usage=S.USAGE_DEPTH, msaa=c["msaa"], filt=S.FILTER_NEAREST,
                      wrap=S.WRAP_CLAMP_TO_EDGE)
    eye, light = _eye(rng, 2.7), tuple(np.array(_eye(rng, 2.5)) + (0.0, 2.5, 0.0))
    rz = c["shading"] != "blinn"  # the PBR frames use reversed depth
    func, far = (S.DEPTH_GREATER, 0.0) if rz else (S.DEPTH_LESS, 1.0)
    ident = np.eye(4)
    view = scenes.look_at(eye, (0, 0, 0), (0, 1, 0))
    proj = scenes.projection(math.radians(60.0), w / h, 0.1, reverse_z=rz)
    scene_u = S.uniforms_scene((0.1, 0.1, 0.1), eye, light, (2.0, 2.0, 2.0))
    bias, shadow_map = np.eye(4), None
    if c["shadow"]:
        lview = scenes.look_at(light, (0, 0, 0), (0, 1, 0))
        lproj = scenes.projection(math.radians(60.0), 1.0, 0.1, reverse_z=rz)
        shadow_map = p.texture(width=c["shadow"], height=c["shadow"], fmt=S.FMT_FLOAT32,
                               usage=S.USAGE_DEPTH | S.USAGE_SAMPLER, filt=S.FILTER_NEAREST, wrap=S.WRAP_CLAMP_TO_BORDER)
        p.begin(p.target(depth=shadow_map), c["shadow"], c["shadow"], depth=far, clear_color=False)
        p.draw(vao, S.SHADING_BASIC, 0, _states(func), S.uniforms_model(ident, lproj @ lview, reverse_z=rz),
               material=S.uniforms_material(0, 0, 0))
        p.end()
        bias = np.array([[0.5, 0, 0, 0.5], [0, 0.5, 0, 0.5], [0, 0, 1, 0], [0, 0, 0, 1]]) @ lproj @ lview
    p.begin(p.target(color, depth), w, h, depth=far)
    model_u = S.uniforms_model(ident, proj @ view, bias if c["shadow"] else None, reverse_z=rz)
    if c["floor"]:
        fm = {"u_albedoMap": ta}
        if c["shadow"]:
            fm["u_shadowMap"] = shadow_map
        p.draw(p.mesh(*_floor(4.0, -1.3)), S.SHADING_BLINN_PHONG, S.DEF_ALBEDO, _states(func, cull=False), model_u, scene_u,
               S.uniforms_material(1, 0, 1 if c["shadow"] else 0, 1.0, 0.3, (1, 1, 1, 1)), fm)
    if c["shading"] == "blinn":
        smp = {"u_albedoMap": ta}
        if c["shadow"]:
            smp["u_shadowMap"] = shadow_map
        p.draw(vao, S.SHADING_BLINN_PHONG, S.DEF_ALBEDO, _states(func), model_u, scene_u,
               S.uniforms_material(1, 0, 1 if c["shadow"] else 0, 1.0, 0.5, (1, 1, 1, 1)), smp)
    else:
        ti, tp = _ibl_textures(p, int(rng.integers(1 << 20)))
        tn, tm = p.texture(normal, mip=True, layout=c["layout"]), p.texture(mr, mip=True, layout=c["layout"])
        learned = c["shading"] == "neural"
        if learned:
            p.r.neural_set_weights(_weights(rng))
        p.draw(vao, S.SHADING_NEURAL_PBR if learned else S.SHADING_PBR, S.DEF_ALBEDO | S.DEF_NORMAL | S.DEF_METALROUGH,
               _states(func), model_u, scene_u, S.uniforms_material(0 if learned else 1, 1, 0, 1.0, 0.5, (1, 1, 1, 1)),
               {"u_albedoMap": ta, "u_normalMap": tn, "u_metalRoughnessMap": tm, "u_irradianceMap": ti,
                "u_prefilterMap": tp})
    if c["translucent"]:
        tv, tidx = _unit_sphere(max(4, c["freq"] // 7))
        tv = tv.copy()
        tv[:, 0:3] *= 0.35
        right, up = view[0, :3], view[1, :3]
        at = np.asarray(eye) * (1.25 / 2.7) + 0.4 * right - 0.25 * up
        tm4 = _translate(*at)
        mu = S.uniforms_model(tm4, proj @ view @ tm4, reverse_z=rz)
        if c["shading"] == "blinn":
            p.draw(p.mesh(tv, tidx), S.SHADING_BLINN_PHONG, 0, _states(func, blend=True), mu, scene_u,
                   S.uniforms_material(1, 0, 0, 1.0, 0.5, (0.2, 0.6, 1.0, 0.5)))
        else:
            p.draw(p.mesh(tv, tidx), S.SHADING_PBR, 0, _states(func, blend=True), mu, scene_u,
                   S.uniforms_material(1, 1, 0, 1.0, 0.5, (0.2, 0.6, 1.0, 0.5)),
                   {"u_irradianceMap": ti, "u_prefilterMap": tp})
    p.end()
    p.read(color)
    if c["depth"]:
        p.read(depth)
    return p


def _prepare_viewer(c, rng):
    p = Program()
    w, h = c["width"], c["height"]
    ti, tp = _ibl_textures(p, int(rng.integers(1 << 20)))
    sky = p.texture(cube=scenes.env_cube_faces(c["sky"], int(rng.integers(1 << 20))), mip=True, wrap=S.WRAP_CLAMP_TO_EDGE)
    color = p.texture(width=w, height=h, usage=S.USAGE_COLOR | S.USAGE_SAMPLER, wrap=S.WRAP_CLAMP_TO_EDGE)
    depth = p.texture(width=w, height=h, fmt=S.FMT_FLOAT32, usage=S.USAGE_DEPTH, filt=S.FILTER_NEAREST)
    eye = np.asarray(_eye(rng, 4.2)) + (0.0, 1.5, 0.0)
    view = scenes.look_at(eye, (0, 0, 0), (0, 1, 0))
    proj = scenes.projection(math.radians(60.0), w / h, 0.1)
    scene_u = S.uniforms_scene((0.1, 0.1, 0.1), tuple(eye), (2.0, 3.0, 2.0), (2.0, 2.0, 2.0))
    p.begin(p.target(color, depth), w, h)
    grid = p.texture(_rgba(_u8(_noise(c["tex"], rng))), mip=True)
    p.draw(p.mesh(*_floor(6.0, -0.6)), S.SHADING_BLINN_PHONG, S.DEF_ALBEDO, _states(cull=False),
           S.uniforms_model(np.eye(4), proj @ view), scene_u, S.uniforms_material(1, 0, 0, 1.0, 0.3, (1, 1, 1, 1)),
           {"u_albedoMap": grid})
    side = math.ceil(math.sqrt(c["nodes"]))
    for k in range(c["nodes"]):
        f = max(3, int(round(c["freq"] * 2.0 ** rng.uniform(-1.0, 0.0))))
        vao = p.mesh(*_blob(f, rng, radius=0.42))
        at = _translate((k % side - 0.5 * (side - 1)) * 1.1, 0.0, (k // side - 0.5 * (side - 1)) * 1.1)
        mu = S.uniforms_model(at, proj @ view @ at)
        col = tuple(rng.uniform(0.2, 1.0, 3)) + (1.0,)
        if k % 2:
            p.draw(vao, S.SHADING_BLINN_PHONG, S.DEF_ALBEDO, _states(), mu, scene_u,
                   S.uniforms_material(1, 0, 0, 1.0, 0.5, col),
                   {"u_albedoMap": p.texture(_rgba(_u8(_noise(c["tex"], rng))), mip=True)})
        else:
            p.draw(vao, S.SHADING_PBR, 0, _states(), mu, scene_u, S.uniforms_material(1, 1, 0, 1.0, 0.5, col),
                   {"u_irradianceMap": ti, "u_prefilterMap": tp})
    axis = np.zeros((6, 16), np.float32)
    axis[1::2, 0:3] = np.eye(3) * 2.0
    lines = _states(S.DEPTH_LEQUAL, cull=False)
    lines.primitive_type = S.PRIM_LINE
    p.draw(p.mesh(axis, np.arange(6, dtype=np.int32)), S.SHADING_BASIC, 0, lines, S.uniforms_model(np.eye(4), proj @ view),
           material=S.uniforms_material(0, 0, 0, 1.0, 0.5, (0.9, 0.9, 0.2, 1.0)))
    cube_v, cube_i = scenes.cube_mesh()
    sky_states = S.RenderStates(depth_test=True, depth_mask=False, depth_func=S.DEPTH_LEQUAL)
    turn = np.eye(4)
    turn[:3, :3] = view[:3, :3]
    p.draw(p.mesh(cube_v, cube_i), S.SHADING_SKYBOX, 0, sky_states, S.uniforms_model(np.eye(4), proj @ turn),
           samplers={"u_cubeMap": sky})
    p.end()
    if not c["fxaa"]:
        p.read(color)
        return p
    out = p.texture(width=w, height=h, usage=S.USAGE_COLOR)
    quad = np.zeros((4, 16), np.float32)
    quad[:, 0:2] = [[1, -1], [-1, -1], [1, 1], [-1, 1]]
    quad[:, 4:6] = [[1, 0], [0, 0], [1, 1], [0, 1]]
    p.begin(p.target(out), w, h, clear_depth=False)
    p.draw(p.mesh(quad, np.array([[0, 1, 2], [1, 2, 3]], np.int32)), S.SHADING_FXAA, 0, S.RenderStates(),
           S.uniforms_model(np.eye(4), np.eye(4)), material=struct.pack("<2f", float(w), float(h)) + bytes(40),
           samplers={"u_screenTexture": color})
    p.end()
    p.read(out)
    return p


def _prepare_wire(c, rng):
    p = Program()
    w, h = c["width"], c["height"]
    color = p.texture(width=w, height=h, usage=S.USAGE_COLOR, msaa=c["msaa"])
    depth = p.texture(width=w, height=h, fmt=S.FMT_FLOAT32, usage=S.USAGE_DEPTH, msaa=c["msaa"], filt=S.FILTER_NEAREST)
    verts, idx = _blob(c["freq"], rng)
    vao = p.mesh(verts, idx)
    eye = _eye(rng, 2.6)
    mvp = scenes.projection(math.radians(60.0), w / h, 0.1) @ scenes.look_at(eye, (0, 0, 0), (0, 1, 0))
    scene_u = S.uniforms_scene((0.2, 0.2, 0.2), eye, (1.0, 2.0, 1.5), (0.9, 0.9, 0.9))
    p.begin(p.target(color, depth), w, h)
    p.draw(vao, S.SHADING_BLINN_PHONG, 0, _states(), S.uniforms_model(np.eye(4), mvp), scene_u,
           S.uniforms_material(1, 0, 0, 1.0, 0.5, (0.6, 0.6, 0.7, 1.0)))

    def basic(v, prim, mode, col, blend=False, width=1.0, size=1.0, scale=1.0):
        rs = _states(S.DEPTH_LEQUAL, cull=False, blend=blend)
        rs.primitive_type, rs.polygon_mode, rs.line_width = prim, mode, width
        m = np.diag([scale, scale, scale, 1.0])
        p.draw(v, S.SHADING_BASIC, 0, rs, S.uniforms_model(m, mvp @ m),
               material=S.uniforms_material(0, 0, 0, size, 0.5, col))

    basic(vao, S.PRIM_TRIANGLE, S.POLY_LINE, (0.9, 0.9, 0.2, 0.6), blend=True, scale=1.01)
    cloud = np.zeros((len(verts), 16), np.float32)
    cloud[:, 0:3] = verts[:, 0:3] * rng.uniform(1.02, 1.2, (len(verts), 1))
    basic(p.mesh(cloud, np.arange(len(cloud), dtype=np.int32)), S.PRIM_POINT, S.POLY_FILL, (0.2, 0.7, 1.0, 1.0),
          size=c["point_size"])
    seg = np.zeros((128, 16), np.float32)
    seg[:, 0:3] = rng.uniform(-1.4, 1.4, (128, 3))
    basic(p.mesh(seg, np.arange(128, dtype=np.int32)), S.PRIM_LINE, S.POLY_FILL, (1.0, 0.3, 0.3, 1.0),
          width=c["line_width"])
    p.end()
    p.read(color)
    return p


def _prepare_stress(c, rng):
    p = Program()
    w, h = c["width"], c["height"]
    v, i = scenes.random_triangles(c["n"], w, h, int(rng.integers(1 << 30)), 0.25, 16.0, 0.0, 1.0, big=c["big"])
    color = p.texture(width=w, height=h, usage=S.USAGE_COLOR, msaa=c["msaa"])
    depth = p.texture(width=w, height=h, fmt=S.FMT_FLOAT32, usage=S.USAGE_DEPTH, msaa=c["msaa"], filt=S.FILTER_NEAREST)
    p.begin(p.target(color, depth), w, h, color=(0.0, 0.0, 0.0, 0.0))
    p.draw(p.mesh(v, i), S.SHADING_VERTEX_COLOR, 0, _states(cull=False), S.uniforms_model(np.eye(4), np.eye(4)))
    p.end()
    p.read(color)
    return p


def _view_sizes(c):
    """A third of the views each at the full size, a half and a quarter of it."""
    return [max(8, c["size"] >> (v % 3)) for v in range(c["views"])]


def _scene_freqs(c):
    lo, n = 1000.0, c["scenes"]
    return [max(1, int(round(math.sqrt(lo * (c["tri_hi"] / lo) ** (k / max(1, n - 1)) / 20.0)))) for k in range(n)]


def _prepare_views(c, rng):
    p = Program()
    meshes = [p.mesh(*_blob(f, rng)) for f in _scene_freqs(c)]
    texs = [p.texture(_rgba(_u8(_noise(c["tex"], rng))), mip=True, layout=1) for _ in meshes]
    proj = scenes.projection(math.radians(60.0), 1.0, 0.1)
    for v, size in enumerate(_view_sizes(c)):
        color = p.texture(width=size, height=size, usage=S.USAGE_COLOR | S.USAGE_SAMPLER)
        depth = p.texture(width=size, height=size, fmt=S.FMT_FLOAT32, usage=S.USAGE_DEPTH, filt=S.FILTER_NEAREST)
        eye = _eye(rng, 3.0)
        view = scenes.look_at(eye, (0, 0, 0), (0, 1, 0))
        k = v % len(meshes)
        p.begin(p.target(color, depth), size, size, color=(0.05, 0.05, 0.08, 1.0))
        p.draw(meshes[k], S.SHADING_BLINN_PHONG, S.DEF_ALBEDO, _states(), S.uniforms_model(np.eye(4), proj @ view),
               S.uniforms_scene((0.15, 0.15, 0.15), eye, (2.0, 3.0, 4.0), (1.0, 1.0, 1.0)),
               S.uniforms_material(1, 0, 0, 1.0, 0.5, (1, 1, 1, 1)), {"u_albedoMap": texs[k]})
        p.end()
        p.read(color)
    # recorded once, replayed every pass; the configuration the autotuner picks for such batches
    p.r.beginBatch()
    for fn, args in p.frame:
        fn(*args)
    p.batch = p.r.endBatch(32, 2)
    p.recorded, p.frame = p.frame, [(p.batch.run, ())]  # the batch's resources live as long as it does
    return p


_FACES = [((1, 0, 0), (0, -1, 0)), ((-1, 0, 0), (0, -1, 0)), ((0, 1, 0), (0, 0, 1)), ((0, -1, 0), (0, 0, -1)),
          ((0, 0, 1), (0, -1, 0)), ((0, 0, -1), (0, -1, 0))]


def _ibl_levels(c):
    return min(5, int(math.log2(c["pref"])) + 1)


def _prepare_ibl(c, rng):
    p = Program()
    env = p.texture(cube=scenes.env_cube_faces(c["src"], int(rng.integers(1 << 20))), mip=True, wrap=S.WRAP_CLAMP_TO_EDGE)
    usage = S.USAGE_COLOR | S.USAGE_SAMPLER
    irr = p.texture(width=c["irr"], height=c["irr"], is_cube=True, usage=usage, wrap=S.WRAP_CLAMP_TO_EDGE)
    pref = p.texture(width=c["pref"], height=c["pref"], is_cube=True, usage=usage, mip=True, wrap=S.WRAP_CLAMP_TO_EDGE)
    vao = p.mesh(*scenes.cube_mesh())
    proj = scenes.projection(math.radians(90.0), 1.0, 0.1)
    jobs = [(S.SHADING_IBL_IRRADIANCE, irr, 0, c["irr"], bytes(48))]
    n = _ibl_levels(c)
    for lev in range(n):
        mat = struct.pack("<2f", float(c["src"]), lev / max(1, n - 1)) + bytes(40)
        jobs.append((S.SHADING_IBL_PREFILTER, pref, lev, max(1, c["pref"] >> lev), mat))
    for shading, tex, lev, size, mat in jobs:
        for face, (center, up) in enumerate(_FACES):
            turn = np.eye(4)
            turn[:3, :3] = scenes.look_at((0, 0, 0), center, up)[:3, :3]
            p.begin(p.target(tex, face=face, level=lev), size, size, color=(0, 0, 0, 0), clear_depth=False)
            p.draw(vao, shading, 0, S.RenderStates(), S.uniforms_model(np.eye(4), proj @ turn), material=mat,
                   samplers={"u_cubeMap": env})
            p.end()
            p.read(tex, face, lev)
    return p


# the fields of a captured fragment's record that the network reads and is trained on
_N, _V, _ALBEDO, _ROUGH, _METAL, _AO, _TARGET, _PLAIN = 0, 3, 6, 10, 11, 12, 14, 17


def _records(n, rng):
    """Fragments as a capture of PBR draws records them: unit normals and view directions that face the viewer, texels,
    and a smooth colour for the network to learn."""
    r = np.zeros((n, RendererHIP.NN_RECORD_FLOATS), np.float32)
    nrm = rng.normal(size=(n, 3))
    v = rng.normal(size=(n, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    v *= np.where(np.sum(nrm * v, 1, keepdims=True) < 0, -1.0, 1.0)
    alb, rough, metal = rng.random((n, 3)), rng.uniform(0.05, 1, n), (rng.random(n) > 0.6) * 0.9 + 0.05
    r[:, _N:_N + 3], r[:, _V:_V + 3], r[:, _ALBEDO:_ALBEDO + 3], r[:, _ALBEDO + 3] = nrm, v, alb, 1.0
    r[:, _ROUGH], r[:, _METAL], r[:, _AO] = rough, metal, 1.0
    nv = np.sum(nrm * v, 1)
    refl = 2 * nv[:, None] * nrm - v
    lit = 0.5 + 0.3 * nrm[:, 1:2] + 0.2 * (1 - rough[:, None]) * np.sin(np.pi * refl)
    r[:, _TARGET:_TARGET + 3] = np.clip(alb * lit * (1 - 0.5 * metal[:, None]) + 0.1 * (1 - nv[:, None]), 0, 1)
    r[:, _PLAIN:_PLAIN + 3] = np.floor(r[:, _TARGET:_TARGET + 3] * 255) / 255
    r[:, 22:25], r[:, 25:28], r[:, 28], r[:, 29] = nrm, alb, rough, metal
    return r


_LR = (1e-3, 1e-4)


def _prepare_network(c, rng):
    p = Program()
    p.records, p.weights = _records(c["records"], rng), _weights(rng)
    p.seed = int(rng.integers(1, 1 << 16))
    p.r.neural_records(c["records"])
    p.r.neural_write_records(0, p.records)
    p.r.neural_set_weights(p.weights)
    return p


_PREPARE = {"mesh": _prepare_mesh, "viewer": _prepare_viewer, "wire": _prepare_wire, "stress": _prepare_stress,
            "views": _prepare_views, "ibl": _prepare_ibl, "train": _prepare_network, "evaluate": _prepare_network}


def prepare(case, seed):
    p = _PREPARE[case["kind"]](case, np.random.default_rng(seed))
    p.case = case
    p.r.waitIdle()
    return p


def run(p):
    c, r = p.case, p.r
    if c["kind"] == "train":
        # a training run starts from its weights (and fresh Adam state) and ends with the trained ones
        r.neural_set_weights(p.weights)
        losses = r.neural_train(0, c["records"], c["steps"], batch=c["batch"], lr_start=_LR[0], lr_end=_LR[1], seed=p.seed)
        return {"weights": r.neural_get_weights(), "losses": losses}
    if c["kind"] == "evaluate":
        net, plain, rgb = r.neural_evaluate(0, c["records"], outputs=True)
        grad, loss = r.neural_gradient(0, c["records"])
        return {"rgb": rgb, "mean": net["mean"], "max": net["max"], "p99": net["p99"], "plain": plain["mean"],
                "gradient": grad, "loss": loss}
    return p.run()


# ----------------------------------------------------------------------------- what a pass cannot do without


def _sphere(freq):
    return 10 * freq * freq + 2, 20 * freq * freq


def work(case):
    """Every vertex, index, record and source texel read once and every image read back written once; flops are the
    vertices' transforms, the shaders of about the visible pixels (each once per pixel, not per sample) and the network."""
    c = case
    kind = c["kind"]
    if kind in ("mesh", "viewer", "wire"):
        px = c["width"] * c["height"]
    if kind == "mesh":
        v, t = _sphere(c["freq"])
        frag = 0.35 * px  # the sphere's share of the image
        maps = {"blinn": 1, "pbr": 3, "neural": 3}[c["shading"]]
        texels = min(maps * 1.33 * c["tex"] ** 2, maps * 4.0 * frag)
        b = v * 64 + t * 12 + texels * 4 + px * 4 * (2 if c["depth"] else 1)
        per = {"blinn": 150, "pbr": 500, "neural": 12_000}[c["shading"]]
        f = v * 120 + t * 60 + frag * per
        if c["shadow"]:
            b, f = b + c["shadow"] ** 2 * 4, f + v * 60 + t * 60
        if c["floor"]:
            f += 0.4 * px * 200
        if c["translucent"]:
            f += 0.1 * px * 500
        return {"bytes": b, "flops": f}
    if kind == "viewer":
        v, t = _sphere(max(3, int(c["freq"] * 0.72)))
        n = c["nodes"]
        b = n * (v * 64 + t * 12) + px * 4 + (n // 2 + 1) * min(1.33 * c["tex"] ** 2, px / n) * 4 + min(6 * c["sky"] ** 2, px) * 4
        return {"bytes": b, "flops": n * (v * 120 + t * 60) + px * (300 + (100 if c["fxaa"] else 0))}
    if kind == "wire":
        v, t = _sphere(c["freq"])
        return {"bytes": 3 * v * 64 + t * 12 + px * 4, "flops": v * 200 + t * 120 + px * 50.0}
    if kind == "stress":
        t = c["n"] + c["big"]
        px = c["width"] * c["height"]
        return {"bytes": t * (3 * 32 + 12) + px * 4, "flops": t * 3 * 40 + t * 60 + px * 60.0}
    if kind == "views":
        freqs = _scene_freqs(c)
        px = sum(s * s for s in _view_sizes(c))
        vt = [_sphere(freqs[v % len(freqs)]) for v in range(c["views"])]
        b = sum(_sphere(f)[0] * 64 + _sphere(f)[1] * 12 for f in freqs) + len(freqs) * 1.33 * c["tex"] ** 2 * 4 + px * 4
        return {"bytes": b, "flops": sum(v * 120 + t * 60 for v, t in vt) + 0.3 * px * 150}
    if kind == "ibl":
        px = [6 * max(1, c["pref"] >> k) ** 2 for k in range(_ibl_levels(c))]
        irr = 6 * c["irr"] ** 2
        # one environment sample is about 60 operations; the shaders take 2,500 and 1,024 of them for a texel
        return {"bytes": 4 * (6 * 1.33 * c["src"] ** 2 + irr + sum(px)), "flops": 60.0 * (2500 * irr + 1024 * sum(px))}
    net = 2 * (24 * 64 + 64 * 64 + 64 * 3)
    if kind == "train":
        n = c["steps"] * c["batch"]
        return {"bytes": min(n, c["records"]) * 64.0 + 5955 * 4 * 2, "flops": 3.0 * net * n}
    return {"bytes": c["records"] * (96.0 + 12.0), "flops": 4.0 * net * c["records"]}


def tolerance(case):
    """Images are whole bytes (and depths whose every bit the tests pin). The network's operands are 16-bit and its sums
    32-bit: with the same rounded operands, sums in 32 and in 64 bits differ by 8e-7 in the trained weights and losses
    after 64 steps, and by 7e-6 in the outputs, where a hidden value next to a rounding boundary rounds the other way."""
    if case["kind"] == "train":
        return {"rel": 1e-5}
    if case["kind"] == "evaluate":
        return {"rel": 3e-5}
    return "exact"


def _features64(r):
    r = r.astype(np.float64)
    nrm, v = r[:, _N:_N + 3], r[:, _V:_V + 3]
    d = np.sum(nrm * v, 1, keepdims=True)
    refl = 2 * d * nrm - v
    a = np.pi * refl
    return np.concatenate([nrm, v, np.maximum(d, 0), r[:, [_ROUGH]], r[:, [_METAL]], r[:, _ALBEDO:_ALBEDO + 3], refl,
                           np.sin(a), np.sin(2 * a), np.sin(4 * a)], 1)


def _split(w):
    w = torch.from_numpy(w.astype(np.float64)) if isinstance(w, np.ndarray) else w
    return torch.split(w, [64 * 24, 64, 64 * 64, 64, 3 * 64, 3])


def _network64(w, x):
    w1, b1, w2, b2, w3, b3 = _split(w)
    h = torch.relu(x @ w1.view(64, 24).T + b1)
    h = torch.relu(h @ w2.view(64, 64).T + b2)
    return h @ w3.view(3, 64).T + b3


def exact(case, seed):
    """The network in 64 bits, without the 16-bit operands; None for images, whose bytes follow from the reference's
    own 32-bit arithmetic, and for training, whose records are drawn by the library."""
    if case["kind"] != "evaluate":
        return None
    rng = np.random.default_rng(seed)
    rec, w = _records(case["records"], rng), _weights(rng)
    x = torch.from_numpy(_features64(rec))
    t = torch.from_numpy(rec[:, _TARGET:_TARGET + 3].astype(np.float64))
    plain = rec[:, _PLAIN:_PLAIN + 3].astype(np.float64)
    wt = torch.from_numpy(w.astype(np.float64)).requires_grad_(True)
    y = _network64(wt, x)
    loss = ((y - t) ** 2).sum()
    loss.backward()
    err = (y.detach().clamp(0, 1) - t).abs().numpy() * 255
    return {"rgb": y.detach().numpy(), "mean": float(err.mean()), "max": None, "p99": None,
            "plain": float(np.abs(plain - t.numpy()).mean() * 255), "gradient": wt.grad.numpy(), "loss": float(loss.detach())}
