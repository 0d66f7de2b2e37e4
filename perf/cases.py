"""The work a renderer that binds this library has it do, as cases that can be timed and checked.

Five kinds of pass, each through the public entry points:

  frame     one engine tick: rsy_update, rsy_render, rsy_synchronize, the outputs read in place on the device
  replay    the same views rendered repeatedly: rsy_render_graph
  loop      a tick up to the output stage: update, render, rsy_present, the RGBA16F draw image read back
  train     rsy_neural_train, the loss history and the trained parameters read back (a checkpoint)
  evaluate  rsy_neural_evaluate: export for inference and the PSNR gate over every texel
  load      rsy_set_materials: BC7 images with their chains and uncompressed ones whose chains are built

Scenes are the library's seeded synthetic ones (rsy_scene_generate); every input follows from the seed.  `exact`
renders the same frame in plain torch: the fixed-point raster rules in the FP32 / int64 arithmetic they are stated in
(they decide which triangle a pixel shows), everything that is shaded in FP64.
"""
import ctypes as C
import math

import numpy as np
import torch

import rosy_amd
from rosy_amd import abi, lib


# --------------------------------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------------------------------

def frame_case(name, kind="frame", workload=1, triangles=262144, width=1920, height=1080, shadow=2048, materials=16,
               texture=1024, samples=1, shade="plain", mips=False, translucent=0, replays=0):
    return {"name": name, "kind": kind, "workload": workload, "triangles": triangles, "width": width, "height": height,
            "shadow": shadow, "materials": materials, "texture": texture, "samples": samples, "shade": shade,
            "mips": mips, "translucent": translucent, "replays": replays}


def listed():
    return [
        # an asset viewer: one small object in a small window, where launches and latency are the frame
        frame_case("viewer_360p", workload=0, triangles=2048, width=640, height=360, shadow=1024, materials=1),
        # the ordinary frame of the engine's level: plain material maps
        frame_case("level_1080p"),
        # the benchmark's frame: material maps replaced by the decoder
        frame_case("decoder_1080p", workload=3, shade="fp16"),
        # the reference's own main pass: 4 samples per pixel, every image with its mip chain, a laptop window
        frame_case("multisample_mips_768p", width=1366, height=768, samples=4, mips=True),
        # translucent and masked surfaces over the opaque frame
        frame_case("blended_1080p", workload=3, translucent=8),
        # a large level with cascaded shadow maps: five views in one frame
        frame_case("cascades_1440p", workload=2, triangles=1048576, width=2560, height=1440),
        # the largest: four cameras (4K to 360p) and four cascades, decoder weights stored in FP8
        frame_case("cameras_4k", workload=4, triangles=2097152, width=3840, height=2160, shade="fp8"),
        # the same views over and over (a turntable, a capture server): the captured graph
        frame_case("replay_1080p", kind="replay", workload=3, shade="fp16", replays=32),
        # a tick of the engine's loop up to the draw image on the host, 4 samples, a 900p window
        frame_case("loop_900p", kind="loop", width=1600, height=900, samples=4),
        # the decoder fitted to a scene's materials (the default batch of 65,536 samples)
        {"name": "train_decoder", "kind": "train", "materials": 16, "texture": 1024, "latent": 128, "batch": 65536,
         "region": 16, "steps": 256},
        # the gate after training: every texel of every material decoded and compared with its maps
        {"name": "evaluate_decoder", "kind": "evaluate", "materials": 32, "texture": 1024, "latent": 256,
         "weights": "fp16"},
        # a level load: 12 BC7 images with their chains, 12 uncompressed ones whose chains are built
        {"name": "load_images", "kind": "load", "images": 24, "width": 1024, "height": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 7 + ["replay", "loop", "train", "evaluate", "load"])
    if kind in ("frame", "replay", "loop"):
        workload = rng.choice([1, 1, 2, 3, 3, 4] if kind == "frame" else [1, 3])
        many = workload in (2, 4)
        width = rng.randint(320, 2560)
        height = max(200, min(1440, int(width * rng.uniform(0.5, 0.75))))
        samples = rng.choice([1, 1, 4])
        shade = rng.choice(["plain", "plain", "fp16", "fp8"])
        translucent = rng.choice([0, 0, 2, 5]) if workload in (1, 3) and shade == "plain" else 0
        return {"kind": kind, "workload": workload,
                "triangles": _log_int(rng, 20000, 700000 if many else 400000), "width": width, "height": height,
                "shadow": rng.choice([512, 1000, 1024, 2048]), "materials": rng.randint(6, 16),
                "texture": rng.choice([256, 512, 1024]), "samples": samples, "shade": shade,
                "mips": shade == "plain" and rng.random() < 0.4, "translucent": translucent,
                "replays": rng.randint(4, 32) if kind == "replay" else 0}
    if kind == "train":
        return {"kind": kind, "materials": rng.randint(2, 16), "texture": rng.choice([256, 512, 1024]),
                "latent": rng.choice([32, 64, 128]), "batch": 256 * _log_int(rng, 16, 256),
                "region": rng.choice([8, 16, 32]), "steps": _log_int(rng, 16, 200)}
    if kind == "evaluate":
        return {"kind": kind, "materials": rng.randint(2, 24), "texture": rng.choice([256, 500, 512, 1024]),
                "latent": rng.choice([64, 128, 256]), "weights": rng.choice(["fp16", "fp8"])}
    return {"kind": kind, "images": 2 * rng.randint(1, 10), "width": _log_int(rng, 100, 1024),
            "height": _log_int(rng, 100, 1024)}


def work(case):
    """What a pass cannot do without: geometry in, every view's outputs written, the visible maps left out (how much of
    them a frame needs depends on the view); for the decoder its samples' arithmetic and the texels they read."""
    if case["kind"] in ("frame", "replay", "loop"):
        cams, cascades = _extents(case)
        tris, px = case["triangles"], sum(w * h for w, h in cams)
        views = len(cams) + len(cascades)
        nbytes = 24 * tris + sum(4 * s * s for s in cascades) + (8 * case["samples"] + 16) * px
        flops = views * 100 * tris + 300 * px
        if case["kind"] == "loop":
            nbytes += 12 * px
        n = 1 + case["replays"]
        return {"bytes": n * nbytes, "flops": n * flops}
    if case["kind"] == "train":
        n = case["steps"] * case["batch"]
        return {"bytes": 32 * n + 2 * 24 * 4 * case["materials"] * case["latent"] ** 2, "flops": 3 * 1088 * n}
    if case["kind"] == "evaluate":
        n = case["materials"] * case["texture"] ** 2
        return {"bytes": 8 * n + 48 * case["materials"] * case["latent"] ** 2, "flops": 1088 * n}
    texels = case["images"] * case["width"] * case["height"] * 4 / 3
    return {"bytes": texels * (0.5 * 1 + 0.5 * 3 + 3.5), "flops": 40 * texels}


def _extents(case):
    cams = [(case["width"], case["height"])]
    if case["workload"] == 4:
        cams += [(1920, 1080), (1280, 720), (640, 360)]
    return cams, [case["shadow"]] * (4 if case["workload"] in (2, 4) else 1)


# --------------------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------------------

def _scene(case, seed):
    return rosy_amd.Scene(case["workload"], seed=1 + seed % 1000003, width=case["width"], height=case["height"],
                          shadow_size=case["shadow"], total_triangles=case["triangles"],
                          n_materials=case["materials"], texture_size=case["texture"],
                          texture_mips=int(case["mips"]), n_translucent=case["translucent"])


def _material_scene(case, seed):
    """A small scene whose materials are the ones a decoder is fitted to."""
    return rosy_amd.Scene(3, seed=1 + seed % 1000003, width=64, height=64, shadow_size=64, total_triangles=30000,
                          n_materials=case["materials"], texture_size=case["texture"])


WEIGHTS = {"fp16": 0, "fp8": 1}  # rsy_neural_weights


def _levels(w, h):
    return max(w, h).bit_length()


def _image_data(case, seed):
    """Pairs of images: BC7 blocks of every mode with a whole chain, and RGBA8 / RG8 texels of level 0."""
    rng = np.random.default_rng(seed)
    w, h, descs = case["width"], case["height"], []
    blocks = sum(-(-max(1, w >> l) // 4) * -(-max(1, h >> l) // 4) for l in range(_levels(w, h)))
    for i in range(case["images"]):
        if i % 2 == 0:
            data = rng.integers(0, 256, (blocks, 16), dtype=np.uint8)
            mode = rng.integers(0, 8, blocks)
            data[:, 0] = (1 << mode) | (data[:, 0] & (0xFE << mode) & 0xFF)
            fmt, levels = (abi.TEX_BC7_SRGB if i % 4 == 0 else abi.TEX_BC7_UNORM), _levels(w, h)
        else:
            fmt = (abi.TEX_RGBA8_SRGB, abi.TEX_RG8_UNORM, abi.TEX_RGBA8_SRGB, abi.TEX_RG8_SRGB)[(i // 2) % 4]
            channels = 2 if fmt in (abi.TEX_RG8_UNORM, abi.TEX_RG8_SRGB) else 4
            data, levels = rng.integers(0, 256, (h, w, channels), dtype=np.uint8), abi.MIPS_BUILD
            if channels == 4 and (i // 2) % 4 == 0:
                data[..., 3] = 255  # an opaque albedo map
        descs.append((fmt, levels, data))
    return descs


def prepare(case, seed):
    r = rosy_amd.Renderer(device=0)
    if case["kind"] == "load":
        data = _image_data(case, seed)
        descs = (abi.TextureDesc * len(data))()
        for i, (fmt, levels, pixels) in enumerate(data):
            descs[i] = abi.TextureDesc(case["width"], case["height"], fmt, levels, pixels.ctypes.data)
        # read back afterwards: the chains of the first BC7 image and of the first built one
        back = []
        for i in (0, 1):
            channels = 2 if data[i][0] in (abi.TEX_RG8_UNORM, abi.TEX_RG8_SRGB) else 4
            back += [(i, l, np.zeros(max(1, case["width"] >> l) * max(1, case["height"] >> l) * channels, np.uint8))
                     for l in range(_levels(case["width"], case["height"]))]
        return {"kind": "load", "renderer": r, "data": data, "descs": descs, "back": back}
    if case["kind"] in ("train", "evaluate"):
        scene = _material_scene(case, seed)
        r.load(scene)
        more = {"batch": case["batch"], "region": case["region"], "decay_steps": 20000} if case["kind"] == "train" else \
            {"weights": WEIGHTS[case["weights"]]}
        r.neural_init(latent_size=case["latent"], seed=1 + seed % 65521, **more)
        return {"kind": case["kind"], "renderer": r, "scene": scene, "steps": case.get("steps", 0)}
    scene = _scene(case, seed)
    r.load(scene)
    rs = abi.RasterState()
    C.memmove(C.byref(rs), C.byref(scene.s.raster_state), C.sizeof(rs))
    rs.msaa_samples = case["samples"]
    r.update(scene.s.scene_data, rs)
    if case["shade"] != "plain":  # latents from the maps: the decoder that training starts from
        r.neural_init(latent_size=min(256, case["texture"]), weights=WEIGHTS[case["shade"]])
        r.neural_evaluate()
    frame = scene.frame_desc(abi.SHADE_PLAIN if case["shade"] == "plain" else abi.SHADE_NEURAL)
    state = {"kind": case["kind"], "renderer": r, "scene": scene, "raster": rs, "frame": frame, "samples": case["samples"],
             "replays": case["replays"], "seen": {}}
    if case["kind"] == "loop":
        state["draw"] = np.zeros((case["height"], case["width"], 4), np.float16)
    return state


# --------------------------------------------------------------------------------------------------
# A pass
# --------------------------------------------------------------------------------------------------

class _DeviceArray:
    """A device buffer of the library as the array interface torch reads (no copy).  A tensor keeps the object it was
    made from, and this one keeps the renderer whose context owns the buffer."""

    def __init__(self, owner, address, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape, "typestr": kind, "version": 2}


def _outputs(state):
    """The frame's visibility words and colours where the library keeps them."""
    r, out, vis, colour = state["renderer"], {}, C.c_void_p(), C.c_void_p()
    for i, (w, h) in enumerate(r.views):
        rosy_amd._check(lib().rsy_get_device_outputs(r.ctx, i, C.byref(vis), C.byref(colour)),
                        "rsy_get_device_outputs", r.ctx)
        key = (i, vis.value, colour.value)
        if key not in state["seen"]:
            planes = (h, w) if state["samples"] == 1 else (4, h, w)
            state["seen"][key] = (torch.as_tensor(_DeviceArray(r, vis.value, planes, "<i8"), device="cuda"),
                                  torch.as_tensor(_DeviceArray(r, colour.value, (h, w, 4), "<f4"), device="cuda"))
        out[f"visibility{i}"], out[f"colour{i}"] = state["seen"][key]
    return out


def run(state):
    r, kind = state["renderer"], state["kind"]
    if kind == "load":
        d = state["descs"]
        rosy_amd._check(lib().rsy_set_materials(r.ctx, None, 0, d, len(d), None, 0), "rsy_set_materials", r.ctx)
        for i, level, out in state["back"]:
            rosy_amd._check(lib().rsy_read_texture(r.ctx, i, level, out.ctypes.data, out.size), "rsy_read_texture", r.ctx)
        return {f"image{i}_level{level}": out for i, level, out in state["back"]}
    if kind == "train":
        loss = r.neural_train(state["steps"])
        latents, mlp = r.neural_params()
        return {"loss": loss, "latents": latents, "mlp": mlp}
    if kind == "evaluate":
        return {"psnr": r.neural_evaluate()}
    r.update(state["scene"].s.scene_data, state["raster"])
    if kind == "replay":
        r.render_graph(state["frame"], state["replays"])
        return _outputs(state)
    r.render(state["frame"])
    if kind == "loop":
        w, h = r.views[0]
        rosy_amd._check(lib().rsy_present(r.ctx, 0, w, h), "rsy_present", r.ctx)
        rosy_amd._check(lib().rsy_read_draw_image(r.ctx, state["draw"].ctypes.data, w * h), "rsy_read_draw_image", r.ctx)
        return {"draw_image": state["draw"]}
    r.synchronize()
    return _outputs(state)


# --------------------------------------------------------------------------------------------------
# The same in plain torch: FP64, apart from the raster's own fixed-point rules
# --------------------------------------------------------------------------------------------------

F64, F32, I64 = torch.float64, torch.float32, torch.int64
SAMPLES = ((0.375, 0.125), (0.875, 0.375), (0.125, 0.625), (0.625, 0.875))
PIECE = 1 << 20  # pixels shaded at a time


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _fma(a, b, c):
    """FP32 fused multiply-add: the product of two FP32 values is exact in FP64."""
    return (a.to(F64) * b.to(F64) + c.to(F64)).to(F32)


def _matrix(values):
    return torch.tensor(list(values), dtype=F32, device=_device())


class _Level:
    """A scene's arrays on the device."""

    def __init__(self, scene):
        dev, s = _device(), scene.s
        v = scene.vertices
        self.vertex = {k: torch.from_numpy(np.ascontiguousarray(v[k])).to(dev) for k in v.dtype.names}
        self.index = torch.from_numpy(scene.indices.astype(np.int64)).to(dev)
        self.objects = torch.from_numpy(np.frombuffer(C.string_at(s.objects, 164 * s.n_objects), np.float32).copy()
                                        .reshape(-1, 41)).to(dev)
        self.scene, self.sd, self.bias = scene, s.scene_data, s.raster_state
        self.draws = [(d, s.meshes[d.mesh_index]) for d in scene.surfaces()]
        self.textures = [s.textures[i] for i in range(s.n_textures)]
        self.materials = [s.materials[i] for i in range(s.n_materials)]
        chosen = {"all": self.draws, "opaque": [d for d in self.draws if not d[0].blended],
                  "blended": [d for d in self.draws if d[0].blended]}
        self.lists = {}
        for name, draws in chosen.items():  # per triangle of the list: global vertices, object, material
            tri, obj, mat = [], [], []
            for d, m in draws:
                n = d.index_count // 3
                first, base = m.index_offset + d.start_index, m.vertex_buffer_offset // 64
                tri.append(self.index[first:first + 3 * n].reshape(-1, 3) + base)
                obj.append(torch.full((n,), d.graphics_object_index, dtype=I64, device=dev))
                mat.append(torch.full((n,), d.material_index, dtype=I64, device=dev))
            self.lists[name] = tuple(torch.cat(x) if x else torch.zeros((0, 3) if x is tri else (0,), dtype=I64, device=dev)
                                     for x in (tri, obj, mat))

    def clip_positions(self, name, vp):
        """FP32 clip positions (triangles, 3, 4) of a draw list: (vp W) p by chains of fused multiply-adds."""
        tri, obj, _ = self.lists[name]
        w = self.objects[:, :16].reshape(-1, 4, 4)  # [object, column, row]
        vp = _matrix(vp).reshape(4, 4)
        m = (vp[0] * w[:, :, 0:1]).to(F32)
        for k in range(1, 4):
            m = _fma(vp[k].expand_as(m), w[:, :, k:k + 1].expand_as(m), m)
        out = torch.empty(tri.shape[0], 3, 4, dtype=F32, device=tri.device)
        for at in range(0, tri.shape[0], PIECE):
            p, mm = self.vertex["vertex"][tri[at:at + PIECE]], m[obj[at:at + PIECE]][:, None]
            c = mm[:, :, 3].expand(-1, 3, 4)
            for k in range(3):
                c = _fma(mm[:, :, k].expand_as(c), p[:, :, k:k + 1].expand_as(c), c)
            out[at:at + PIECE] = c
        return out


def _planes(v):
    x, y, z, w = v.unbind(-1)
    return torch.stack([w - z, z, x + 4.0 * w, 4.0 * w - x, y + 4.0 * w, 4.0 * w - y], -1)


def _clip(tri):
    """FP32 Sutherland-Hodgman of one (3, 4) triangle, plane by plane, and the fan of what is left."""
    f = np.float32

    def dist(v, p):
        return (v[3] - v[2], v[2], v[0] + f(4) * v[3], f(4) * v[3] - v[0], v[1] + f(4) * v[3], f(4) * v[3] - v[1])[p]

    poly = list(tri)
    for p in range(6):
        out = []
        for i, cur in enumerate(poly):
            nxt = poly[(i + 1) % len(poly)]
            dc, dn = dist(cur, p), dist(nxt, p)
            if dc >= 0 and len(out) < 9:
                out.append(cur)
            if (dc >= 0) != (dn >= 0) and len(out) < 9:
                a, b, da, db = (cur, nxt, dc, dn) if dc >= 0 else (nxt, cur, dn, dc)
                out.append(a + (da / (da - db)) * (b - a))
        poly = out
        if len(poly) < 3:
            return []
    if not all(v[3] > 0 for v in poly):
        return []
    return [(poly[0], poly[k], poly[k + 1]) for k in range(1, len(poly) - 1)]


def _records(clip, width, height, cull, bias, samples):
    """Snapped, culled and set-up triangles: (X, Y int64, z0, dzdx, dzdy FP32, triangle, pixel box)."""
    d = _planes(clip)
    rejected = ((d < 0).sum(1) == 3).any(-1)
    inside = (d >= 0).all(-1).all(-1) & (clip[..., 3] > 0).all(-1)
    ids = torch.arange(clip.shape[0], device=clip.device)
    keep, cut = inside & ~rejected, ~inside & ~rejected
    fan, fan_id = [], []
    for t, i in zip(clip[cut].cpu().numpy(), ids[cut].tolist()):
        for piece in _clip(t):
            fan.append(np.stack(piece))
            fan_id.append(i)
    v, ids = clip[keep], ids[keep]
    if fan:
        v = torch.cat([v, torch.from_numpy(np.stack(fan)).to(v.device)])
        ids = torch.cat([ids, torch.tensor(fan_id, device=v.device)])
    ndc = v[..., :3] / v[..., 3:]
    half = torch.tensor([0.5 * width, 0.5 * height], dtype=F32, device=v.device).expand(*ndc.shape[:2], 2)
    xy = torch.round(_fma(ndc[..., :2], half, half) * 256.0).to(I64)
    X, Y, Z = xy[..., 0], xy[..., 1], ndc[..., 2]
    area = (X[:, 1] - X[:, 0]) * (Y[:, 2] - Y[:, 0]) - (X[:, 2] - X[:, 0]) * (Y[:, 1] - Y[:, 0])
    keep = (area < 0) if cull else (area != 0)
    X, Y, Z, ids, area = X[keep], Y[keep], Z[keep], ids[keep], area[keep]
    swap = torch.where((area > 0)[:, None], torch.tensor([0, 2, 1], device=v.device), torch.tensor([0, 1, 2], device=v.device))
    X, Y, Z = X.gather(1, swap), Y.gather(1, swap), Z.gather(1, swap)
    lo, hi = (32, 224) if samples == 4 else (128, 128)
    x0, x1 = ((X.amin(1) - hi + 255) >> 8).clamp(min=0), ((X.amax(1) - lo) >> 8).clamp(max=width - 1)
    y0, y1 = ((Y.amin(1) - hi + 255) >> 8).clamp(min=0), ((Y.amax(1) - lo) >> 8).clamp(max=height - 1)
    keep = (x0 <= x1) & (y0 <= y1)
    X, Y, Z, ids, x0, x1, y0, y1 = (t[keep] for t in (X, Y, Z, ids, x0, x1, y0, y1))
    fx1, fy1 = (X[:, 1] - X[:, 0]).to(F32), (Y[:, 1] - Y[:, 0]).to(F32)
    fx2, fy2 = (X[:, 2] - X[:, 0]).to(F32), (Y[:, 2] - Y[:, 0]).to(F32)
    dz1, dz2 = Z[:, 1] - Z[:, 0], Z[:, 2] - Z[:, 0]
    den = fx1 * fy2 - fx2 * fy1
    zero = torch.zeros_like(den)
    dzdx = torch.where(den != 0, (dz1 * fy2 - dz2 * fy1) / den, zero)
    dzdy = torch.where(den != 0, (dz2 * fx1 - dz1 * fx2) / den, zero)
    z0 = Z[:, 0]
    if bias is not None:
        m = torch.maximum(dzdx.abs(), dzdy.abs()) * 256.0
        e = ((Z.abs().amax(1).view(torch.int32) >> 23) & 0xFF).clamp(min=1) - 127
        o = m * bias.depth_bias_slope_factor + torch.ldexp(torch.ones_like(m), e - 23) * bias.depth_bias_constant
        limit = bias.depth_bias_clamp
        z0 = z0 + (o.clamp(max=limit) if limit > 0 else o.clamp(min=limit) if limit < 0 else o)
    return X, Y, z0, dzdx, dzdy, ids, x0, x1, y0, y1


def _fragments(records, sx, sy):
    """Pieces of (pixel x, y, depth bits, triangle) covered at the sample point (sx, sy) of a pixel (1/256)."""
    X, Y, z0, dzdx, dzdy, ids, x0, x1, y0, y1 = records
    w = x1 - x0 + 1
    n = w * (y1 - y0 + 1)
    ends = n.cumsum(0)
    k = 0
    while k < n.numel():
        done = int(ends[k - 1]) if k else 0
        j = max(k + 1, int(torch.searchsorted(ends, done + (24 << 20), right=True)))
        t = torch.repeat_interleave(torch.arange(k, j, device=X.device), n[k:j])
        o = torch.arange(t.numel(), device=X.device) - (ends[t] - n[t] - done)
        x, y = x0[t] + o % w[t], y0[t] + o // w[t]
        px, py = x * 256 + sx, y * 256 + sy
        covered = torch.ones_like(px, dtype=torch.bool)
        for a, b in ((0, 1), (1, 2), (2, 0)):
            A, B = Y[t, b] - Y[t, a], X[t, a] - X[t, b]
            e = A * (px - X[t, a]) + B * (py - Y[t, a])
            covered &= (e > 0) | ((e == 0) & ((A > 0) | ((A == 0) & (B > 0))))
        t, x, y, px, py = t[covered], x[covered], y[covered], px[covered], py[covered]
        z = _fma(dzdy[t], (py - Y[t, 0]).to(F32), _fma(dzdx[t], (px - X[t, 0]).to(F32), z0[t])).clamp(0.0, 1.0)
        yield x, y, z.view(torch.int32).to(I64) & 0x7FFFFFFF, ids[t]
        k = j


def _visibility(level, name, vp, width, height, shadow, samples=1):
    """The visibility planes of a view: depth bits << 32 | triangle + 1 (0: background)."""
    rs = level.bias
    records = _records(level.clip_positions(name, vp), width, height, bool(rs.cull_enabled),
                       rs if shadow and rs.depth_bias_enabled else None, samples)
    planes = torch.zeros(samples, height * width, dtype=I64, device=_device())
    for s in range(samples):
        sx, sy = (128, 128) if samples == 1 else (int(256 * SAMPLES[s][0]), int(256 * SAMPLES[s][1]))
        for x, y, z, t in _fragments(records, sx, sy):
            planes[s].scatter_reduce_(0, y * width + x, (z << 32) | (t + 1), "amax")
    return planes


def _linear(c):
    return torch.where(c <= 0.04045, c / 12.92, ((c + 0.055) / 1.055).clamp(min=0) ** 2.4)


def _encoded(c):
    return torch.where(c <= 0.0031308, 12.92 * c, 1.055 * c.clamp(min=0) ** (1 / 2.4) - 0.055)


class _Images:
    """The material maps, one stack per map of (materials, h, w, channels) bytes, with their chains when built."""

    def __init__(self, level, mips):
        dev = _device()
        self.maps = []
        for which in range(3):  # albedo, normal, metallic-roughness
            descs = [level.textures[3 * m + which] for m in range(len(level.materials))]
            channels, srgb = (4 if which == 0 else 2), which != 1
            base = torch.stack([torch.from_numpy(np.frombuffer(
                C.string_at(d.pixels, d.width * d.height * channels), np.uint8).copy().reshape(d.height, d.width, channels))
                for d in descs]).to(dev)
            chain = [base]
            while mips and max(chain[-1].shape[1:3]) > 1:
                chain.append(self.half(chain[-1], srgb))
            self.maps.append((chain, srgb))

    @staticmethod
    def half(img, srgb):
        h, w = img.shape[1:3]
        ys = torch.arange(max(1, h // 2), device=img.device) * 2
        xs = torch.arange(max(1, w // 2), device=img.device) * 2
        c = img.to(F64) / 255.0
        alpha = srgb and img.shape[3] == 4
        if srgb:
            c = torch.cat([_linear(c[..., :3]) * c[..., 3:], c[..., 3:]], -1) if alpha else _linear(c)
        mean = sum(c[:, (ys + j).clamp(max=h - 1)][:, :, (xs + i).clamp(max=w - 1)] for j in (0, 1) for i in (0, 1)) * 0.25
        if alpha:
            a = mean[..., 3:]
            mean = torch.cat([_encoded(torch.where(a > 0, mean[..., :3] / a.clamp(min=1e-300), mean[..., :3])), a], -1)
        elif srgb:
            mean = _encoded(mean)
        return torch.floor(mean.clamp(0, 1) * 255.0 + 0.5).to(torch.uint8)

    def bilinear(self, which, level, material, u, v):
        chain, srgb = self.maps[which]
        img = chain[level]
        h, w = img.shape[1:3]
        x, y = u * w - 0.5, v * h - 0.5
        x0, y0 = torch.floor(x), torch.floor(y)
        ax, ay = (x - x0)[:, None], (y - y0)[:, None]
        x0, y0 = x0.to(I64), y0.to(I64)

        def at(xi, yi):
            c = img[material, yi % h, xi % w].to(F64) / 255.0
            if srgb:
                c = torch.cat([_linear(c[:, :3]), c[:, 3:]], -1) if c.shape[1] == 4 else _linear(c)
            return c

        return ((1 - ax) * (1 - ay) * at(x0, y0) + ax * (1 - ay) * at(x0 + 1, y0) +
                (1 - ax) * ay * at(x0, y0 + 1) + ax * ay * at(x0 + 1, y0 + 1))

    def sample(self, which, material, u, v, duv):
        chain = self.maps[which][0]
        if len(chain) == 1:
            return self.bilinear(which, 0, material, u, v)
        h, w = chain[0].shape[1:3]
        size = torch.tensor([w, h], dtype=F64, device=u.device)
        rho = torch.maximum((duv[0] * size).norm(dim=1), (duv[1] * size).norm(dim=1))
        d = torch.log2(rho).clamp(0, len(chain) - 1)
        out = torch.zeros(u.numel(), chain[0].shape[3], dtype=F64, device=u.device)
        for l in range(len(chain)):  # each level takes part with its weight of the trilinear blend
            weight = (1 - (d - l).abs()).clamp(min=0)
            on = weight > 0
            if bool(on.any()):
                out[on] += weight[on, None] * self.bilinear(which, l, material[on], u[on], v[on])
        return out


class _Latents:
    """The decoder that training starts from: the maps' values at the cell centres, in halves, and an MLP that passes
    them through; decoded values are their bilinear interpolation."""

    def __init__(self, images, size, materials, kind=torch.float16):
        dev = _device()
        at = (torch.arange(size, device=dev, dtype=F64) + 0.5) / size
        u, v = at.repeat(size), at.repeat_interleave(size)
        grids = []
        for m in range(materials):
            which = torch.full_like(u, m, dtype=I64)
            grids.append(torch.cat([images.bilinear(k, 0, which, u, v)[:, :n] for k, n in ((0, 3), (1, 2), (2, 2))], 1))
        self.grid = torch.stack(grids).reshape(materials, size, size, 7).to(F32).to(kind)

    def decode(self, material, u, v):
        n = self.grid.shape[1]
        x, y = u * n - 0.5, v * n - 0.5
        x0, y0 = torch.floor(x), torch.floor(y)
        ax, ay = (x - x0)[:, None], (y - y0)[:, None]
        x0, y0 = x0.to(I64), y0.to(I64)
        at = lambda xi, yi: self.grid[material, yi % n, xi % n].to(F64)  # noqa: E731
        return ((1 - ax) * (1 - ay) * at(x0, y0) + ax * (1 - ay) * at(x0 + 1, y0) +
                (1 - ax) * ay * at(x0, y0 + 1) + ax * ay * at(x0 + 1, y0 + 1)).clamp(0, 1)


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


class _Shader:
    """Cook-Torrance with filtered shadow maps (basic.slang:15-344, lighting.slang:5-43, pcf.slang:1-12) for the state the
    generated scenes have: tangent-space lighting, normal maps on, every material with its three maps."""

    def __init__(self, level, images, latents, view, shadow_maps):
        self.level, self.images, self.latents, self.maps = level, images, latents, shadow_maps
        self.width, self.height, self.vp = view.width, view.height, list(view.view_projection)
        self.clips = {}

    def colours(self, name, pixel, triangle):
        """(pixels, 4) FP64 colours of a list's triangles at pixel centres, with each one's alpha-mask verdict."""
        parts = [self._piece(name, pixel[a:a + PIECE], triangle[a:a + PIECE]) for a in range(0, pixel.numel(), PIECE)]
        if not parts:
            return torch.zeros(0, 4, dtype=F64, device=pixel.device), torch.zeros(0, dtype=torch.bool, device=pixel.device)
        return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])

    def _barycentrics(self, clip, pixel):
        """At the pixel centre from the vertices as the raster snapped them (clip positions where it clipped)."""
        x, y = (pixel % self.width), (pixel // self.width)
        d = _planes(clip)
        inside = (d >= 0).all(-1).all(-1)
        ndc = clip[..., :2] / clip[..., 3:]
        half = torch.tensor([0.5 * self.width, 0.5 * self.height], dtype=F32, device=clip.device).expand_as(ndc)
        xy = torch.round(_fma(ndc, half, half) * 256.0).to(F64)
        w = clip[..., 3].to(F64)
        px, py = (x * 256 + 128).to(F64)[:, None], (y * 256 + 128).to(F64)[:, None]
        X, Y = xy[..., 0] - px, xy[..., 1] - py
        r1, r2 = [1, 2, 0], [2, 0, 1]
        n = (X[:, r1] * Y[:, r2] - X[:, r2] * Y[:, r1]) * w[:, r1] * w[:, r2]
        nx = 256.0 * (Y[:, r1] - Y[:, r2]) * w[:, r1] * w[:, r2]
        ny = 256.0 * (X[:, r2] - X[:, r1]) * w[:, r1] * w[:, r2]
        if not bool(inside.all()):
            o = ~inside
            c = clip[o].to(F64)
            u, v = (x[o].to(F64) + 0.5) * 2 / self.width - 1, (y[o].to(F64) + 0.5) * 2 / self.height - 1
            a, b = c[..., 0] - u[:, None] * c[..., 3], c[..., 1] - v[:, None] * c[..., 3]
            da, db = -c[..., 3] * 2 / self.width, -c[..., 3] * 2 / self.height
            n[o], nx[o], ny[o] = (torch.linalg.cross(p, q) for p, q in ((a, b), (da, b), (a, db)))
        s = n.sum(1, keepdim=True)
        lam = n / s
        return lam, (nx - lam * nx.sum(1, keepdim=True)) / s, (ny - lam * ny.sum(1, keepdim=True)) / s, (w * lam).sum(1)

    def _piece(self, name, pixel, triangle):
        L, sd = self.level, self.level.sd
        if name not in self.clips:
            self.clips[name] = L.clip_positions(name, self.vp)
        tri, obj, mat = (t[triangle] for t in L.lists[name])
        lam, dx, dy, depth = self._barycentrics(self.clips[name][triangle], pixel)
        v = {k: t[tri].to(F64) for k, t in L.vertex.items()}
        mix = lambda t: (lam[:, :, None] * t).sum(1)  # noqa: E731
        o = L.objects[obj].to(F64)
        world4, to_object = o[:, :16].reshape(-1, 4, 4), o[:, 16:32].reshape(-1, 4, 4)  # [n, column, row]
        eye, sun = _matrix(sd.camera_position).to(F64), _matrix(sd.sun_position).to(F64)
        pos = mix(v["vertex"])
        world = (world4[:, :3] * pos[:, :, None]).sum(1) + world4[:, 3]
        view_dir = (to_object * eye[:, None]).sum(1)[:, :3] - pos
        light = _unit((to_object * sun[:, None]).sum(1)[:, :3] - pos)
        normal, tangent, sigma = mix(v["normal"]), mix(v["tangents"][..., :3]), mix(v["tangents"][..., 3:])
        uv, vertex_alpha = mix(v["uv"]), mix(v["color"])[:, 3]
        duv = tuple((d[:, :, None] * v["uv"]).sum(1) for d in (dx, dy))
        factor = torch.tensor([m.color[3] for m in L.materials], dtype=F64, device=lam.device)[mat]
        alpha = torch.minimum(factor, vertex_alpha)
        if self.latents is not None and name != "blended":
            dec = self.latents.decode(mat, uv[:, 0], uv[:, 1])
            albedo, bump, metal, rough = dec[:, :3], dec[:, 3:5], dec[:, 5:6], dec[:, 6:7]
            alpha = alpha.clamp(max=1.0)
        else:
            maps = [self.images.sample(k, mat, uv[:, 0], uv[:, 1], duv) for k in range(3)]
            albedo, bump, metal, rough = maps[0][:, :3], maps[1], maps[2][:, :1], maps[2][:, 1:2]
            alpha = torch.minimum(maps[0][:, 3], alpha)
        bump = bump * 2 - 1
        bump = torch.cat([bump, (1 - _dot(bump, bump)).clamp(min=0).sqrt()], -1)
        n = _unit(normal)
        t = _unit(tangent - n * _dot(tangent, n))
        b = _unit(torch.linalg.cross(normal, tangent) * sigma)
        N = _unit(t * bump[:, :1] + b * bump[:, 1:2] + n * bump[:, 2:])
        V = _unit(view_dir)
        H = _unit(light + V)
        shadow = self._shadow(world, depth)[:, None]
        ldn, ndv = _dot(light, N).clamp(0, 1), _dot(N, V).clamp(0, 1)
        f0 = 0.04 + (albedo - 0.04) * metal
        a2 = rough ** 4
        ndh = _dot(N, H).clamp(min=0)
        dist = a2 / (3.14159265359 * (ndh * ndh * (a2 - 1) + 1) ** 2)
        k = (rough + 1) ** 2 / 8
        smith = [c / (c * (1 - k) + k) for c in (_dot(N, light).clamp(min=0), _dot(N, V).clamp(min=0))]
        F = f0 + (1 - f0) * (1 - _dot(H, V).clamp(min=0)).clamp(0, 1) ** 5
        spec = F * (dist * smith[0] * smith[1]) / (4 * ndv * ldn + 0.0001)
        diffuse = albedo / 3.14159265
        lit = ((1 - F) * (1 - metal) * diffuse + spec) * _matrix(sd.sunlight_color)[:3].to(F64) * sd.light_intensity * ldn
        colour = torch.maximum(_matrix(sd.ambient_color)[:3].to(F64) * diffuse, lit * shadow)
        masked = torch.tensor([m.alpha_mode == 1 for m in L.materials], device=lam.device)[mat]
        cutoff = torch.tensor([m.alpha_cutoff for m in L.materials], dtype=F64, device=lam.device)[mat]
        return torch.cat([colour, alpha[:, None]], 1), masked & (alpha < cutoff)

    def _shadow(self, world, depth):
        out = torch.ones_like(depth)
        left = torch.ones_like(depth, dtype=torch.bool)
        for c, m in self.maps:
            on = left & (depth <= c.split_far)
            left &= ~on
            if not bool(on.any()):
                continue
            s = (_matrix(c.light_view_projection).to(F64).reshape(4, 4)[None] * world[on][:, :, None]).sum(1)
            x, y, ref = 0.5 * s[:, 0] + 0.5 * s[:, 3], 0.5 * s[:, 1] + 0.5 * s[:, 3], s[:, 2]
            if self.level.bias.pcf_mode == 1:
                taps = [(i / c.size, j / c.size) for j in (-1, 0, 1) for i in (-1, 0, 1)]
            else:
                e = 0.00025
                taps = [(-e, -e), (2 * e, 0), (0, 2 * e), (2 * e, 2 * e), (-2 * e, -2 * e)]
            out[on] = sum(self._tap(m, c.size, x + i, y + j, ref) for i, j in taps) / len(taps)
        return out

    @staticmethod
    def _tap(m, size, u, v, ref):
        x, y = u * size - 0.5, v * size - 0.5
        x0, y0 = torch.floor(x), torch.floor(y)
        ax, ay = x - x0, y - y0
        xs = [(x0.clamp(-2, size + 1) + i).clamp(0, size - 1).to(I64) for i in (0, 1)]
        ys = [(y0.clamp(-2, size + 1) + i).clamp(0, size - 1).to(I64) for i in (0, 1)]
        r = torch.zeros_like(x)
        for j in (0, 1):
            for i in (0, 1):
                r += (ax if i else 1 - ax) * (ay if j else 1 - ay) * (ref >= m[ys[j] * size + xs[i]].to(F64)).to(F64)
        return r


def _blend(level, shader, samples, planes, colours):
    """The blended list over each sample's colour, in primitive order (both faces, depth tested, not written)."""
    w, h = shader.width, shader.height
    rec = _records(level.clip_positions("blended", shader.vp), w, h, False, None, samples)
    for s in range(samples):
        sx, sy = (128, 128) if samples == 1 else (int(256 * SAMPLES[s][0]), int(256 * SAMPLES[s][1]))
        keys = [torch.zeros(0, dtype=I64, device=planes.device)]
        for x, y, z, t in _fragments(rec, sx, sy):
            o = y * w + x
            on = z >= (planes[s][o] >> 32)
            keys.append((o[on] << 32) | t[on])
        keys = torch.cat(keys).sort().values
        pixel, tri = keys >> 32, keys & 0xFFFFFFFF
        src, dropped = shader.colours("blended", pixel, tri)
        pixel, src = pixel[~dropped], src[~dropped]
        first = torch.searchsorted(pixel, pixel)  # of the pixel's own fragments
        rank = torch.arange(pixel.numel(), device=pixel.device) - first
        for k in range(int(rank.max()) + 1 if rank.numel() else 0):
            o, f = pixel[rank == k], src[rank == k]
            a = f[:, 3:]
            colours[s][o] = torch.cat([f[:, :3] * a + colours[s][o][:, :3] * (1 - a), a], 1)


def _exact_frame(case, seed):
    scene = _scene(case, seed)
    level = _Level(scene)
    images = _Images(level, case["mips"])
    latents = None
    if case["shade"] != "plain":
        latents = _Latents(images, min(256, case["texture"]), case["materials"])
    maps = []
    for c in scene.cascades():
        z = _visibility(level, "all", list(c.light_view_projection), c.size, c.size, True)[0]
        maps.append((c, (z >> 32).to(torch.int32).view(F32)))
    clear = torch.tensor(list(level.bias.clear_color), dtype=F64, device=_device())
    out = {}
    for i, view in enumerate(scene.camera_views()):
        shader = _Shader(level, images, latents, view, maps)
        n = case["samples"]
        planes = _visibility(level, "opaque", list(view.view_projection), view.width, view.height, False, n)
        colours = clear.repeat(n, view.width * view.height, 1)
        for s in range(n):
            pixel = planes[s].nonzero()[:, 0]
            colours[s][pixel] = shader.colours("opaque", pixel, (planes[s][pixel] & 0xFFFFFFFF) - 1)[0]
        if case["translucent"]:
            _blend(level, shader, n, planes, colours)
        out[f"visibility{i}"], out[f"colour{i}"] = None, colours.mean(0).reshape(view.height, view.width, 4)
    scene.close()
    return {"draw_image": out["colour0"]} if case["kind"] == "loop" else out


def _exact_evaluate(case, seed):
    scene = _material_scene(case, seed)
    level = _Level(scene)
    images = _Images(level, False)
    latents = _Latents(images, case["latent"], case["materials"])
    size = case["texture"]
    at = (torch.arange(size, device=_device(), dtype=F64) + 0.5) / size
    u, v = at.repeat(size), at.repeat_interleave(size)
    psnr = []
    for m in range(case["materials"]):
        which = torch.full_like(u, m, dtype=I64)
        want = torch.cat([images.bilinear(k, 0, which, u, v)[:, :n] for k, n in ((0, 3), (1, 2), (2, 2))], 1)
        psnr.append(-10 * torch.log10(((latents.decode(which, u, v) - want) ** 2).mean()))
    scene.close()
    return {"psnr": torch.stack(psnr)}


_MASK = (1 << 64) - 1


def _mix(z):
    """The SplitMix64 finaliser that the training draws its samples with, on Python integers or int64 tensors."""
    if isinstance(z, int):
        z = (z + 0x9E3779B97F4A7C15) & _MASK
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
        return z ^ (z >> 31)
    signed = lambda c: c - (1 << 64) if c >> 63 else c  # noqa: E731
    shifted = lambda x, n: (x >> n) & ((1 << (64 - n)) - 1)  # noqa: E731
    z = z + signed(0x9E3779B97F4A7C15)
    z = (z ^ shifted(z, 30)) * signed(0xBF58476D1CE4E5B9)
    z = (z ^ shifted(z, 27)) * signed(0x94D049BB133111EB)
    return z ^ shifted(z, 31)


def _start_mlp(seed):
    """The MLP that passes latent channels 0..6 through, its spare hidden units with small random inputs."""
    w1, w2 = np.zeros((32, 10), np.float32), np.zeros((7, 32), np.float32)
    for c in range(7):
        w1[2 * c, c], w1[2 * c + 1, c], w2[c, 2 * c], w2[c, 2 * c + 1] = 1, -1, 1, -1
    s = seed ^ 0x6A09E667F3BCC909
    for j in range(14, 32):
        for k in range(10):
            unit = np.float32((_mix(s) >> 11) * 2.0 ** -53)
            s = (s + 0x9E3779B97F4A7C15) & _MASK
            w1[j, k] = np.float32(-0.1) + (np.float32(0.1) - np.float32(-0.1)) * unit
    return [torch.from_numpy(a).to(_device(), F64) for a in (w1, np.zeros(32, np.float32), w2, np.zeros(7, np.float32))]


def _exact_train(case, seed):
    """The same Adam steps on the same samples in FP64."""
    scene, dev = _material_scene(case, seed), _device()
    images = _Images(_Level(scene), False)
    scene.close()
    n, size, R, seed = case["materials"], case["latent"], case["region"], 1 + seed % 65521
    lat = _Latents(images, size, n, torch.float32).grid.to(F64)
    lat = torch.cat([lat, torch.zeros_like(lat[..., :1])], -1).reshape(-1, 8)
    mlp = _start_mlp(seed)
    moments = [[torch.zeros_like(p) for p in [lat] + mlp] for _ in range(2)]
    across = size // R
    regions = n * across * across
    wgs = min(case["batch"] // 256, regions)
    per = -(-case["batch"] // wgs)
    wg = torch.arange(wgs, device=dev)
    cell = torch.arange(R, device=dev)
    losses = []
    for step in range(case["steps"]):
        r = (step * wgs + wg) % regions
        slot, reg = r % n, ((r // n) * 2654435761) & (across * across - 1)
        shift = _mix(seed ^ _mix((0x5BD1E995 + step) & 0xFFFFFFFF))
        rx = (reg % across) * R + (shift & (R - 1))
        ry = (reg // across) * R + ((shift >> 32) & (R - 1))
        key = _mix((seed + 0x632BE59BD9B4E019 * (step + 1)) & _MASK)
        key = key - (1 << 64) if key >> 63 else key
        h = _mix(key + (wg << 32)[:, None] + torch.arange(per, device=dev))
        xl, yl = ((((h >> s) & 0xFFFFFFFF) >> 8).to(F32) * (1.0 / 16777216.0) * float(R - 1) for s in (0, 32))
        i, j = (t.to(I64).clamp(max=R - 2) for t in (xl, yl))
        ax, ay = ((t - k.to(F32)).to(F64)[..., None] for t, k in ((xl, i), (yl, j)))
        u, v = ((o[:, None] + t.to(F64) + 0.5) / size for o, t in ((rx, xl), (ry, yl)))
        which = slot[:, None].expand_as(i).reshape(-1)
        want = torch.cat([images.bilinear(k, 0, which, u.reshape(-1), v.reshape(-1))[:, :m]
                          for k, m in ((0, 3), (1, 2), (2, 2))], 1)
        at = lambda x, y: (slot[:, None] * size + (ry[:, None] + y) % size) * size + (rx[:, None] + x) % size  # noqa: E731
        params = [p.requires_grad_(True) for p in [lat] + mlp]
        w1, b1, w2, b2 = mlp
        f = ((1 - ax) * (1 - ay) * lat[at(i, j)] + ax * (1 - ay) * lat[at(i + 1, j)] +
             (1 - ax) * ay * lat[at(i, j + 1)] + ax * ay * lat[at(i + 1, j + 1)])
        f = torch.cat([f, 1 - (2 * ax - 1).abs(), 1 - (2 * ay - 1).abs()], -1).reshape(-1, 10)
        loss = ((torch.relu(f @ w1.T + b1) @ w2.T + b2 - want) ** 2).mean()
        losses.append(loss.detach())
        grads = torch.autograd.grad(loss, params)
        rate = 1e-3 * 0.5 * (1 + math.cos(math.pi * step / 20000))
        touched = (at(cell.repeat(R)[None], cell.repeat_interleave(R)[None])).reshape(-1)
        with torch.no_grad():
            for k, (p, g) in enumerate(zip(params, grads)):
                rows = touched if k == 0 else slice(None)
                m = moments[0][k][rows] * 0.9 + 0.1 * g[rows]
                s = moments[1][k][rows] * 0.999 + 0.001 * g[rows] ** 2
                moments[0][k][rows], moments[1][k][rows] = m, s
                p[rows] -= rate * (m / (1 - 0.9 ** (step + 1))) / ((s / (1 - 0.999 ** (step + 1))).sqrt() + 1e-8)
        lat, mlp = params[0].detach(), [p.detach() for p in params[1:]]
    return {"loss": torch.stack(losses), "latents": lat.reshape(n, size, size, 8),
            "mlp": torch.cat([p.reshape(-1) for p in mlp])}


def exact(case, seed):
    if case["kind"] in ("frame", "replay", "loop"):
        return _exact_frame(case, seed)
    if case["kind"] == "evaluate":
        return _exact_evaluate(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None  # load: whole bytes
