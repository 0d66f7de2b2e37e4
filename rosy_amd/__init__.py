"""rosy_amd -- MI355X raster-and-shade frame path behind a C ABI (include/rosy_amd.h).

This Python module is a thin ctypes harness over librosy_amd.so for tests and benchmarks; the
product is the shared library.  Importing works without a GPU (host-only entry points such as the
scene generator and the matrix closed forms can be called); creating a Renderer needs a HIP device
and fails loudly when there is none or when the library has not been built.
"""
import ctypes as C
import os

import numpy as np

from . import abi

__all__ = ["lib", "RosyError", "Scene", "Renderer", "abi"]

_lib = None


def lib():
    """The loaded librosy_amd.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(abi.LIB_PATH):
            raise ImportError(f"{abi.LIB_PATH} is missing: build it with `make -C rosy_amd` or __graft_entry__.build()")
        _lib = abi.bind(C.CDLL(abi.LIB_PATH))
    return _lib


class RosyError(RuntimeError):
    def __init__(self, code, what, detail=""):
        self.code = code
        name = abi.RESULT_NAMES.get(code, str(code))
        super().__init__(f"{what} failed: rosy::result::{name} ({code}) {detail}".rstrip())


def _check(code, what, ctx=None):
    if code != abi.RSY_OK:
        detail = ""
        if ctx:
            msg = lib().rsy_last_error(ctx)
            detail = msg.decode() if msg else ""
        raise RosyError(code, what, detail)


def _arr(ptr, n, dtype):
    if n == 0:
        return np.zeros(0, dtype=dtype)
    return np.ctypeslib.as_array(C.cast(ptr, C.POINTER(C.c_uint8)), shape=(n * np.dtype(dtype).itemsize,)).view(dtype)


class Scene:
    """A seeded synthetic workload generated by rsy_scene_generate (host memory)."""

    def __init__(self, workload, seed=1, **overrides):
        d = abi.SceneDesc()
        d.workload = workload
        d.seed = seed
        for k, v in overrides.items():
            setattr(d, k, v)
        p = C.POINTER(abi.Scene)()
        _check(lib().rsy_scene_generate(C.byref(d), C.byref(p)), "rsy_scene_generate")
        self._p = p
        self.s = p.contents
        self.workload = workload
        self.seed = seed

    def close(self):
        if getattr(self, "_p", None):
            lib().rsy_scene_free(self._p)
            self._p = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    # numpy views of the scene arrays (valid while the Scene is alive)
    @property
    def vertices(self):
        return _arr(self.s.vertices, self.s.n_vertices, np.dtype([("vertex", "<f4", 3), ("normal", "<f4", 3),
                                                                  ("tangents", "<f4", 4), ("color", "<f4", 4),
                                                                  ("uv", "<f4", 2)]))

    @property
    def indices(self):
        return _arr(self.s.indices, self.s.n_indices, np.uint32)

    @property
    def n_triangles(self):
        return int(self.s.n_indices // 3)

    def camera_views(self):
        return [self.s.camera_views[i] for i in range(self.s.n_camera_views)]

    def cascades(self):
        return [self.s.cascades[i] for i in range(self.s.n_cascades)]

    def surfaces(self):
        return [self.s.surfaces[i] for i in range(self.s.n_surfaces)]

    def frame_desc(self, shade_mode=abi.SHADE_PLAIN, explicit=True):
        f = abi.FrameDesc()
        f.shade_mode = shade_mode
        f.default_shadow_size = self.s.default_shadow_size
        if explicit:
            f.n_camera_views = self.s.n_camera_views
            f.camera_views = self.s.camera_views
            f.n_cascades = self.s.n_cascades
            f.cascades = self.s.cascades
        return f


class Renderer:
    """One rsy_ctx (one HIP stream) holding a scene's geometry, materials and objects."""

    def __init__(self, device=0):
        cfg = abi.Config(abi.RSY_ABI_VERSION, device, 0, 0)
        ctx = C.c_void_p()
        _check(lib().rsy_create(C.byref(cfg), C.byref(ctx)), "rsy_create")
        self.ctx = ctx
        self.views = []
        self.cascade_sizes = []

    def close(self):
        if getattr(self, "ctx", None):
            lib().rsy_destroy(self.ctx)
            self.ctx = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _c(self, code, what):
        _check(code, what, self.ctx)

    def load(self, scene: Scene):
        s = scene.s
        L = lib()
        self._c(L.rsy_set_geometry(self.ctx, s.vertices, s.n_vertices, s.indices, s.n_indices, s.meshes, s.n_meshes),
                "rsy_set_geometry")
        self._c(L.rsy_set_materials(self.ctx, s.materials, s.n_materials, s.textures, s.n_textures, s.samplers,
                                    s.n_samplers), "rsy_set_materials")
        self._c(L.rsy_set_graphic_objects(self.ctx, s.objects, s.n_objects, s.surfaces, s.n_surfaces),
                "rsy_set_graphic_objects")
        self.update(s.scene_data, s.raster_state)
        self.scene = scene

    def update(self, scene_data, raster_state=None):
        self._c(lib().rsy_update(self.ctx, C.byref(scene_data), C.byref(raster_state) if raster_state else None),
                "rsy_update")
        if raster_state is not None:
            self.samples = 4 if raster_state.msaa_samples == 4 else 1

    def _remember(self, frame):
        if frame is not None and frame.n_camera_views:
            self.views = [(frame.camera_views[i].width, frame.camera_views[i].height)
                          for i in range(frame.n_camera_views)]
        elif getattr(self, "scene", None) is not None:
            sd = self.scene.s.scene_data
            self.views = [(int(sd.draw_extent[0]), int(sd.draw_extent[1]))]
        if frame is not None and frame.n_cascades:
            self.cascade_sizes = [frame.cascades[i].size for i in range(frame.n_cascades)]
        else:
            self.cascade_sizes = [frame.default_shadow_size if frame is not None and frame.default_shadow_size else 2048]

    def render(self, frame=None):
        self._remember(frame)
        self._c(lib().rsy_render(self.ctx, C.byref(frame) if frame is not None else None), "rsy_render")

    def render_graph(self, frame, n_replays):
        self._remember(frame)
        self._c(lib().rsy_render_graph(self.ctx, C.byref(frame), n_replays), "rsy_render_graph")

    def synchronize(self):
        self._c(lib().rsy_synchronize(self.ctx), "rsy_synchronize")

    def packed_materials(self):
        """(materials sampled as one packed image, bytes of those images)."""
        n, b = C.c_uint32(), C.c_uint64()
        self._c(lib().rsy_get_packed_materials(self.ctx, C.byref(n), C.byref(b)), "rsy_get_packed_materials")
        return n.value, b.value

    def set_debug_flags(self, flags):
        self._c(lib().rsy_set_debug_flags(self.ctx, flags), "rsy_set_debug_flags")

    def autotune(self, frame, n_iters=3):
        t = C.c_uint32()
        self._remember(frame)
        self._c(lib().rsy_autotune(self.ctx, C.byref(frame), n_iters, C.byref(t)), "rsy_autotune")
        return t.value

    def visibility(self, view=0):
        """The view's visibility words (h, w), or (4, h, w) sample planes in a 4-sample frame."""
        w, h = self.views[view]
        n = getattr(self, "samples", 1)
        out = np.empty((n, h, w) if n > 1 else (h, w), dtype=np.uint64)
        self._c(lib().rsy_read_visibility(self.ctx, view, out.ctypes.data, out.size), "rsy_read_visibility")
        return out

    def color(self, view=0):
        w, h = self.views[view]
        out = np.empty((h, w, 4), dtype=np.float32)
        self._c(lib().rsy_read_color(self.ctx, view, out.ctypes.data, h * w), "rsy_read_color")
        return out

    def shadow_factor(self, view=0):
        w, h = self.views[view]
        out = np.empty((h, w), dtype=np.float32)
        self._c(lib().rsy_read_shadow_factor(self.ctx, view, out.ctypes.data, out.size), "rsy_read_shadow_factor")
        return out

    def present(self, view=0, width=None, height=None, readback=True):
        """Output stage of the last shaded frame: returns (RGBA16F draw image as float16 (h, w, 4),
        B8G8R8A8_SRGB image as uint8 (height, width, 4)); None without `readback`."""
        w, h = self.views[view]
        width, height = (w if width is None else width), (h if height is None else height)
        self._c(lib().rsy_present(self.ctx, view, width, height), "rsy_present")
        if not readback:
            return None
        draw = np.empty((h, w, 4), dtype=np.float16)
        self._c(lib().rsy_read_draw_image(self.ctx, draw.ctypes.data, h * w), "rsy_read_draw_image")
        out = np.empty((height, width, 4), dtype=np.uint8)
        self._c(lib().rsy_read_present(self.ctx, out.ctypes.data, height * width), "rsy_read_present")
        return draw, out

    def shadow_map(self, cascade=0):
        s = self.cascade_sizes[cascade]
        out = np.empty((s, s), dtype=np.float32)
        self._c(lib().rsy_read_shadow_map(self.ctx, cascade, out.ctypes.data, out.size), "rsy_read_shadow_map")
        return out

    def stats(self):
        st = abi.FrameStats()
        self._c(lib().rsy_get_frame_stats(self.ctx, C.byref(st)), "rsy_get_frame_stats")
        return st

    # ---- neural material decoder --------------------------------------------------------------

    def neural_init(self, **overrides):
        """rsy_neural_init with the default configuration updated by `overrides`; returns it."""
        cfg = abi.NeuralConfig()
        lib().rsy_neural_default_config(C.byref(cfg))
        for k, v in overrides.items():
            setattr(cfg, k, v)
        self._c(lib().rsy_neural_init(self.ctx, C.byref(cfg)), "rsy_neural_init")
        self.neural_cfg = cfg
        return cfg

    def neural_train(self, steps):
        """Runs `steps` Adam steps; returns the per-step mean squared error."""
        loss = np.zeros(max(1, steps), dtype=np.float32)
        self._c(lib().rsy_neural_train(self.ctx, steps, loss.ctypes.data), "rsy_neural_train")
        return loss[:steps]

    def neural_evaluate(self):
        """Exports the inference parameters; returns the per-material PSNR (NaN = not decodable)."""
        n = self.scene.s.n_materials
        psnr = np.zeros(max(1, n), dtype=np.float32)
        self._c(lib().rsy_neural_evaluate(self.ctx, psnr.ctypes.data, n), "rsy_neural_evaluate")
        return psnr[:n]

    def neural_stats(self):
        st = abi.NeuralStats()
        self._c(lib().rsy_neural_get_stats(self.ctx, C.byref(st)), "rsy_neural_get_stats")
        return st

    def neural_set_active(self, active):
        a = np.ascontiguousarray(active, dtype=np.uint32)
        self._c(lib().rsy_neural_set_active(self.ctx, a.ctypes.data, a.size), "rsy_neural_set_active")

    def neural_params(self):
        """(latents [eligible, L, L, 8], mlp [583]) FP32 master parameters."""
        st = self.neural_stats()
        L = self.neural_cfg.latent_size
        lat = np.zeros((st.n_eligible, L, L, abi.NEURAL_CHANNELS), dtype=np.float32)
        mlp = np.zeros(abi.NEURAL_PARAMS, dtype=np.float32)
        self._c(lib().rsy_neural_get_params(self.ctx, lat.ctypes.data, lat.size, mlp.ctypes.data, mlp.size),
                "rsy_neural_get_params")
        return lat, mlp

    def neural_set_params(self, latents, mlp):
        lat = np.ascontiguousarray(latents, dtype=np.float32)
        p = np.ascontiguousarray(mlp, dtype=np.float32)
        self._c(lib().rsy_neural_set_params(self.ctx, lat.ctypes.data, lat.size, p.ctypes.data, p.size),
                "rsy_neural_set_params")

    def neural_gradients(self, material, uv, target):
        """Loss and exact gradients of the training objective on an explicit batch."""
        m = np.ascontiguousarray(material, dtype=np.uint32)
        uv = np.ascontiguousarray(uv, dtype=np.float32)
        t = np.ascontiguousarray(target, dtype=np.float32)
        st = self.neural_stats()
        L = self.neural_cfg.latent_size
        g_lat = np.zeros((st.n_eligible, L, L, abi.NEURAL_CHANNELS), dtype=np.float32)
        g_mlp = np.zeros(abi.NEURAL_PARAMS, dtype=np.float32)
        loss = C.c_float()
        self._c(lib().rsy_neural_gradients(self.ctx, m.ctypes.data, uv.ctypes.data, t.ctypes.data, m.size,
                                           C.byref(loss), g_mlp.ctypes.data, g_lat.ctypes.data, g_lat.size),
                "rsy_neural_gradients")
        return loss.value, g_mlp, g_lat

    def neural_set_weights(self, weights):
        self._c(lib().rsy_neural_set_weights(self.ctx, weights), "rsy_neural_set_weights")

    def neural_inference_mlp(self):
        """The MLP the inference path evaluates (quantised weights, FP32 values, [583])."""
        out = np.zeros(abi.NEURAL_PARAMS, dtype=np.float32)
        self._c(lib().rsy_neural_get_inference_mlp(self.ctx, out.ctypes.data, out.size), "rsy_neural_get_inference_mlp")
        return out

    def neural_decode(self, material, uv, targets=False):
        m = np.ascontiguousarray(material, dtype=np.uint32)
        uv = np.ascontiguousarray(uv, dtype=np.float32)
        out = np.zeros((m.size, abi.NEURAL_OUTPUTS), dtype=np.float32)
        self._c(lib().rsy_neural_decode(self.ctx, m.ctypes.data, uv.ctypes.data, m.size, 1 if targets else 0,
                                        out.ctypes.data), "rsy_neural_decode")
        return out
