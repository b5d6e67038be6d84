"""clovers_amd -- MI355X wavefront spectral path tracer (HIP, gfx950).

Python host front of libclovers_hip.so, the C ABI in include/clovers_hip.h.
The render path is `draw()`, the drop-in for the reference's
`draw_cpu::draw(&GlobalOptions, &RenderOptions, &Scene, Sampler) -> Vec<Xyz<E>>`
(clovers-cli/src/draw_cpu.rs:26-98): it returns the same pixel buffer, linear
XYZ with white point E, row 0 = top, index x + row*W, mean over samples.

There is no CPU fallback: if the HIP library or a GPU is missing, every entry
point raises.
"""
import ctypes as C
import os

import numpy as np

from . import abi

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libclovers_hip.so")
HEADER = os.path.join(os.path.dirname(HERE), "include", "clovers_hip.h")

_lib = None


class ClvError(RuntimeError):
    def __init__(self, status, msg):
        super().__init__("%s: %s" % (abi.STATUS_NAMES.get(status, status), msg))
        self.status = status


def load_library(path=LIB_PATH):
    """Load the HIP library (raises if it was not built)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(path):
        raise ImportError("libclovers_hip.so is not built (run __graft_entry__.build() or "
                          "make -C clovers_amd/csrc); there is no CPU fallback")
    lib = C.CDLL(path)
    vp = C.c_void_p
    lib.clv_abi_version.restype = C.c_uint32
    lib.clv_create.restype = C.c_int
    lib.clv_create.argtypes = [C.c_int, C.POINTER(vp)]
    lib.clv_destroy.argtypes = [vp]
    lib.clv_last_error.restype = C.c_char_p
    lib.clv_last_error.argtypes = [vp]
    lib.clv_scene_upload.restype = C.c_int
    lib.clv_scene_upload.argtypes = [vp, vp, C.POINTER(C.c_uint32)]
    lib.clv_scene_upload_ex.restype = C.c_int
    lib.clv_scene_upload_ex.argtypes = [vp, vp, C.c_uint32, C.POINTER(C.c_uint32)]
    lib.clv_scene_free.restype = C.c_int
    lib.clv_scene_free.argtypes = [vp, C.c_uint32]
    lib.clv_render.restype = C.c_int
    lib.clv_render.argtypes = [vp, C.c_uint32, vp, vp, vp]
    lib.clv_render_batch.restype = C.c_int
    lib.clv_render_batch.argtypes = [vp, vp, C.c_uint32]
    lib.clv_tuning_get.restype = C.c_int
    lib.clv_tuning_get.argtypes = [vp, vp]
    lib.clv_tuning_set.restype = C.c_int
    lib.clv_tuning_set.argtypes = [vp, vp]
    lib.clv_autotune.restype = C.c_int
    lib.clv_autotune.argtypes = [vp, vp, C.c_uint32, C.c_uint64, vp]
    lib.clv_guide_reset.restype = C.c_int
    lib.clv_guide_reset.argtypes = [vp, C.c_uint64]
    lib.clv_guide_params.restype = C.c_int
    lib.clv_guide_params.argtypes = [vp, vp, C.c_uint32]
    lib.clv_guide_set_params.restype = C.c_int
    lib.clv_guide_set_params.argtypes = [vp, vp, C.c_uint32]
    lib.clv_guide_eval.restype = C.c_int
    lib.clv_guide_eval.argtypes = [vp, vp, C.c_uint32, vp, vp]
    lib.clv_guide_grad.restype = C.c_int
    lib.clv_guide_grad.argtypes = [vp, vp, C.c_uint32, vp]
    lib.clv_plan_passes.restype = C.c_int
    lib.clv_plan_passes.argtypes = [vp, C.c_uint32, vp, vp, C.c_uint32, C.POINTER(C.c_uint32), C.POINTER(C.c_uint32)]
    lib.clv_primary_hits.restype = C.c_int
    lib.clv_primary_hits.argtypes = [vp, C.c_uint32, vp, vp, vp]
    lib.clv_primary_hits_noalloc.restype = C.c_int
    lib.clv_primary_hits_noalloc.argtypes = [vp, C.c_uint32, vp, vp, vp]
    lib.clv_counters_get.restype = C.c_int
    lib.clv_counters_get.argtypes = [vp, vp]
    lib.clv_spectral_power.restype = C.c_float
    lib.clv_spectral_power.argtypes = [C.POINTER(C.c_float), C.c_uint32]
    lib.clv_wavelength_into_xyz.restype = C.c_int
    lib.clv_wavelength_into_xyz.argtypes = [C.c_uint32, C.POINTER(C.c_float)]
    lib.clv_scene_validate.restype = C.c_int
    lib.clv_scene_validate.argtypes = [vp, vp]
    lib.clv_scene_file_parse.restype = C.c_int
    lib.clv_scene_file_parse.argtypes = [C.c_char_p, C.c_char_p, C.c_uint32, C.POINTER(vp), C.c_char_p, C.c_uint32]
    lib.clv_scene_file_desc.restype = vp
    lib.clv_scene_file_desc.argtypes = [vp]
    lib.clv_scene_file_free.argtypes = [vp]
    lib.clv_render_debug.restype = C.c_int
    lib.clv_render_debug.argtypes = [vp, C.c_uint32, vp, C.c_uint32, vp]
    lib.clv_write_png.restype = C.c_int
    lib.clv_write_png.argtypes = [vp, C.c_uint32, C.c_uint32, C.c_char_p, C.c_char_p]
    lib.clv_write_exr.restype = C.c_int
    lib.clv_write_exr.argtypes = [vp, C.c_uint32, C.c_uint32, C.c_char_p]
    if lib.clv_abi_version() != abi.ABI_VERSION:
        raise ImportError("libclovers_hip.so ABI %d != %d" % (lib.clv_abi_version(), abi.ABI_VERSION))
    _lib = lib
    return lib


def spectral_power(xyz, lam):
    """clovers::spectrum::spectral_power (spectrum.rs:46-56), the library's host implementation."""
    a = (C.c_float * 3)(*[float(v) for v in xyz])
    return float(load_library().clv_spectral_power(a, int(lam)))


def wavelength_into_xyz(lam):
    """clovers::wavelength::wavelength_into_xyz (wavelength.rs:62-83) as the library tabulates it."""
    out = (C.c_float * 3)()
    st = load_library().clv_wavelength_into_xyz(int(lam), out)
    if st != abi.OK:
        raise ClvError(st, "wavelength out of range")
    return np.array(out[:], np.float32)


def validate(scene):
    """clv_scene_validate: host build only (no device) -> dict of the scene's
    shape; raises ClvError with the builder's message if the scene is invalid."""
    desc, keep = scene.as_ctypes()
    info = abi.SceneInfo()
    st = load_library().clv_scene_validate(C.byref(desc), C.byref(info))
    if st != abi.OK:
        raise ClvError(st, info.error.decode())
    return {k: getattr(info, k) for k, _ in abi.SceneInfo._fields_ if k != "error"}


class SceneFile:
    """A scene file parsed by the library (clv_scene_file_parse): usable
    wherever a SceneDescription is (upload, validate); `objects`,
    `materials` and `xforms` are numpy copies of its descriptor."""

    def __init__(self, src, mesh_root=None, bvh_algorithm=abi.BVH_SAH):
        lib = load_library()
        if not src.lstrip().startswith("{"):
            with open(src) as f:
                src = f.read()
        h = C.c_void_p()
        err = C.create_string_buffer(512)
        st = lib.clv_scene_file_parse(src.encode(), mesh_root.encode() if mesh_root else None, bvh_algorithm,
                                      C.byref(h), err, 512)
        if st != abi.OK:
            raise ClvError(st, err.value.decode())
        self._lib, self.h = lib, h
        d = abi.SceneDesc.from_address(lib.clv_scene_file_desc(h))
        self._desc = d

        def arr(ptr, n, dt):
            if n == 0:
                return np.zeros(0, dt)
            return np.frombuffer((C.c_char * (n * dt.itemsize)).from_address(ptr), dt).copy()
        self.objects = arr(d.objects, d.n_objects, abi.OBJECT_DTYPE)
        self.materials = arr(d.materials, d.n_materials, abi.MATERIAL_DTYPE)
        self.xforms = arr(d.xforms, d.n_xforms, abi.XFORM_DTYPE)
        self.background = np.array(d.background[:], np.float32)
        self.camera = {k: (list(getattr(d.camera, k)) if k in ("look_from", "look_at", "up") else getattr(d.camera, k))
                       for k, _ in abi.CameraInit._fields_}

    def as_ctypes(self):
        return self._desc, self

    def close(self):
        if getattr(self, "h", None):
            self._lib.clv_scene_file_free(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def _image(img):
    img = np.ascontiguousarray(img, dtype=np.float32)
    if img.ndim != 3 or img.shape[2] != 3:
        raise ValueError("expected an [H, W, 3] Xyz<E> image")
    return img


def write_png(img, path, comment=None):
    """clv_write_png: Xyz<E> [H, W, 3] (row 0 = top) -> 8-bit sRGB PNG (write.rs:18-84)."""
    img = _image(img)
    st = load_library().clv_write_png(img.ctypes.data, img.shape[1], img.shape[0], os.fsencode(path),
                                      comment.encode() if comment else None)
    if st != abi.OK:
        raise ClvError(st, "cannot write %s" % path)


def write_exr(img, path):
    """clv_write_exr: Xyz<E> [H, W, 3] -> OpenEXR, R/G/B = X/Y/Z (write.rs:86-125)."""
    img = _image(img)
    st = load_library().clv_write_exr(img.ctypes.data, img.shape[1], img.shape[0], os.fsencode(path))
    if st != abi.OK:
        raise ClvError(st, "cannot write %s" % path)


def load_scene_file(src, mesh_root=None, bvh_algorithm=abi.BVH_SAH):
    """Parse a scene file (path or JSON text) in the library; see SceneFile."""
    return SceneFile(src, mesh_root, bvh_algorithm)


class Renderer:
    """One context on one HIP device (not re-entrant, like clv_ctx)."""

    def __init__(self, device=0):
        self.lib = load_library()
        h = C.c_void_p()
        st = self.lib.clv_create(device, C.byref(h))
        if st != abi.OK:
            raise ClvError(st, "clv_create(%d) failed (no HIP device?)" % device)
        self.h = h

    def _check(self, st):
        if st != abi.OK:
            raise ClvError(st, self.lib.clv_last_error(self.h).decode())

    def close(self):
        if getattr(self, "h", None):
            self.lib.clv_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def __enter__(self):
        return self

    def __exit__(self, *a):
        self.close()

    def upload(self, scene, builder="host"):
        """scene: clovers_amd.scenefile.SceneDescription -> scene id.  builder:
        "host" (binned SAH on the host, clv_scene_upload) or "device" (the GPU
        builder, clv_scene_upload_ex with CLV_BUILD_DEVICE)."""
        desc, keep = scene.as_ctypes()
        sid = C.c_uint32()
        if builder == "host":
            self._check(self.lib.clv_scene_upload(self.h, C.byref(desc), C.byref(sid)))
        elif builder == "device":
            self._check(self.lib.clv_scene_upload_ex(self.h, C.byref(desc), abi.BUILD_DEVICE, C.byref(sid)))
        else:
            raise ValueError("builder is 'host' or 'device'")
        return sid.value

    def free(self, scene_id):
        self._check(self.lib.clv_scene_free(self.h, scene_id))

    def render(self, scene_id, opts, want_sq=False):
        """clv_render -> (xyz[H, W, 3] f32, mean of squared samples or None)."""
        W, H = opts.width, opts.height
        out = np.empty((H, W, 3), np.float32)
        sq = np.empty((H, W, 3), np.float32) if want_sq else None
        self._check(self.lib.clv_render(self.h, scene_id, C.byref(opts), out.ctypes.data,
                                        sq.ctypes.data if sq is not None else None))
        return out, sq

    @staticmethod
    def _reuse(buf, shape, what):
        if not (isinstance(buf, np.ndarray) and buf.dtype == np.float32 and buf.shape == shape
                and buf.flags.c_contiguous and buf.flags.writeable):
            raise ValueError("%s must be a writeable C-contiguous float32 array of shape %s" % (what, shape))
        return buf

    def _jobs(self, jobs, want_sq, outs_in=None):
        arr = (abi.Job * len(jobs))()
        outs = []
        if outs_in is not None and len(outs_in) != len(jobs):
            raise ValueError("outs must hold one (xyz, sq) pair per job")
        for k, jb in enumerate(jobs):
            sid, opts = jb[0], jb[1]
            cam = jb[2] if len(jb) > 2 else None
            shape = (opts.height, opts.width, 3)
            if outs_in is not None:
                out = self._reuse(outs_in[k][0], shape, "outs[%d][0]" % k)
                sq = self._reuse(outs_in[k][1], shape, "outs[%d][1]" % k) if want_sq else None
            else:
                out = np.empty(shape, np.float32)
                sq = np.empty(shape, np.float32) if want_sq else None
            arr[k].scene_id = sid
            arr[k].use_camera = 1 if cam is not None else 0
            if cam is not None:
                arr[k].camera = cam
            arr[k].opts = opts
            arr[k].xyz_out = out.ctypes.data
            arr[k].xyz_sq_out = sq.ctypes.data if sq is not None else None
            outs.append((out, sq))
        return arr, outs

    def tuning(self):
        t = abi.Tuning()
        self._check(self.lib.clv_tuning_get(self.h, C.byref(t)))
        return {k: getattr(t, k) for k, _ in abi.Tuning._fields_ if k != "_pad"}

    def set_tuning(self, **kw):
        t = abi.Tuning()
        self._check(self.lib.clv_tuning_get(self.h, C.byref(t)))
        for k, v in kw.items():
            setattr(t, k, v)
        self._check(self.lib.clv_tuning_set(self.h, C.byref(t)))

    def autotune(self, jobs, trial_samples=0):
        """clv_autotune over the batch `jobs` (as render_batch); returns the kept tuning."""
        arr, _ = self._jobs(jobs, False)
        t = abi.Tuning()
        self._check(self.lib.clv_autotune(self.h, arr, len(jobs), trial_samples, C.byref(t)))
        return {k: getattr(t, k) for k, _ in abi.Tuning._fields_ if k != "_pad"}

    # -- guiding network probes
    def guide_reset(self, seed=1):
        self._check(self.lib.clv_guide_reset(self.h, seed))

    def guide_params(self):
        p = np.zeros(abi.GUIDE_NPARAM, np.float32)
        self._check(self.lib.clv_guide_params(self.h, p.ctypes.data, p.size))
        return p

    def guide_set_params(self, params):
        p = np.ascontiguousarray(params, np.float32)
        self._check(self.lib.clv_guide_set_params(self.h, p.ctypes.data, p.size))

    def guide_eval(self, inputs):
        """inputs [n, 7] -> (raw outputs [n, 40], lobes [n, 8, 5])"""
        x = np.ascontiguousarray(inputs, np.float32)
        n = x.shape[0]
        raw = np.zeros((n, abi.GUIDE_OUT), np.float32)
        lob = np.zeros((n, abi.GUIDE_OUT), np.float32)
        self._check(self.lib.clv_guide_eval(self.h, x.ctypes.data, n, raw.ctypes.data, lob.ctypes.data))
        return raw, lob.reshape(n, 8, 5)

    def guide_grad(self, samples):
        """samples [n, 11] -> mean loss gradient [GUIDE_NPARAM]"""
        x = np.ascontiguousarray(samples, np.float32)
        g = np.zeros(abi.GUIDE_NPARAM, np.float32)
        self._check(self.lib.clv_guide_grad(self.h, x.ctypes.data, x.shape[0], g.ctypes.data))
        return g

    def render_batch(self, jobs, want_sq=False, outs=None):
        """clv_render_batch.  jobs: list of (scene_id, opts) or (scene_id, opts,
        camera) with camera an abi.CameraInit replacing the scene's camera.
        Returns [(xyz[H, W, 3], sq or None)] in job order.  outs: the list a
        previous call returned, to be overwritten instead of allocating new
        arrays (a caller's framebuffers)."""
        arr, outs = self._jobs(jobs, want_sq, outs)
        self._check(self.lib.clv_render_batch(self.h, arr, len(jobs)))
        return outs

    def primary_hits(self, scene_id, opts):
        W, H = opts.width, opts.height
        ids = np.empty((H, W), np.uint32)
        ts = np.empty((H, W), np.float32)
        self._check(self.lib.clv_primary_hits(self.h, scene_id, C.byref(opts), ids.ctypes.data, ts.ctypes.data))
        return ids, ts

    def render_debug(self, scene_id, opts, mode):
        """clv_render_debug: abi.MODE_NORMAL_MAP / MODE_BVH_TEST_COUNT /
        MODE_PRIMITIVE_TEST_COUNT image, Xyz<E> [H, W, 3]."""
        img = np.empty((opts.height, opts.width, 3), np.float32)
        self._check(self.lib.clv_render_debug(self.h, scene_id, C.byref(opts), int(mode), img.ctypes.data))
        return img

    def counters(self):
        c = abi.Counters()
        self._check(self.lib.clv_counters_get(self.h, C.byref(c)))
        return {k: getattr(c, k) for k, _ in abi.Counters._fields_ if k != "_pad"}


def plan_passes(opts_list, target_paths=1 << 22, guide_train_spp=4, guide_rounds=16, guide_warmup=0):
    """clv_plan_passes (host only): the wavefront passes clv_render_batch would
    run for jobs with these render options -> list of dicts (pass, job,
    samples, sample_base, pass_paths, train)."""
    lib = load_library()
    jobs = (abi.Job * len(opts_list))()
    for k, o in enumerate(opts_list):
        jobs[k].opts = o
    t = abi.Tuning()
    t.target_paths, t.guide_train_spp, t.guide_rounds = target_paths, guide_train_spp, guide_rounds
    t.guide_warmup = guide_warmup
    n_items, n_passes = C.c_uint32(), C.c_uint32()
    st = lib.clv_plan_passes(jobs, len(opts_list), C.byref(t), None, 0, C.byref(n_items), C.byref(n_passes))
    if st != abi.OK:
        raise ClvError(st, "clv_plan_passes rejected the jobs")
    items = (abi.PassItem * max(1, n_items.value))()
    st = lib.clv_plan_passes(jobs, len(opts_list), C.byref(t), items, n_items.value, C.byref(n_items),
                             C.byref(n_passes))
    if st != abi.OK:
        raise ClvError(st, "clv_plan_passes rejected the jobs")
    return [{"pass": it.pass_, "job": it.job, "samples": it.samples, "sample_base": it.sample_base,
             "pass_paths": it.pass_paths, "train": it.train, "warmup": it.warmup} for it in items[:n_items.value]]


def draw(scene, width, height, samples, max_depth, seed=1, device=0, **kw):
    """draw_cpu::draw for RenderMode::PathTracing: scene -> XYZ<E> pixel buffer [H, W, 3]."""
    with Renderer(device) as r:
        sid = r.upload(scene)
        out, _ = r.render(sid, abi.render_opts(width, height, samples, max_depth, seed=seed, **kw))
        return out
