"""What the renderer is timed on: whole calls through the package's public entry points.

Each case is a render, a probe or a scene upload as a program using `clovers_amd.Renderer` makes it, with
the launch shapes a new context has (nothing is tuned beforehand).  The scenes are the package's seeded
synthetic ones; sizes, samples per pixel and depths are those of its configurations, or span the range
around them.  `prepare` creates the context and uploads the scenes, which a program does once; `run` is
one call as the program repeats it.
"""
import math

import numpy as np
import torch

import clovers_amd
from clovers_amd import abi, synth


def listed():
    return [
        # the Cornell configuration: a thumbnail or an editor's preview; 1M samples do not fill the GPU,
        # so launches and the host's part of the call count
        {"name": "cornell_preview", "kind": "cornell", "width": 256, "height": 256, "samples": 16, "depth": 8},
        # an editor that refines an image while it is looked at: one sample per pixel and call, every
        # call with the next sample index, so that no call repeats another
        {"name": "spheres_progressive", "kind": "progressive", "width": 640, "height": 360, "samples": 1, "depth": 16,
         "calls": 4},
        # the sphere-field configuration: the final frame of a small scene, whose tree fits in LDS
        {"name": "spheres_1080p", "kind": "spheres", "width": 1920, "height": 1080, "samples": 64, "depth": 16},
        # moving spheres at an odd size, sums in float64 and second moments returned: a reference image
        # with error bars
        {"name": "motion_f64_odd", "kind": "motion", "width": 1023, "height": 577, "samples": 9, "depth": 16},
        # the large-mesh configuration: 4 views of a 1M-triangle thin-film blob in one batch
        {"name": "mesh_1m_4views", "kind": "mesh", "width": 1920, "height": 1080, "samples": 8, "depth": 12,
         "freq": 224, "views": 4},
        # the caustics configuration, plain and guided (the guided render trains its network)
        {"name": "prism_plain", "kind": "prism", "width": 1024, "height": 1024, "samples": 64, "depth": 24,
         "guiding": False},
        {"name": "prism_guided", "kind": "prism", "width": 1024, "height": 1024, "samples": 64, "depth": 24,
         "guiding": True},
        # a render queue: scenes of uneven size, resolution and sample count, guided, in one batch
        {"name": "batch_uneven_guided", "kind": "batch", "count": 6, "max_tris": 300000, "max_side": 640,
         "max_samples": 64, "depth": 12, "guiding": True},
        # checker textures, a cone light, moving spheres and instance chains in one room
        {"name": "features_room", "kind": "features", "width": 800, "height": 600, "samples": 32, "depth": 12},
        # smoke and fog: constant media with Isotropic phase functions
        {"name": "media_room", "kind": "media", "width": 641, "height": 479, "samples": 16, "depth": 12},
        # picking and depth: object ids, distances and normals of the first hits of a whole frame
        {"name": "hits_1080p", "kind": "hits", "width": 1920, "height": 1080},
        # opening a scene: a mesh uploaded with the GPU tree builder, looked at once, and freed
        {"name": "upload_mesh_82k", "kind": "upload", "freq": 64, "width": 256, "height": 256},
    ]


#: Per kind: pixels (least, most), samples per pixel, depth, and the most samples of a call.
RANGES = {
    "cornell": ((48 * 48, 1024 * 1024), (1, 64), (4, 16), 1 << 24),
    "progressive": ((160 * 90, 1280 * 720), (1, 2), (8, 24), 1 << 20),
    "spheres": ((256 * 144, 1920 * 1080), (1, 64), (8, 24), 1 << 26),
    "motion": ((256 * 144, 1280 * 720), (1, 32), (8, 24), 1 << 24),
    "mesh": ((256 * 144, 1920 * 1080), (1, 16), (6, 16), 1 << 24),
    "prism": ((256 * 256, 1024 * 1024), (16, 64), (12, 24), 1 << 26),
    "features": ((256 * 144, 1280 * 720), (1, 64), (6, 16), 1 << 24),
    "media": ((256 * 144, 1280 * 720), (1, 32), (6, 16), 1 << 23),
    "hits": ((160 * 90, 1920 * 1080), None, None, None),
    "upload": ((64 * 64, 512 * 512), None, None, None),
}


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(sorted(RANGES) + ["batch"])
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(2, 6), "max_tris": int(_log(rng, 4000, 300000)),
                "max_side": rng.randint(200, 640), "max_samples": rng.randint(33, 64), "depth": rng.randint(6, 16),
                "guiding": rng.random() < 0.7}
    pixels, samples, depth, most = RANGES[kind]
    n, aspect = _log(rng, *pixels), rng.uniform(0.7, 2.0)
    case = {"kind": kind, "width": max(8, int(math.sqrt(n * aspect))), "height": max(8, int(math.sqrt(n / aspect)))}
    n = case["width"] * case["height"]
    if kind == "mesh":
        case.update(freq=int(_log(rng, 40, 224)), views=rng.randint(1, 4))
        most //= case["views"]
    if kind == "upload":
        case["freq"] = int(_log(rng, 16, 90))
    if kind == "progressive":
        case["calls"] = 4
    if kind == "prism":
        case["guiding"] = rng.random() < 0.6
    if samples:
        case["samples"] = min(max(1, int(_log(rng, samples[0], samples[1] + 1))), max(1, most // n))
        case["depth"] = rng.randint(*depth)
    return case


def _scene(case, seed):
    kind = case["kind"]
    if kind == "cornell":
        return synth.cornell()
    if kind in ("spheres", "progressive", "hits"):
        return synth.spheres(seed=seed)
    if kind == "motion":
        return synth.spheres(seed=seed, moving=True)
    if kind in ("mesh", "upload"):
        return synth.mesh(freq=case["freq"], seed=seed % 1000003)
    if kind == "prism":
        return synth.prism()
    return {"features": synth.features, "media": synth.media}[kind]()


def _batch(case, seed):
    """(scene, side, samples) of each job: triangles, resolution and samples log-uniform, as the package's
    64-scene batch has them, up to the case's own limits; the seed decides what the scenes hold"""
    r = np.random.Generator(np.random.PCG64(case["max_tris"] + case["max_side"]))
    log = lambda lo, hi: math.exp(r.uniform(math.log(lo), math.log(hi)))  # noqa: E731
    out = []
    for k in range(case["count"]):
        tris = int(log(1000, case["max_tris"]))
        side, spp = int(log(128, case["max_side"])), int(log(16, case["max_samples"]))
        out.append((synth.batch_scene(seed + k, n_tris=tris)[0], side, spp))
    return out


def prepare(case, seed):
    r = clovers_amd.Renderer(0)
    st = {"case": case, "renderer": r}
    kind, depth = case["kind"], case.get("depth")
    if kind == "batch":
        guide = int(case["guiding"])
        st["jobs"] = [(r.upload(scene), abi.render_opts(side, side, spp, depth, seed=seed, guiding=guide))
                      for scene, side, spp in _batch(case, seed)]
    elif kind == "upload":
        st["scene"] = _scene(case, seed)
        st["opts"] = abi.render_opts(case["width"], case["height"], 1, 1, seed=seed)
        return st
    else:
        W, H = case["width"], case["height"]
        opts = abi.render_opts(W, H, case.get("samples", 1), depth or 1, seed=seed,
                               guiding=int(case.get("guiding", False)), fp64_accum=int(kind == "motion"))
        sid = st["scene_id"] = r.upload(_scene(case, seed), builder="device" if kind == "mesh" else "host")
        st["opts"] = opts
        if kind == "mesh":
            st["jobs"] = [(sid, opts)] + [(sid, opts, abi.camera_init(synth.MESH_VIEWS[v], (0.0, 1.0, 0.0)))
                                          for v in range(1, case["views"])]
        if kind == "progressive":
            st["steps"] = [abi.render_opts(W, H, case["samples"], depth, seed=seed, sample_offset=k * case["samples"])
                           for k in range(case["calls"])]
    if "jobs" in st:  # the caller's framebuffers, rendered into by every call
        st["outs"] = [(np.zeros((j[1].height, j[1].width, 3), np.float32), None) for j in st["jobs"]]
    return st


def run(st):
    kind, r = st["case"]["kind"], st["renderer"]
    if "jobs" in st:
        return [img for img, _ in r.render_batch(st["jobs"], outs=st["outs"])]
    if kind == "upload":
        sid = r.upload(st["scene"], builder="device")
        ids, ts = r.primary_hits(sid, st["opts"])
        r.free(sid)
        return {"ids": ids.astype(np.int64), "ts": ts}
    if kind == "progressive":
        return [r.render(st["scene_id"], o)[0] for o in st["steps"]]
    if kind == "hits":
        ids, ts = r.primary_hits(st["scene_id"], st["opts"])
        return {"ids": ids.astype(np.int64), "ts": ts,
                "normals": r.render_debug(st["scene_id"], st["opts"], abi.MODE_NORMAL_MAP)}
    img, sq = r.render(st["scene_id"], st["opts"], want_sq=kind == "motion")
    return img if sq is None else {"xyz": img, "xyz_sq": sq}


#: Rays per camera sample and primitives of each kind's scene, roughly.
SHAPE = {"cornell": (3.0, 18), "progressive": (2.7, 490), "spheres": (2.7, 490), "motion": (2.7, 490),
         "mesh": (3.0, 0), "prism": (3.0, 16), "features": (3.5, 20), "media": (4.0, 6), "hits": (1.0, 490),
         "upload": (1.0, 0)}


def work(case):
    """Bytes: the scene read once, the images written once.  Operations: a ray meets one node of four boxes
    per level of a 4-wide tree (12 operations a box) and one primitive (60), and each hit is shaded (200)."""
    def rays(n, prims):
        return n * (math.log(max(prims, 4), 4) * 4 * 12 + 60 + 200)
    if case["kind"] == "batch":
        # means of the log-uniform ranges; 16 B a triangle corner
        mean = lambda lo, hi: (hi - lo) / math.log(hi / lo)  # noqa: E731
        tris = mean(1000, case["max_tris"])
        px = mean(128 ** 2, case["max_side"] ** 2)
        return {"bytes": case["count"] * (48 * tris + 12 * px),
                "flops": case["count"] * rays(px * mean(16, case["max_samples"]) * 2.5, tris)}
    per_sample, prims = SHAPE[case["kind"]]
    prims = prims or 20 * case["freq"] ** 2
    n = case["width"] * case["height"] * case.get("views", 1) * case.get("calls", 1)
    out = {"motion": 24, "hits": 20, "upload": 8}.get(case["kind"], 12)
    scene = prims * (48 if case["kind"] in ("mesh", "upload") else 16)
    flops = rays(n * case.get("samples", 1) * per_sample, prims)
    if case["kind"] == "upload":
        flops += prims * math.log2(prims) * 20  # a sort of the primitives and a tree over them
    return {"bytes": scene + out * n, "flops": flops}


# ---------------------------------------------------------------- exact
# The first hits have a value in 64 bits: the closest intersection of the camera's rays.  A path-traced
# image has none: it is a sum over the paths of one random stream, and the last bit of any hit decides
# where a path goes next.

M64 = (1 << 64) - 1


def _u64(x):
    return np.asarray(x, np.uint64)


def _splitmix(x):
    with np.errstate(over="ignore"):
        x = x + _u64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> _u64(30))) * _u64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> _u64(27))) * _u64(0x94D049BB133111EB)
        return x ^ (x >> _u64(31))


class _Stream:
    """One PCG32 stream per pixel, keyed by (seed, pixel, sample 0)"""

    def __init__(self, seed, pixels):
        self.s = _splitmix(_u64(seed & M64) ^ _splitmix(_u64(pixels)))
        self.next()

    def next(self):
        old = self.s
        with np.errstate(over="ignore"):
            self.s = old * _u64(6364136223846793005) + _u64(1442695040888963407)
        xs = (((old >> _u64(18)) ^ old) >> _u64(27)).astype(np.uint32)
        rot = (old >> _u64(59)).astype(np.uint32)
        return (xs >> rot) | (xs << ((np.uint32(32) - rot) & np.uint32(31)))

    def uniform(self):
        return (self.next() >> np.uint32(8)).astype(np.float64) * 2.0 ** -24


def _camera_rays(cam, W, H, seed, corner):
    """Origins and directions of a pinhole camera's rays, image rows from the top: through each pixel's
    first sample point, or through its corner"""
    f = {k: np.array([float(x) for x in getattr(cam, k)]) for k in ("look_from", "look_at", "up")}
    r, x = np.divmod(np.arange(W * H), W)
    y = H - 1 - r
    dx = dy = 0.0
    if not corner:
        s = _Stream(seed, x + y * W)
        dx, dy = s.uniform(), s.uniform()
    half = math.tan(math.radians(float(cam.vertical_fov)) / 2)
    w = f["look_from"] - f["look_at"]
    w /= np.linalg.norm(w)
    u = np.cross(f["up"], w)
    u /= np.linalg.norm(u)
    v = np.cross(w, u)
    a = (2 * (x + dx) / W - 1) * half * W / H
    b = (2 * (y + dy) / H - 1) * half
    d = a[:, None] * u + b[:, None] * v - w
    return f["look_from"], d / np.linalg.norm(d, axis=1, keepdims=True)


def _closest(objects, origin, dirs):
    """(distance, normal towards the ray, hit) of the closest sphere, quad or triangle along each ray"""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float64), device=dev)  # noqa: E731
    o, n = T(origin), len(dirs)
    kind, p = objects["kind"], objects["p"].astype(np.float64)
    sph, flat = p[kind == abi.OBJ_SPHERE], p[kind != abi.OBJ_SPHERE]
    tri = kind[kind != abi.OBJ_SPHERE] == abi.OBJ_TRIANGLE
    q, e1, e2 = flat[:, 0:3], flat[:, 3:6].copy(), flat[:, 6:9].copy()
    e1[tri] -= q[tri]
    e2[tri] -= q[tri]
    nn = np.cross(e1, e2)
    ln = np.linalg.norm(nn, axis=1, keepdims=True)
    planes = [T(a) for a in (q, e1, e2, nn / ln, nn / ln ** 2)]
    tri = torch.as_tensor(tri, device=dev)
    C, R = T(sph[:, 0:3]), T(sph[:, 3])
    inf = float("inf")
    ts, ns = np.empty(n), np.empty((n, 3))
    step = max(1, 20_000_000 // (len(sph) + len(flat)))
    for k in range(0, n, step):
        d = T(dirs[k:k + step])
        best = torch.full((len(d),), inf, dtype=torch.float64, device=dev)
        normal = torch.zeros_like(d)
        if len(sph):
            oc = o - C
            hb = d @ oc.T
            root = (hb * hb - (oc * oc).sum(1) + R * R).sqrt()  # NaN where the ray passes by
            t = torch.where(-hb - root > 1e-3, -hb - root, -hb + root)
            t = torch.where(t > 1e-3, t, inf).nan_to_num(nan=inf, posinf=inf)
            best, at = t.min(1)
            normal = (o + torch.where(best < inf, best, 0.0)[:, None] * d - C[at]) / R[at, None]
        if len(flat):
            Q, U, V, N, Wn = planes
            den = d @ N.T
            t = ((Q - o) * N).sum(1) / den
            # plane coordinates of o + t d: linear in t, so no point per ray and plane is kept
            a0, a1 = (torch.cross(o - Q, V, dim=1) * Wn).sum(1), d @ torch.cross(V, Wn, dim=1).T
            b0, b1 = (torch.cross(U, o - Q, dim=1) * Wn).sum(1), d @ torch.cross(Wn, U, dim=1).T
            a, b = a0 + t * a1, b0 + t * b1
            ok = (den.abs() >= 1e-4) & (t >= 1e-3) & (a >= 0) & (b >= 0) & (a <= 1) & (b <= 1) & (~tri | (a + b <= 1))
            t, at = torch.where(ok, t, inf).min(1)
            nearer = t < best
            best = torch.where(nearer, t, best)
            normal = torch.where(nearer[:, None], N[at], normal)
        ts[k:k + step] = best.cpu().numpy()
        ns[k:k + step] = torch.where((d * normal).sum(1, keepdim=True) < 0, normal, -normal).cpu().numpy()
    return ts, ns, np.isfinite(ts)


def _normal_colors(ns, hit):
    """A normal's colour (x and y over [-1, 1], z towards the viewer), as linear sRGB, in XYZ with white E"""
    n = ns * [-1.0, 1.0, -1.0]
    rgb = np.stack([0.5 + 0.5 * n[:, 0], 0.5 + 0.5 * n[:, 1], np.maximum(n[:, 2], 0.0)], 1) * hit[:, None]
    xy = np.array([[0.64, 0.33], [0.30, 0.60], [0.15, 0.06]])
    P = np.stack([xy[:, 0] / xy[:, 1], np.ones(3), (1 - xy[:, 0] - xy[:, 1]) / xy[:, 1]])
    white = np.array([0.95047, 1.0, 1.08883])
    B = np.array([[0.8951, 0.2664, -0.1614], [-0.7502, 1.7135, 0.0367], [0.0389, -0.0685, 1.0296]])
    to_e = np.linalg.inv(B) @ np.diag(B.sum(1) / (B @ white)) @ B
    return rgb @ (to_e @ (P * np.linalg.solve(P, white))).T


def exact(case, seed):
    if case["kind"] not in ("hits", "upload"):
        return None
    W, H = case["width"], case["height"]
    scene = _scene(case, seed)
    cam, objects = scene.as_ctypes()[0].camera, scene.objects
    o, d = _camera_rays(cam, W, H, seed, corner=False)
    ts, _, _ = _closest(objects, o, d)
    out = {"ids": None, "ts": ts.reshape(H, W)}
    if case["kind"] == "hits":
        o, d = _camera_rays(cam, W, H, seed, corner=True)
        _, ns, hit = _closest(objects, o, d)
        out["normals"] = _normal_colors(ns, hit).reshape(H, W, 3)
    return out
