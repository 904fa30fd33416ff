"""Performance cases: the calls that a program makes of this library, over the
range of sizes and options that it declares.

A case is a dict of plain values.  Its "path" says which entry point it takes:

  viewer   Renderer.render_mesh of a host mesh and Renderer.get_back_buffer,
           with the camera, light and shader set again: what an interactive
           viewer does per frame.
  frame    Renderer.render_mesh of a mesh resident in device memory, colour,
           depth and triangle IDs left there; one call per frame, eager or as a
           captured graph ("graph"), 2^"msaa" samples per pixel.
  noalloc  edxr_render_mesh_noalloc into the caller's own tensors: a serving
           loop or a caller that may not allocate.
  batch    Renderer.render_batch of many independent jobs.
  train    diff.render_views of several views, an L2 loss against an image and
           the gradients of every vertex plane, the light and the material.

Scenes are the library's seeded ones ("sphere", "heightfield", "grid": a grid
of spheres with the eye close to the surface of one, so that triangles cross
the near plane; train: a sphere above a heightfield).  Every seed gives other
geometry or vertex colours, another light and a slightly moved camera.
"""
import ctypes as C
import math

import numpy as np
import torch

from edxraster_amd import Mesh, Renderer, configs, diff, look_at, perspective, raster_matrix
from edxraster_amd import _lib as L

MATERIAL = (0.2, 3.0, 3.0, 32.0)  # ambient, kd, ks, shininess of the train cases


def listed():
    return [
        # An interactive viewer's frame of a small host mesh, read back to be
        # shown: uploads, launches and the copy back set its time.
        dict(name="viewer_sphere_800x600", path="viewer", scene="sphere", n=32, width=800, height=600),
        # The smallest call with everything resident: launches and latency.
        dict(name="frame_sphere_800x600", path="frame", scene="sphere", n=32, width=800, height=600,
             shader=2, filter=2, msaa=0, graph=False),
        # A service's frame into its own buffers, ragged in every size: a
        # resolution that is no multiple of a tile, an odd vertex count.
        dict(name="noalloc_heightfield_1283x719", path="noalloc", scene="heightfield", n=223, width=1283, height=719,
             shader=1),
        # The standard scene: 2.1M triangles at full HD, captured.
        dict(name="frame_grid_1920x1080", path="frame", scene="grid", n=64, width=1920, height=1080,
             shader=2, filter=2, msaa=0, graph=True),
        # The same with four samples per pixel, as a final frame is rendered.
        dict(name="frame_grid_1920x1080_4x", path="frame", scene="grid", n=64, width=1920, height=1080,
             shader=2, filter=2, msaa=2, graph=True),
        # The largest frame: 10M triangles at 4K, most smaller than a pixel.
        dict(name="frame_heightfield_3840x2160", path="frame", scene="heightfield", n=2236, width=3840, height=2160,
             shader=2, filter=2, msaa=0, graph=True),
        # The viewer's default shader and filter (textured, trilinear), 2M
        # triangles of a few pixels each, at QHD.
        dict(name="frame_textured_2560x1440", path="frame", scene="heightfield", n=1001, width=2560, height=1440,
             shader=3, filter=2, msaa=0, graph=True),
        # Its anisotropic filter on larger triangles, eager.
        dict(name="frame_aniso8_1920x1080", path="frame", scene="heightfield", n=200, width=1920, height=1080,
             shader=3, filter=4, msaa=0, graph=False),
        # A queue of uneven jobs of 1K to 500K triangles at 256^2 to 1024^2,
        # in one captured sequence.
        dict(name="batch_256", path="batch", jobs=256, tmin=1000, tmax=500000, res=1024, graph=True),
        # A short queue of thumbnails, different every time, hence eager.
        dict(name="batch_17_thumbnails", path="batch", jobs=17, tmin=1000, tmax=20000, res=256, graph=False),
        # One optimisation step on many views (forward, loss, backward).
        dict(name="train_64x512", path="train", views=64, res=512, n=71),
        # A small one, as a fit of a few views starts.
        dict(name="train_4x200", path="train", views=4, res=200, n=41),
    ]


def _log_int(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    path = rng.choice(["viewer", "frame", "frame", "frame", "noalloc", "batch", "train", "train"])
    width = _log_int(rng, 200, 3840)
    height = max(120, min(2160, int(width * rng.uniform(0.45, 0.8))))
    if path == "viewer":
        return dict(path=path, scene=rng.choice(["sphere", "heightfield"]), n=_log_int(rng, 12, 120),
                    width=min(width, 1300), height=min(height, 900))
    if path == "noalloc":
        return dict(path=path, scene=rng.choice(["sphere", "heightfield"]), n=_log_int(rng, 12, 180),
                    width=min(width, 1500), height=min(height, 900), shader=rng.choice([0, 1, 2]))
    if path == "batch":
        tmax = _log_int(rng, 3000, 300000)
        return dict(path=path, jobs=_log_int(rng, 3, 128), tmin=1000, tmax=tmax, res=rng.choice([100, 256, 513, 1024]),
                    graph=rng.random() < 0.5)
    if path == "train":
        return dict(path=path, views=_log_int(rng, 1, 40), res=_log_int(rng, 64, 512), n=_log_int(rng, 9, 150))
    scene = rng.choice(["sphere", "heightfield", "heightfield", "grid"])
    n = {"sphere": _log_int(rng, 16, 500), "heightfield": _log_int(rng, 20, 1800),
         "grid": _log_int(rng, 8, 64)}[scene]
    shader = rng.choice([0, 1, 2, 2, 3]) if scene == "heightfield" else rng.choice([0, 1, 2])
    msaa = 0 if shader == 3 or width > 2200 else rng.choice([0, 0, 0, 1, 2, 3])
    return dict(path=path, scene=scene, n=n, width=width, height=height, shader=shader,
                filter=rng.choice([0, 1, 2, 2, 3, 5]), msaa=msaa, graph=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _unit(rng):
    v = rng.normal(size=3)
    return v / np.linalg.norm(v)


def _mesh(scene, n, rng, textured):
    a, b = (int(x) for x in rng.integers(1, 1 << 30, 2))
    if scene == "sphere":
        m = Mesh.sphere(2 * n, n, 1.0, (0.0, 0.0, 0.0), color_seed=a)
    elif scene == "grid":
        m = Mesh.sphere_grid(16, n, seed=a)
    else:
        m = Mesh.load_heightfield(n, 0.2, height_seed=a, color_seed=b)
    if textured:
        m.tu = ((m.px + 1.0) * 16.0).astype(np.float32)
        m.tv = ((m.pz + 1.0) * 16.0).astype(np.float32)
        m.tex_ids = ((np.arange(m.num_triangles) // 2) % 2).astype(np.uint32)
    return m


def _camera(scene, n, mesh, rng):
    """(eye, at) of the scene, moved a little by the seed."""
    j = rng.uniform(-0.03, 0.03, 3)
    if scene == "sphere":
        return np.array([0.0, 0.0, -3.0]) + j, np.zeros(3)
    if scene == "heightfield":
        return np.array([0.0, 1.2, -1.6]) + j, np.zeros(3)
    # beside the near pole of sphere (8, 8), 0.05 inside its surface
    pole = (8 * 16 + 8) * (n + 1) * (n + 1)
    c = np.array([mesh.px[pole], 0.0, mesh.pz[pole]], np.float64)
    eye = c + (float(mesh.py[pole]) - 0.05) * np.array([0.0, 0.0, -1.0])
    return eye, eye + 50.0 * np.array([-1.0, -0.08 + j[0], j[1]])


def _view(width, height, eye, at, up=(0.0, 1.0, 0.0)):
    return look_at(eye, at, up), perspective(60.0, width / height, 0.1, 100.0), raster_matrix(width, height)


def _scene(case, seed):
    """Mesh, camera matrices and light of a single-frame case."""
    rng = np.random.default_rng(seed)
    mesh = _mesh(case["scene"], case["n"], rng, case.get("shader") == L.SHADER_TEXTURED_LAMBERT)
    eye, at = _camera(case["scene"], case["n"], mesh, rng)
    mv, proj, raster = _view(case["width"], case["height"], eye, at)
    light = tuple(float(x) for x in np.array([1.0, 1.0, -1.0]) + rng.uniform(-0.2, 0.2, 3))
    return configs.Workload("case", case["width"], case["height"], mesh, mv, proj, raster, light=light,
                            shader=case.get("shader", L.SHADER_VC_BLINN_PHONG),
                            shininess={0: 0.0, 1: 200.0, 2: 32.0, 3: 0.0}[case.get("shader", 2)])


def _batch_scenes(case, seed):
    jobs = []
    sizes = np.random.default_rng(case["jobs"])  # the case's own: every seed's queue has the same sizes
    for k in range(case["jobs"]):
        rng = np.random.default_rng([seed, k])
        target = math.exp(sizes.uniform(math.log(case["tmin"]), math.log(case["tmax"])))
        res = max(64, case["res"] >> int(sizes.integers(3)))
        d = _unit(rng)
        if sizes.random() < 0.5:
            mesh = _mesh("sphere", max(2, round(math.sqrt(target / 4.0))), rng, False)
        else:
            mesh = _mesh("heightfield", max(3, round(1.0 + math.sqrt(target / 2.0))), rng, False)
        up = (0.0, 1.0, 0.0) if abs(d[1]) < 0.99 else (0.0, 0.0, 1.0)
        mv, proj, raster = _view(res, res, 3.0 * d, np.zeros(3), up)
        jobs.append(configs.Workload("job", res, res, mesh, mv, proj, raster, light=tuple(map(float, _unit(rng)))))
    return jobs


def _train_scene(case, seed):
    """Mesh, views, light and the target image (device tensor) of a train case."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    hf = _mesh("heightfield", n, rng, False)
    sph = Mesh.sphere(max(6, 8 * n // 7), max(4, 9 * n // 10), 0.35, (0.0, 0.55, 0.0), color_seed=int(rng.integers(1, 1 << 30)))
    mesh = Mesh.merge(hf, sph)
    at, el = np.array([0.0, 0.15, 0.0]), math.radians(30.0 + rng.uniform(-3, 3))
    light = tuple(float(x) for x in np.array([1.0, 1.0, -1.0]) + rng.uniform(-0.2, 0.2, 3))
    views, phase = [], rng.uniform(0, 2 * math.pi)
    for k in range(case["views"]):
        az = phase + 2 * math.pi * k / case["views"]
        eye = at + 3.0 * np.array([math.cos(el) * math.sin(az), math.sin(el), -math.cos(el) * math.cos(az)])
        mv, proj, raster = _view(case["res"], case["res"], eye, at)
        views.append(configs.Workload("view", case["res"], case["res"], mesh, mv, proj, raster, light=light))
    coarse = torch.from_numpy(rng.uniform(0.1, 0.9, (len(views), 3, 9, 9)).astype(np.float32)).cuda()
    target = torch.nn.functional.interpolate(coarse, size=(case["res"], case["res"]), mode="bilinear", align_corners=True)
    return mesh, views, light, target.permute(0, 2, 3, 1).contiguous()


def _device_mesh(mesh):
    """(edxr_mesh over device memory, the tensors that hold it)."""
    up = lambda a: None if a is None else torch.from_numpy(a if a.dtype == np.float32 else a.view(np.int32)).cuda()
    planes, idx = [up(a) for a in mesh.planes()], up(mesh.indices)
    extra = [up(a) for a in (mesh.tu, mesh.tv, mesh.tex_ids)]
    ptr = lambda t, kind: None if t is None else C.cast(C.c_void_p(t.data_ptr()), kind)
    m = L.Mesh(*[ptr(t, L.F) for t in planes], ptr(idx, L.U32), mesh.num_vertices, mesh.num_triangles, L.MEM_DEVICE,
               ptr(extra[0], L.F), ptr(extra[1], L.F), ptr(extra[2], L.U32))
    return m, (planes, idx, extra)


class _Buffer:
    """A renderer's device buffer for torch.as_tensor, which keeps the renderer alive."""

    def __init__(self, renderer, address, shape, typestr):
        self.renderer = renderer
        self.__cuda_array_interface__ = {"data": (int(address), False), "shape": tuple(shape), "typestr": typestr,
                                         "strides": None, "version": 2}


def _buffers(renderer, addresses, pixels, planes):
    color, depth, ids = addresses
    shape = pixels if planes == 1 else (planes,) + pixels
    t = lambda address, shape, typestr: torch.as_tensor(_Buffer(renderer, address, shape, typestr), device="cuda")
    return {"color": t(color, pixels + (4,), "|u1"), "depth": t(depth, shape, "<f4"), "ids": t(ids, shape, "<i4")}


def _textures():
    return [configs.checker_texture(1024, 16, 21), configs.checker_texture(1024, 32, 22)]


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        jobs = _batch_scenes(case, seed)
        meshes = [_device_mesh(w.mesh) for w in jobs]
        r = Renderer(64, 64)
        r.set_graph(case["graph"])
        arr = (L.Job * len(jobs))(*[w.job(mesh=m) for w, (m, _) in zip(jobs, meshes)])
        torch.cuda.synchronize()
        return dict(path=path, r=r, jobs=arr, keep=meshes, pixels=sum(w.width * w.height for w in jobs), out=None)
    if path == "train":
        mesh, views, light, target = _train_scene(case, seed)
        idx, planes = diff.mesh_tensors(mesh)
        for t in planes:
            t.requires_grad_(True)
        lt = torch.tensor(light, dtype=torch.float32, requires_grad=True)
        mt = torch.tensor(MATERIAL, dtype=torch.float32, requires_grad=True)
        return dict(path=path, r=Renderer(64, 64), views=views, idx=idx, planes=planes, light=lt, material=mt,
                    target=target)
    w = _scene(case, seed)
    if w.shader == L.SHADER_TEXTURED_LAMBERT:
        w.textures, w.tex_filter = _textures(), case["filter"]
    r = Renderer(w.width, w.height)
    if path == "viewer":
        return dict(path=path, r=r, w=w)
    mesh, keep = _device_mesh(w.mesh)
    S = 1 << case.get("msaa", 0)
    if S > 1:
        r.set_msaa_mode(case["msaa"])
    w.apply(r)
    w.mesh = None
    state = dict(path=path, r=r, w=w, mesh=mesh, keep=keep)
    pixels = (w.height, w.width)
    if path == "noalloc":
        state["out"] = {"color": torch.empty(pixels + (4,), dtype=torch.uint8, device="cuda"),
                        "depth": torch.empty(pixels, dtype=torch.float32, device="cuda"),
                        "ids": torch.empty(pixels, dtype=torch.int32, device="cuda")}
        state["args"] = [C.c_void_p(state["out"][k].data_ptr()) for k in ("color", "depth", "ids")]
    else:
        r.set_graph(case["graph"])
        state["out"] = _buffers(r, r.device_buffers(), pixels, S)
    torch.cuda.synchronize()
    return state


def run(state):
    path, r = state["path"], state["r"]
    if path == "viewer":
        state["w"].apply(r)
        r.render_mesh(state["w"].mesh)
        return r.get_back_buffer()
    if path == "frame":
        r.render_mesh(state["mesh"])
        return state["out"]
    if path == "noalloc":
        rc = L.lib().edxr_render_mesh_noalloc(r.ctx, C.byref(state["mesh"]), *state["args"])
        if rc != L.EDXR_OK:
            raise L.EdxrError(rc, L.lib().edxr_last_error(r.ctx).decode())
        return state["out"]
    if path == "batch":
        r.render_batch(state["jobs"])
        if state["out"] is None:  # the buffers exist after the first batch
            state["out"] = _buffers(r, r.batch_device_buffers()[:3], (state["pixels"],), 1)
        return state["out"]
    image = diff.render_views(r, state["views"], state["idx"], *state["planes"], state["light"], state["material"])
    loss = ((image - state["target"]) ** 2).sum()
    grads = torch.autograd.grad(loss, [*state["planes"], state["light"], state["material"]])
    return {"image": image.detach(), "grads": list(grads)}


# ---------------------------------------------------------------------------
# What a pass cannot do without: the mesh read once, the images written once.
# ---------------------------------------------------------------------------
def _counts(scene, n):
    """(vertices, triangles)"""
    return {"sphere": ((n + 1) * (2 * n + 1), 4 * n * n), "heightfield": (n * n, 2 * (n - 1) ** 2),
            "grid": (256 * (n + 1) ** 2, 512 * n * n)}[scene]


def work(case):
    path = case["path"]
    if path == "batch":  # the mean of the log-uniform triangle counts and of the three resolutions
        t = (case["tmax"] - case["tmin"]) / math.log(case["tmax"] / case["tmin"]) * case["jobs"]
        v, p, s, tex = 0.5 * t, case["jobs"] * sum(max(64, case["res"] >> k) ** 2 for k in range(3)) / 3, 1, 0
    elif path == "train":
        n, views = case["n"], case["views"]
        sl, st = max(6, 8 * n // 7), max(4, 9 * n // 10)
        v, t, p = n * n + (sl + 1) * (st + 1), 2 * (n - 1) ** 2 + 2 * sl * st, views * case["res"] ** 2
        # forward: float image out; loss and backward: image and target in, per-pixel gradient in double precision
        return {"bytes": 2 * (36 * v + 12 * t) + 36 * v + 36 * p, "flops": 60 * v * views + 40 * t * views + 500 * p}
    else:
        v, t = _counts(case["scene"], case["n"])
        p, s = case["width"] * case["height"], 1 << case.get("msaa", 0)
        tex = case.get("shader") == L.SHADER_TEXTURED_LAMBERT
    return {"bytes": (36 + 8 * tex) * v + (12 + 4 * tex) * t + (4 + 8 * s) * p, "flops": 60 * v + 40 * t + (120 + 20 * s) * p}


# ---------------------------------------------------------------------------
# The same outputs in 64 bits, by plain torch and numpy.  Which pixels a
# triangle covers is a decision on whole numbers, the vertices' positions in
# 28.4 fixed point, and those are defined by float32 transforms; everything
# after that decision is computed in float64.
# ---------------------------------------------------------------------------
_SAMPLES = [[(0, 0)], [(4, 4), (-4, -4)], [(-2, -6), (6, -2), (-6, 2), (2, 6)],
            [(1, -3), (-1, 3), (5, 1), (-3, -5), (-5, 5), (-7, -1), (3, 7), (7, -7)]]


def _transform32(m, p):
    """m (4x4) times (p, 1) in float32, in the order of the rasteriser's definition."""
    return [((m[i, 0] * p[0] + m[i, 1] * p[1]) + m[i, 2] * p[2]) + m[i, 3] * np.float32(1.0) for i in range(4)]


def _mvp32(w):
    a, b = np.asarray(w.proj, np.float32).reshape(4, 4), np.asarray(w.mv, np.float32).reshape(4, 4)
    out = np.zeros((4, 4), np.float32)
    for i in range(4):
        for j in range(4):
            out[i, j] = ((a[i, 0] * b[0, j] + a[i, 1] * b[1, j]) + a[i, 2] * b[2, j]) + a[i, 3] * b[3, j]
    return out


class _Visible:
    """Snapped triangles of a view and the pixels that they cover."""

    def __init__(self, w, mesh):
        self.w, self.h = w.width, w.height
        m, p = _mvp32(w), [mesh.px, mesh.py, mesh.pz]
        with np.errstate(all="ignore"):
            c = _transform32(m, p)
            outside = [c[0] < -c[3], c[0] > c[3], c[1] < -c[3], c[1] > c[3], c[2] > c[3], c[2] < 0]
            s = _transform32(np.asarray(w.raster, np.float32).reshape(4, 4), [c[k] / c[3] for k in range(3)])
            xy = np.stack([np.trunc(np.nan_to_num(s[k] * np.float32(16.0))).astype(np.int64) for k in (0, 1)], 1)
        code = sum((o.astype(np.int64) << k) for k, o in enumerate(outside))
        idx = mesh.indices.reshape(-1, 3).astype(np.int64)
        k = code[idx]
        inside = (k == 0).all(1)
        # a triangle that crosses a plane is cut up, and the pieces' corners
        # snapped: there is no plain form of that
        self.clipped = bool((~inside & ((k[:, 0] & k[:, 1] & k[:, 2]) == 0)).any())
        tri = np.nonzero(inside)[0]
        X, Y = xy[idx[tri], 0], xy[idx[tri], 1]
        det = (X[:, 0] - X[:, 2]) * (Y[:, 1] - Y[:, 2]) - (X[:, 2] - X[:, 1]) * (Y[:, 2] - Y[:, 0])
        keep = det > 0
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
        self.tri, self.X, self.Y, self.det = dev(tri[keep]), dev(X[keep]), dev(Y[keep]), dev(det[keep]).double()
        clip = [m64 @ np.stack([*(q.astype(np.float64) for q in p), np.ones(len(p[0]))]) for m64 in [m.astype(np.float64)]][0]
        self.Z = dev((clip[2] / clip[3])[idx[tri[keep]]])
        X, Y = self.X, self.Y
        lo = lambda a, size: a.amin(1).div(16, rounding_mode="floor").clamp(0, size)
        hi = lambda a, size: a.amax(1).div(16, rounding_mode="floor").clamp(-1, size - 1)
        self.x0, self.y0 = lo(X, self.w), lo(Y, self.h)
        self.nx = (hi(X, self.w) - self.x0 + 1).clamp(min=0)
        self.count = self.nx * (hi(Y, self.h) - self.y0 + 1).clamp(min=0)

    def pairs(self, offset):
        """Chunks of (row of the triangle arrays, pixel, l0, l1, depth) for the sample at
        `offset` from the pixel's centre, over every covered (triangle, pixel)."""
        ends = torch.cumsum(self.count, 0)
        total, at, first = int(ends[-1]) if len(ends) else 0, 0, 0
        while at < total:
            last = int(torch.searchsorted(ends, torch.tensor(at + 8_000_000, device="cuda")))
            last = max(last, first + 1)
            rows = torch.arange(first, min(last, len(ends)), device="cuda")
            n = self.count[rows]
            t = torch.repeat_interleave(rows, n)
            k = torch.arange(len(t), device="cuda") + at - (ends[t] - self.count[t])
            x, y = self.x0[t] + k % self.nx[t], self.y0[t] + k // self.nx[t]
            px, py = 16 * x + 8 + offset[0], 16 * y + 8 + offset[1]
            e, cover = [], torch.ones_like(x, dtype=torch.bool)
            for a, b in ((0, 1), (1, 2), (2, 0)):
                ax, ay, bx, by = self.X[t, a], self.Y[t, a], self.X[t, b], self.Y[t, b]
                v = (ay - by) * (px - ax) + (bx - ax) * (py - ay)
                cover &= v - ((by > ay) | ((by == ay) & (ax > bx))).long() >= 0
                e.append(v)
            t, pixel = t[cover], (y * self.w + x)[cover]
            l0, l1 = e[1][cover].double() / self.det[t], e[2][cover].double() / self.det[t]
            z = self.Z[t]
            yield t, pixel, l0, l1, l0 * z[:, 0] + l1 * z[:, 1] + (1 - l0 - l1) * z[:, 2]
            at, first = int(ends[min(last, len(ends)) - 1]), last

    def depth(self, offset=(0, 0)):
        d = torch.ones(self.w * self.h, dtype=torch.float64, device="cuda")
        for _, pixel, _, _, z in self.pairs(offset):
            d.scatter_reduce_(0, pixel, z, "amin")
        return d.view(self.h, self.w)

    def winners(self):
        """(pixel, triangle, l0, l1) of every covered pixel's nearest triangle."""
        near, row = self.depth().view(-1), torch.full((self.w * self.h,), -1, dtype=torch.int64, device="cuda")
        for t, pixel, _, _, z in self.pairs((0, 0)):
            won = z == near[pixel]
            row.scatter_reduce_(0, pixel[won], t[won], "amax")
        pixel = torch.nonzero(row >= 0).view(-1)
        t = row[pixel]
        x, y = 16 * (pixel % self.w) + 8, 16 * (pixel // self.w) + 8
        edge = lambda a, b: ((self.Y[t, a] - self.Y[t, b]) * (x - self.X[t, a])
                             + (self.X[t, b] - self.X[t, a]) * (y - self.Y[t, a])).double() / self.det[t]
        return pixel, self.tri[t], edge(1, 2), edge(2, 0)


def _colours(w, light, material, bary, p, n, c):
    """Clamped vertex-colour Blinn-Phong of perspective-correct weights `bary`; p, n, c: (N, 3 vertices, 3)."""
    P, Nn, Cc = ((bary[:, :, None] * a).sum(1) for a in (p, n, c))
    unit = lambda a: a / a.norm(dim=-1, keepdim=True)
    nh, lh = unit(Nn), unit(light)
    inv = np.linalg.inv(np.asarray(w.mv, np.float64).reshape(4, 4))
    eye = torch.from_numpy(inv[:3, 3] / inv[3, 3]).cuda()
    hh = unit(lh + unit(eye - P))
    sa = (nh * hh).sum(1)
    k = int(round(MATERIAL[3]))
    # the exponent's own derivative, sa^s ln(sa), taken at the whole exponent
    log = torch.where(sa > 0, torch.log(sa.clamp(min=1e-300)), torch.zeros_like(sa))
    spec = sa ** k * (1.0 + (material[3] - k) * log) * material[2]
    diffuse = ((nh * lh).sum(1).clamp(min=0.0) + material[0]) * material[1] / math.pi
    return (diffuse[:, None] * Cc + spec[:, None]).clamp(0.0, 1.0)


def _exact_train(case, seed):
    mesh, views, light, target = _train_scene(case, seed)
    planes = torch.stack([torch.from_numpy(a.astype(np.float64)) for a in mesh.planes()], 1).cuda().requires_grad_(True)
    lt = torch.tensor(light, dtype=torch.float32).double().cuda().requires_grad_(True)
    mt = torch.tensor(MATERIAL, dtype=torch.float32).double().cuda().requires_grad_(True)
    idx = torch.from_numpy(mesh.indices.reshape(-1, 3).astype(np.int64)).cuda()
    res, images = case["res"], []
    for w, goal in zip(views, target.double()):
        vis = _Visible(w, mesh)
        if vis.clipped:
            return None
        pixel, tri, l0, l1 = vis.winners()
        x, y = pixel % res, pixel // res
        at = torch.index_select(planes, 0, idx[tri].view(-1)).view(-1, 3, 9)
        p, n, c = at[:, :, 0:3], at[:, :, 3:6], at[:, :, 6:9]
        m = torch.from_numpy(_mvp32(w).astype(np.float64)).cuda()
        clip = [(p * m[i, :3]).sum(2) + m[i, 3] for i in (0, 1, 3)]
        # the image: the snapped triangle's barycentrics made perspective-correct
        with torch.no_grad():
            q = torch.stack([l0, l1, 1 - l0 - l1], 1) / clip[2]
            image = torch.zeros((res * res, 3), dtype=torch.float64, device="cuda")
            image[(res - 1 - y) * res + x] = _colours(w, lt, mt, q / q.sum(1, keepdim=True), p, n, c)
            image = image.view(res, res, 3)
            images.append(image)
            g = 2.0 * (image - goal)[res - 1 - y, x]
        # the gradient: of the unsnapped projection's barycentrics at the pixel's centre
        xn, yn = (x.double() + 0.5) * 2 / res - 1, 1 - (y.double() + 0.5) * 2 / res
        A, B = clip[0] - xn[:, None] * clip[2], clip[1] - yn[:, None] * clip[2]
        q = torch.stack([A[:, i] * B[:, j] - A[:, j] * B[:, i] for i, j in ((1, 2), (2, 0), (0, 1))], 1)
        (_colours(w, lt, mt, q / q.sum(1, keepdim=True), p, n, c) * g).sum().backward()
    return {"image": torch.stack(images), "grads": [planes.grad[:, k] for k in range(9)] + [lt.grad, mt.grad]}


def exact(case, seed):
    path = case["path"]
    if path == "viewer":
        return None  # bytes
    if path == "train":
        return _exact_train(case, seed)
    depths = []
    for w in _batch_scenes(case, seed) if path == "batch" else [_scene(case, seed)]:
        vis = _Visible(w, w.mesh)
        if vis.clipped:
            return None
        depths.append(torch.stack([vis.depth(o) for o in _SAMPLES[case.get("msaa", 0)]]).flip(1))
    if path == "batch":
        depth = torch.cat([d.reshape(-1) for d in depths])
    else:
        depth = depths[0] if len(depths[0]) > 1 else depths[0][0]
    return {"color": None, "depth": depth, "ids": None}
