"""The workloads that a program built on this library has it do, as cases to time and compare.

Every case goes through the library's public entry points, with the buffers where such a program
keeps them: device-resident rays, films and samples for the wavefront paths, host arrays where a
program calls the numpy interface.  Six paths are covered:

  trace    Scene.trace_device / Scene.trace: batches of probes against a committed scene.  "sphere" is
           the UV sphere over its ground quad, "field" the flattened icosphere field, "moving" the
           spheres with two motion keys, "instances" the room of instances, a procedural and a
           transformed mesh.  Rays leave a pinhole, a uniform box or the scene's own surfaces
           (bounce); shadow rays stop at any hit.
  render   Renderer.render_pass_device: one pass over every pixel, in the reference's shading
           (depth 0) or as paths (depth 1 and up).
  path     PathTracer.render_pass_device: one plain path-tracing pass in the occluded-light room.
  infer    vgpu_guide_infer on device queries: the guiding network's lobes (or raw outputs).
  train    vgpu_guide_train_step on a device batch, a few Adam steps, then the
           parameters and the last gradient read back.
  build    vgpu_qbvh_build_gpu: the BVH over a mesh's boxes, host arrays in and out.

Sizes are those of the repository's tests and benchmark and what lies between them.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

import vermeer_amd as va
from vermeer_amd import _lib, guide, pathtrace, render, scenes

NPARAMS = _lib.VGPU_GUIDE_NPARAMS
ROOM_LO, ROOM_HI = (-0.9, 0.1, -0.9), (0.9, 1.9, 0.9)   # inside the instance scene's room


def listed():
    return [
        # a viewer's preview tile or a picking batch: few rays, the latency of one launch
        {"name": "trace-tile", "kind": "trace", "scene": "sphere", "size": 256, "rays": "pinhole", "n": 4096,
         "shadow": False, "geoms": False, "host": False},
        # a host renderer handing over its probes as numpy arrays, an odd number of them
        {"name": "trace-host", "kind": "trace", "scene": "sphere", "size": 256, "rays": "uniform", "n": 50021,
         "shadow": False, "geoms": True, "host": True},
        # ambient-occlusion style shadow rays in a mid-size mesh
        {"name": "trace-shadow", "kind": "trace", "scene": "field", "size": 500, "rays": "bounce", "n": 300007,
         "shadow": True, "geoms": False, "host": False},
        # one bounce of a large incoherent batch (the flattened 5.2M-triangle field)
        {"name": "trace-bounce", "kind": "trace", "scene": "field", "size": 4096, "rays": "bounce", "n": 2097152,
         "shadow": False, "geoms": True, "host": False},
        # motion-blurred camera rays, each at its own time
        {"name": "trace-motion", "kind": "trace", "scene": "moving", "size": 2000, "rays": "pinhole", "n": 1048576,
         "shadow": False, "geoms": False, "host": False},
        # rays through instances, a procedural and a moving transform
        {"name": "trace-instances", "kind": "trace", "scene": "instances", "size": 60, "rays": "uniform", "n": 262144,
         "shadow": False, "geoms": True, "host": False},
        # the reference's shading of an ordinary frame
        {"name": "render-frame", "kind": "render", "scene": "box", "width": 512, "height": 512, "depth": 0},
        # paths of five segments at a preview's size
        {"name": "render-paths", "kind": "render", "scene": "box", "width": 320, "height": 199, "depth": 5},
        # a full-size plain pass of the path tracer in the million-triangle room
        {"name": "path-room", "kind": "path", "boxes": 66667, "res": 20, "width": 1024, "height": 1024, "depth": 8},
        # one bounce's guide queries, a megapixel frame
        {"name": "infer-frame", "kind": "infer", "n": 1048576, "raw": False},
        # online training between two passes: eight Adam steps on full batches
        {"name": "train-steps", "kind": "train", "batch": 65536, "steps": 8},
        # a mesh's BVH built on the device for a scene commit
        {"name": "build-mesh", "kind": "build", "n": 300001, "leaf": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(["trace", "trace", "trace", "trace", "render", "render", "path", "infer", "train", "build"])
    if kind == "trace":
        scene = rng.choice(["sphere", "field", "moving", "instances"])
        lo, hi = {"sphere": (16, 256), "field": (32, 4096), "moving": (50, 2000), "instances": (6, 60)}[scene]
        rays = rng.choice({"sphere": ["pinhole", "uniform"], "field": ["bounce"], "moving": ["pinhole", "uniform"],
                           "instances": ["uniform"]}[scene])
        most = {"sphere": 2000000, "field": 2000000, "moving": 1000000, "instances": 260000}[scene]
        host = rng.random() < 0.2
        return {"kind": kind, "scene": scene, "size": _log_int(rng, lo, hi), "rays": rays,
                "n": _log_int(rng, 1024, 200000 if host else most), "shadow": rng.random() < 0.4,
                "geoms": True if host else rng.random() < 0.5, "host": host}
    if kind == "render":
        return {"kind": kind, "scene": rng.choice(["box", "feature", "moving"]), "width": _log_int(rng, 32, 512),
                "height": _log_int(rng, 32, 512), "depth": rng.choice([0, 0, 1, 2, 3, 5])}
    if kind == "path":
        return {"kind": kind, "boxes": _log_int(rng, 500, 66000), "res": rng.randint(4, 20),
                "width": _log_int(rng, 48, 1000), "height": _log_int(rng, 48, 1000), "depth": rng.randint(2, 8)}
    if kind == "infer":
        return {"kind": kind, "n": _log_int(rng, 256, 1000000), "raw": rng.random() < 0.3}
    if kind == "train":
        return {"kind": kind, "batch": 1024 * rng.randint(8, 64), "steps": rng.randint(1, 8)}
    return {"kind": kind, "n": _log_int(rng, 5000, 300000), "leaf": rng.choice([1, 4, 8, 16])}


# ------------------------------------------------------------------ inputs

def _small(seed):
    """Any integer as a seed that every generator here takes, with room for the offsets added to it."""
    return int(seed) % (1 << 16)


def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1).copy()).cuda()


def _add_mesh(sc, mesh):
    """A scene description's mesh without its shading."""
    sc.add_geom(va.PolyMesh(np.asarray(mesh["verts"], np.float32).reshape(-1, 3), mesh["idx"]))


def _scene(case, seed):
    """(committed scene, verts, idx): geometry of the case's kind and size; the field and the moving
    spheres lie elsewhere for another seed."""
    sc = va.Scene(0)
    kind, size = case["scene"], case["size"]
    verts = idx = None
    if kind == "sphere":
        sc.add_geom(va.PolyMesh(*scenes.uv_sphere(1.0, size, max(3, size // 2))))
        sc.add_geom(va.PolyMesh(*scenes.ground_quad()))
    elif kind == "field":
        # the density of 4096 spheres in a cube of edge 100
        verts, idx = scenes.icosphere_field(size, extent=100.0 * (size / 4096.0) ** (1.0 / 3.0), seed=seed + 7)[:2]
        sc.add_geom(va.PolyMesh(verts, idx))
    elif kind == "moving":
        verts, idx = scenes.moving_spheres(size, extent=20.0 * (size / 2000.0) ** (1.0 / 3.0), seed=seed + 21)
        sc.add_geom(va.PolyMesh(verts, idx))
    else:
        desc = scenes.instance_scene(seed=seed + 11, count=size)
        for mesh in desc["meshes"]:
            _add_mesh(sc, mesh)
        sc.add_transforms(desc)
    sc.pre_render()
    return sc, verts, idx


def _rays(case, seed, verts, idx):
    """The case's rays as a device byte tensor (RAY_DTYPE records)."""
    n, kind = case["n"], case["scene"]
    g = torch.Generator(device="cuda").manual_seed(seed + 1000)

    def uniform(k):
        return torch.rand(n, k, generator=g, device="cuda", dtype=torch.float64)

    if case["rays"] == "bounce":
        d, _ = scenes.bounce_rays_device(verts, idx, n, seed=seed + 17)
        rec = d.view(torch.float32).reshape(n, 8)
        if case["shadow"]:
            rec[:, 3] = (uniform(1)[:, 0] * 20.0).float()   # occlusion within a distance
        return rec.reshape(-1).view(torch.uint8)
    rec = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    rec[:, 3] = math.inf
    if case["rays"] == "pinhole":
        far, fov = (45.0 * (case["size"] / 2000.0) ** (1.0 / 3.0), 60.0) if kind == "moving" else (4.0, 45.0)
        eye = np.array([0.05 * math.sin(seed), 0.25 if kind == "sphere" else 0.0, 1.0]) * far
        w = max(1, math.isqrt(n))
        i = torch.arange(n, device="cuda")
        sx = ((i % w).double() + 0.5) / w * 2.0 - 1.0
        sy = -(((i // w).double() + 0.5) / (n / w) * 2.0 - 1.0)
        u, v, back = (torch.from_numpy(a).cuda() for a in scenes.lookat_basis(eye, (0.0, 0.0, 0.0), (0.0, 1.0, 0.0)))
        tn = math.tan(math.radians(fov) / 2.0)
        d = (sx[:, None] * tn) * u + (sy[:, None] * tn) * v - back
        rec[:, 0:3] = torch.from_numpy(eye).float().cuda()
    else:
        lo, hi = {"sphere": ((-5.0, -1.0, -5.0), (5.0, 1.0, 5.0)), "instances": (ROOM_LO, ROOM_HI)}.get(
            kind, ((-20.0,) * 3, (20.0,) * 3))
        lo, hi = (torch.tensor(a, dtype=torch.float64, device="cuda") for a in (lo, hi))
        rec[:, 0:3] = (lo + uniform(3) * (hi - lo)).float()
        d = torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float64)
    rec[:, 4:7] = (d / d.norm(dim=1, keepdim=True)).float()
    if kind in ("moving", "instances"):
        rec[:, 7] = uniform(1)[:, 0].float().clamp_(max=1.0 - 2.0 ** -24)
    return rec.reshape(-1).view(torch.uint8)


def _render_scene(kind, seed):
    if kind == "feature":
        return scenes.feature_scene(seed=seed + 5)
    if kind == "moving":
        return scenes.moving_scene(seed=seed + 7)
    return scenes.box_spheres_scene(seed=seed + 3)


@functools.lru_cache(maxsize=2)
def _room(res, boxes):
    return scenes.guided_room_scene(res=res, nboxes=boxes)


_LAYERS = [(64, 144), (64, 64), (64, 64), (64, 64), (40, 64)]
_BOUNDS = np.array([-4.0, 0.0, -4.0, 4.8, 4.0, 4.0], np.float32)


def _params(seed):
    """He-uniform weights, small biases; the last layer scaled down so that the lobes start broad."""
    g = np.random.default_rng(seed + 31)
    out = []
    for i, (no, ni) in enumerate(_LAYERS):
        b = math.sqrt(6.0 / ni) * (0.3 if i == 4 else 1.0)
        out += [g.uniform(-b, b, no * ni), g.uniform(-0.05, 0.05, no)]
    return np.concatenate(out).astype(np.float32)


def _points(n, seed):
    """Hit positions on the room's walls and clutter and their unit normals (float32, device)."""
    g = torch.Generator(device="cuda").manual_seed(seed + 41)
    lo, hi = (torch.tensor(b, device="cuda") for b in (_BOUNDS[:3], _BOUNDS[3:]))
    p = lo + torch.rand(n, 3, generator=g, device="cuda") * (hi - lo)
    nrm = torch.randn(n, 3, generator=g, device="cuda")
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    return p, nrm, g


def _samples(n, seed):
    """Training samples: position, weight c (heavy-tailed, as path radiances are), normal, direction
    gathered about a few preferred ones."""
    p, nrm, g = _points(n, seed)
    c = torch.exp(torch.randn(n, generator=g, device="cuda"))
    mode = torch.randn(4, 3, generator=g, device="cuda")
    pick = torch.randint(0, 4, (n,), generator=g, device="cuda")
    d = mode[pick] + 0.5 * torch.randn(n, 3, generator=g, device="cuda")
    d = d / d.norm(dim=1, keepdim=True)
    z = torch.zeros(n, 1, device="cuda")
    return torch.cat([p, c[:, None], nrm, z, d, z], dim=1).contiguous()


def _elements(n, seed):
    """Boxes, centroids and indices of the first n triangles of an icosphere field."""
    verts, idx = scenes.icosphere_field(-(-n // 1280), seed=seed + 7)[:2]
    tri = verts[idx[:n].astype(np.int64)]
    boxes = np.concatenate([tri.min(1), tri.max(1)], axis=1)
    cent = (tri[:, 0] + tri[:, 1] + tri[:, 2]) / np.float32(3.0)
    return np.ascontiguousarray(boxes, np.float32), np.ascontiguousarray(cent, np.float32), np.arange(n, dtype=np.int32)


def prepare(case, seed):
    kind, seed = case["kind"], _small(seed)
    s = {"case": dict(case)}
    if kind == "trace":
        n = case["n"]
        s["scene"], verts, idx = _scene(case, seed)
        rays = _rays(case, seed, verts, idx)
        if case["host"]:
            s["rays"] = rays.cpu().numpy().view(va.RAY_DTYPE)
        else:
            s["rays"] = rays
            s["hits"] = torch.empty(n, 4, dtype=torch.int32, device="cuda")
            s["geoms"] = torch.empty(n, dtype=torch.int32, device="cuda") if case["geoms"] else None
    elif kind == "render":
        w, h = case["width"], case["height"]
        desc = _render_scene(case["scene"], seed)
        c = desc["camera"]
        cam = render.lookat_camera(c["from"], c["to"], c["up"], c["fov"], c["focal"], w, h)
        s["render"] = render.Renderer(desc, w, h, cam)
        if case["depth"]:
            s["render"].set_path_depth(case["depth"])
        if case["scene"] == "feature":
            s["render"].set_filter("gaussian")
        s["scrambles"] = _device(scenes.pixel_scrambles(w, h, seed=seed + 99))
        s["film"] = torch.zeros(h, w, 3, device="cuda")
        s["sample"] = torch.zeros(h, w, 3, device="cuda")
        s["pass"] = 0
    elif kind == "path":
        w, h = case["width"], case["height"]
        s["pt"] = pathtrace.PathTracer(_room(case["res"], case["boxes"]), w, h, max_depth=case["depth"], seed=seed + 1)
        s["accum"] = torch.zeros(h, w, 3, dtype=torch.float64, device="cuda")
        s["pass"] = 0
    elif kind in ("infer", "train"):
        s["guide"] = guide.Guide(_BOUNDS, seed=1, max_batch=max(case.get("batch", 0), 1024))
        s["guide"].params = _params(seed)
        if kind == "infer":
            p, nrm, _ = _points(case["n"], seed)
            z = torch.zeros(case["n"], 1, device="cuda")
            s["queries"] = torch.cat([p, z, nrm, z], dim=1).contiguous()
            s["out"] = torch.empty(case["n"], 40, device="cuda")
        else:
            s["samples"] = [_samples(case["batch"], seed + 100 * k) for k in range(min(4, case["steps"]))]
    else:
        s["given"] = _elements(case["n"], seed)
        s["arrays"] = tuple(a.copy() for a in s["given"])
        s["nodes"] = np.zeros(case["n"], _lib.NODE_DTYPE)
        s["bounds"] = np.zeros(6, np.float32)
    torch.cuda.synchronize()   # the inputs were made on torch's stream
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    st = torch.cuda.current_stream().cuda_stream
    if kind == "trace":
        if case["host"]:
            hits, geoms, _ = s["scene"].trace(s["rays"], shadow=case["shadow"])
            return {"hits": hits.view(np.int32).reshape(-1, 4), "geoms": geoms}
        g = s["geoms"]
        s["scene"].trace_device(s["rays"].data_ptr(), case["n"], s["hits"].data_ptr(), shadow=case["shadow"],
                                d_geoms=0 if g is None else g.data_ptr(), stream=st)
        return {"hits": s["hits"]} if g is None else {"hits": s["hits"], "geoms": g}
    if kind == "render":
        s["pass"] += 1
        s["render"].render_pass_device(s["scrambles"].data_ptr(), s["pass"], s["film"].data_ptr(),
                                       s["sample"].data_ptr(), stream=st)
        return {"film": s["film"], "sample": s["sample"]}
    if kind == "path":
        s["pt"].render_pass_device(s["accum"].data_ptr(), s["pass"], stream=st)
        s["pass"] += 1
        return s["accum"]
    lib = _lib.load()
    if kind == "infer":
        flags = _lib.VGPU_TRACE_DEVICE_PTRS | (_lib.VGPU_GUIDE_RAW if case["raw"] else 0)
        _lib.check(lib.vgpu_guide_infer(s["guide"]._h, flags, C.c_void_p(s["queries"].data_ptr()), case["n"],
                                        C.c_void_p(s["out"].data_ptr()), C.c_void_p(st)))
        return s["out"]
    if kind == "train":
        for k in range(case["steps"]):
            b = s["samples"][k % len(s["samples"])]
            _lib.check(lib.vgpu_guide_train_step(s["guide"]._h, _lib.VGPU_TRACE_DEVICE_PTRS, C.c_void_p(b.data_ptr()),
                                                 case["batch"], 1e-3, C.c_void_p(st), None))
        return {"params": s["guide"].params, "grad": s["guide"].grad()}
    for a, b in zip(s["arrays"], s["given"]):
        np.copyto(a, b)   # the build permutes its arrays in place
    boxes, cent, idx = s["arrays"]
    count = C.c_int32(0)
    _lib.check(lib.vgpu_qbvh_build_gpu(_lib.ptr(boxes), _lib.ptr(cent), _lib.ptr(idx), case["n"], case["leaf"],
                                       _lib.ptr(s["nodes"]), case["n"], C.byref(count), _lib.ptr(s["bounds"]), None))
    return {"nodes": s["nodes"].view(np.int32).reshape(-1, 32), "count": count.value, "bounds": s["bounds"], "boxes": boxes,
            "centroids": cent, "idx": idx}


# ------------------------------------------------------------------ what a pass cannot do without

def _scene_bytes(case):
    """Triangles (48 bytes a key) and nodes (about one 128-byte node per 22 triangles at leaf size 16)."""
    size = case["size"]
    tris = {"sphere": size * size, "field": 1280 * size, "moving": 500 * size, "instances": 900}[case["scene"]]
    return tris * 54


def work(case):
    kind = case["kind"]
    if kind == "trace":
        n = case["n"]
        # about 12 box tests of four children and 8 triangle tests a ray
        return {"bytes": n * (32 + 16 + (4 if case["geoms"] else 0)) + min(_scene_bytes(case), n * 1000),
                "flops": n * (12 * 4 * 12 + 8 * 40)}
    if kind == "render":
        # scrambles, film in and out, sample; per segment a closest-hit and two shadow rays and the shading
        px = case["width"] * case["height"]
        return {"bytes": px * (48 + 24 + 12), "flops": px * max(1, case["depth"]) * 5000}
    if kind == "path":
        px = case["width"] * case["height"]
        return {"bytes": px * 48 + 54 * (12 * case["boxes"] + 512 * case["res"] ** 2), "flops": px * case["depth"] * 4000}
    macs = sum(no * ni for no, ni in _LAYERS)
    if kind == "infer":
        return {"bytes": case["n"] * (32 + 160) + 4 * NPARAMS, "flops": case["n"] * 2 * macs}
    if kind == "train":
        # forward, input gradients (not of the first layer) and weight gradients; weights and moments in and out
        return {"bytes": case["steps"] * (case["batch"] * 48 + NPARAMS * 28),
                "flops": case["steps"] * case["batch"] * 2 * (3 * macs - 144 * 64)}
    return {"bytes": case["n"] * (40 * 2 + 128 / 8), "flops": case["n"] * 60}


def tolerance(case):
    """Traversal, shading, path sums and the BVH are specified to the bit, the network is not: its
    operands are bf16, so a sum in another order moves some activations by a bf16 step.  Against the same
    roundings with sums in 64 bits the outputs differ by 1.2e-4 (one value by 0.06).  A training step with
    its batch in another order differs by 2e-7, and by as much as a bf16 step's effect where an activation
    moves; Adam's normalised steps carry that on (up to 1.2e-2 of the gradient, 0.25 of one value, after
    eight to sixteen steps)."""
    if case["kind"] == "infer":
        return {"rel": 5e-4, "max": 0.25}
    if case["kind"] == "train":
        return {"rel": 1e-3, "max": 0.1} if case["steps"] == 1 else {"rel": 0.03, "max": 0.95}
    return "exact"


# ------------------------------------------------------------------ 64-bit reference of the network

def _split(P):
    out, k = [], 0
    for no, ni in _LAYERS:
        out.append((P[k:k + no * ni].reshape(no, ni), P[k + no * ni:k + no * ni + no]))
        k += no * ni + no
    return out


def _forward(P, p, nrm):
    """Raw outputs (n, 8, 5) in float64."""
    lo, hi = (torch.tensor(b, device="cuda", dtype=torch.float64) for b in (_BOUNDS[:3], _BOUNDS[3:]))
    x = torch.cat([(p.double() - 0.5 * (lo + hi)) / (0.5 * (hi - lo)), nrm.double()], dim=1)
    a = math.pi * x[:, :, None] * 2.0 ** torch.arange(12, device="cuda", dtype=torch.float64)
    y = torch.stack([torch.sin(a), torch.cos(a)], dim=-1).reshape(len(x), 144)
    layers = _split(P)
    for i, (W, b) in enumerate(layers):
        y = y @ W.t() + b
        if i < 4:
            y = torch.relu(y)
    return y.reshape(-1, 8, 5)


def _lobes(raw):
    u = raw[..., 0:3]
    mu = u / u.norm(dim=-1, keepdim=True)
    return mu, torch.exp(raw[..., 3].clamp(-5.0, 7.0)), torch.softmax(raw[..., 4], dim=-1)


def exact(case, seed):
    """The network's outputs and the trained parameters in 64 bits.  The other paths are compared bit
    for bit (their results are float32 operations in a stated order) and have no 64-bit value."""
    seed = _small(seed)
    if case["kind"] == "infer":
        P = torch.from_numpy(_params(seed)).cuda().double()
        p, nrm, _ = _points(case["n"], seed)
        out = []
        for a in range(0, case["n"], 1 << 17):
            raw = _forward(P, p[a:a + (1 << 17)], nrm[a:a + (1 << 17)])
            if not case["raw"]:
                mu, kappa, w = _lobes(raw)
                raw = torch.cat([mu, kappa[..., None], w[..., None]], dim=-1)
            out.append(raw.reshape(-1, 40))
        return torch.cat(out)
    if case["kind"] != "train":
        return None
    P = torch.from_numpy(_params(seed)).cuda().double()
    m, v = torch.zeros_like(P), torch.zeros_like(P)
    batches = [_samples(case["batch"], seed + 100 * k) for k in range(min(4, case["steps"]))]
    for k in range(case["steps"]):
        b = batches[k % len(batches)]
        Q = P.clone().requires_grad_(True)
        c = b[:, 3].double()
        mu, kappa, w = _lobes(_forward(Q, b[:, 0:3], b[:, 4:7]))
        cos = (mu * b[:, None, 8:11].double()).sum(-1)
        logp = (torch.log(w) + torch.log(kappa) - math.log(2.0 * math.pi) - torch.log(-torch.expm1(-2.0 * kappa))
                + kappa * (cos - 1.0))
        (-(c * torch.logsumexp(logp, dim=-1)).sum() / c.sum()).backward()
        g = Q.grad
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        t = k + 1
        P = P - 1e-3 * (m / (1.0 - 0.9 ** t)) / (torch.sqrt(v / (1.0 - 0.999 ** t)) + 1e-8)
    return {"params": P, "grad": g}
