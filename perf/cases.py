"""The work that users of this framework have it do, as cases that can be timed.

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program has in hand before the call, run() is one pass through
the public entry points and work() the bytes and operations that the pass
cannot do without.  exact() gives ray-query results in 64 bits from plain
torch.
"""
import ctypes
import math

import numpy as np
import torch

import nanogi_amd as ngi

DEVICE = "cuda:0"
FAR = 1000.0   # ray queries end here: beyond every scene's extent

SCENES = {"cornell": ngi.GEN_CORNELL, "nave": ngi.GEN_NAVE, "field": ngi.GEN_SPHERE_FIELD, "room": ngi.GEN_BATCH_ROOM}
ENGINES = {"persistent": ngi.ENGINE_PERSISTENT, "wavefront": ngi.ENGINE_WAVEFRONT}
PRECISIONS = {"fp32": ngi.PRECISION_FP32_FP64ACC, "fp32all": ngi.PRECISION_FP32_ALL, "fp64": ngi.PRECISION_FP64_ALL}

# Box from which ray origins are drawn, per scene (inside the geometry).
ORIGINS = {"cornell": ((0.05, 0.05, 0.05), (0.95, 0.95, 0.95)), "room": ((0.05, 0.05, 0.05), (0.95, 0.95, 0.95)),
           "nave": ((-19.0, 0.8, -7.5), (19.0, 11.5, 7.5)), "field": ((-3.0, 0.2, -3.0), (3.0, 2.5, 3.0))}


def listed():
    return [
        # A few rays from the host: picking under the cursor, a collision or visibility probe.
        {"name": "probe_rays", "kind": "trace", "scene": "nave", "detail": 0, "rays": 64, "any": False, "where": "host"},
        # Closest hits of incoherent rays that a program already has on the GPU, 1.8M triangles.
        {"name": "trace_field", "kind": "trace", "scene": "field", "detail": 8, "rays": 1500007, "any": False, "where": "device"},
        # Occlusion of point pairs from host arrays (Scene::Visible): light baking, line of sight.
        {"name": "occlusion_nave", "kind": "trace", "scene": "nave", "detail": 0, "rays": 300007, "any": True, "where": "host"},
        # A viewer's frame: one sample per pixel of a small image into its own device buffer.
        {"name": "preview", "kind": "noalloc", "scene": "room", "detail": 2000, "renderer": "ptdirect", "precision": "fp32",
         "width": 320, "height": 181, "spp": 1, "max_vertices": 9, "rr_depth": 3},
        # The command line's defaults: pt, 1280x720, 10M samples uniform over the image, unlimited vertices, roulette from the first bounce.
        {"name": "pt_defaults", "kind": "render", "scene": "cornell", "detail": 0, "renderer": "pt", "precision": "fp32",
         "engine": "persistent", "sampling": "uniform", "width": 1280, "height": 720, "samples": 10000000, "max_vertices": -1, "rr_depth": 1},
        # An interior with many bounces, one call.
        {"name": "ptdirect_nave", "kind": "render", "scene": "nave", "detail": 0, "renderer": "ptdirect", "precision": "fp32",
         "engine": "persistent", "sampling": "pixel", "width": 1024, "height": 1024, "spp": 64, "max_vertices": 17, "rr_depth": 4},
        # The benchmark's scene, rendered progressively in batches of 16 spp with the variance estimate.
        {"name": "ptdirect_field", "kind": "session", "scene": "field", "detail": 8, "renderer": "ptdirect", "precision": "fp32",
         "engine": "persistent", "width": 1024, "height": 1024, "spp": 16, "batches": 4, "max_vertices": 33, "rr_depth": 4},
        # The same scene at the reference's precision (FP64 shading), a smaller image of another shape.
        {"name": "ptdirect_field_fp64", "kind": "render", "scene": "field", "detail": 8, "renderer": "ptdirect", "precision": "fp64",
         "engine": "persistent", "sampling": "pixel", "width": 641, "height": 363, "spp": 32, "max_vertices": 33, "rr_depth": 4},
        # Light tracing of the interior.
        {"name": "ltdirect_nave", "kind": "render", "scene": "nave", "detail": 0, "renderer": "ltdirect", "precision": "fp32",
         "engine": "persistent", "sampling": "uniform", "width": 512, "height": 512, "samples": 8000000, "max_vertices": 17, "rr_depth": 4},
        # Bidirectional path tracing of the small box.
        {"name": "bdpt_cornell", "kind": "render", "scene": "cornell", "detail": 0, "renderer": "bdpt", "precision": "fp32",
         "engine": "persistent", "sampling": "pixel", "width": 256, "height": 256, "spp": 32, "max_vertices": 9, "rr_depth": -1},
        # Many small scenes per frame: a data set of rooms.
        {"name": "batch_rooms", "kind": "batch", "scenes": 24, "tris": 5000, "side": 256, "spp": 64, "renderer": "ptdirect",
         "max_vertices": 17, "rr_depth": 4},
        # One step of inverse rendering: the image and, through autograd, the gradients of a loss on it.
        {"name": "grad_nave", "kind": "grad", "scene": "nave", "detail": 0, "renderer": "ptdirect", "width": 512, "height": 512,
         "spp": 32, "max_vertices": 17, "rr_depth": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "render", "render", "render", "session", "noalloc", "batch", "grad"])
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 32), "tris": _log(rng, 40, 5000), "side": _log(rng, 32, 256), "spp": _log(rng, 2, 64),
                "renderer": rng.choice(["pt", "ptdirect"]), "max_vertices": rng.randint(4, 17), "rr_depth": rng.choice([-1, 1, 4])}
    scene = rng.choice(["cornell", "room", "nave", "field"])
    detail = {"cornell": 0, "nave": 0, "field": rng.randint(4, 8), "room": _log(rng, 20, 12000)}[scene]
    c = {"kind": kind, "scene": scene, "detail": detail}
    if kind == "trace":
        c.update(rays=_log(rng, 1, 2000000), any=rng.random() < 0.5, where=rng.choice(["host", "device"]))
        return c
    width, height = _log(rng, 24, 1100), _log(rng, 24, 1100)
    # Paths: up to about the listed cases' largest counts, fewer where a path costs more.
    most = {"render": 3e7, "session": 3e7, "noalloc": 8e6, "grad": 4e6}[kind]
    paths = min(most, math.exp(rng.uniform(math.log(2e3), math.log(most))))
    renderer = rng.choice(["pt", "ptdirect"] if kind == "grad" else
                          ["pt", "ptdirect", "ptdirect", "ltdirect"] if kind == "noalloc" else ["pt", "ptdirect", "ptdirect", "ltdirect", "bdpt"])
    if renderer == "bdpt":
        paths = max(1000.0, paths / 16)
    spp = max(1, int(paths / (width * height)))
    c.update(renderer=renderer, width=width, height=height, spp=spp, max_vertices=rng.randint(4, 17), rr_depth=rng.choice([1, 4, 4, -1]))
    if kind == "grad":
        return c
    c["precision"] = "fp32" if renderer == "bdpt" else rng.choice(["fp32", "fp32", "fp32", "fp64", "fp32all"])
    if kind == "noalloc":
        return c
    c["engine"] = "wavefront" if renderer in ("pt", "ptdirect") and c["precision"] != "fp64" and rng.random() < 0.2 else "persistent"
    if kind == "session":
        c["batches"] = rng.randint(2, 4)
        c["spp"] = max(1, spp // c["batches"])
        return c
    c["sampling"] = rng.choice(["pixel", "pixel", "uniform"])
    if c["sampling"] == "uniform":
        c["samples"] = int(paths)
    return c


def _scene(case, seed):
    s = ngi.Scene.generate(SCENES[case["scene"]], 1 + seed % 100003, case.get("width", 1) / case.get("height", 1), case["detail"])
    s.build()
    return s


def _params(case, seed):
    p = ngi.default_params(renderer=case["renderer"], width=case["width"], height=case["height"], sampling=ngi.SAMPLING_PER_PIXEL,
                           spp=case["spp"] if "spp" in case else 1, max_num_vertices=case["max_vertices"], rr_depth=case["rr_depth"],
                           seed=seed & 0xFFFFFFFF, precision=PRECISIONS[case.get("precision", "fp32")],
                           engine=ENGINES[case.get("engine", "persistent")])
    if case.get("sampling") == "uniform":
        p.sampling = ngi.SAMPLING_REFERENCE_UNIFORM
        p.num_samples = case["samples"]
    return p


def _rays(case, seed):
    """Rays between random points of the scene (any hit), or from them in random directions."""
    rng = np.random.default_rng(seed)
    lo, hi = (np.array(v) for v in ORIGINS[case["scene"]])
    o = lo + (hi - lo) * rng.random((case["rays"], 3))
    if case["any"]:
        d = lo + (hi - lo) * rng.random((case["rays"], 3)) - o
        far = np.linalg.norm(d, axis=1)
        d /= far[:, None]
        return ngi.make_rays(o, d, tmax=far.astype(np.float32))
    d = rng.normal(size=(case["rays"], 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    return ngi.make_rays(o, d, tmax=FAR)


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "batch":
        rng = np.random.default_rng(case["scenes"])   # the sizes belong to the case, the rooms to the seed
        scenes, params = [], []
        for i in range(case["scenes"]):
            s = ngi.Scene.generate(ngi.GEN_BATCH_ROOM, 1 + (seed + 7919 * i) % 1000003, 1.0, max(12, int(case["tris"] ** rng.uniform(0.5, 1.0))))
            s.build()
            scenes.append(s)
            side = max(16, int(case["side"] * rng.uniform(0.3, 1.0)))
            p = _params(dict(case, width=side, height=side, spp=max(1, int(case["spp"] * rng.uniform(0.3, 1.0)))), seed)
            p.stream_id = i
            params.append(p)
        st["batch"] = ngi.Batch(scenes, params)
        return st
    scene = st["scene"] = _scene(case, seed)
    if kind == "trace":
        rays = _rays(case, seed)
        st["any"] = case["any"]
        if case["where"] == "host":
            st["rays"] = rays
        else:
            st["kind"] = "trace_device"
            st["rays"] = torch.from_numpy(rays.view(np.float32).reshape(-1, 8)).to(DEVICE)
            st["hits"] = torch.zeros((case["rays"], 4), dtype=torch.float32, device=DEVICE)
        scene.trace(rays[:1])   # the scene is resident
        return st
    st["params"] = _params(case, seed)
    if kind == "noalloc":
        scene.trace(ngi.make_rays([(0.5, 0.5, 0.5)], [(0.0, 1.0, 0.0)]))   # the scene is resident
        single = case["precision"] == "fp32all"
        st["film"] = torch.zeros((case["height"], case["width"], 3), dtype=torch.float32 if single else torch.float64, device=DEVICE)
        st["stats"] = ngi.Stats()
    elif kind == "session":
        st["session"] = ngi.Session(scene, st["params"])
        st["spp"], st["batches"] = case["spp"], case["batches"]
    elif kind == "grad":
        from nanogi_amd.autograd import render_fn, scene_parameters
        refl, Le, _, _ = scene_parameters(scene)
        st["refl"] = refl.clone().requires_grad_(True)
        st["Le"] = Le.clone().requires_grad_(True)
        st["fn"] = render_fn(scene, st["params"])
        rng = np.random.default_rng(seed)
        st["target"] = torch.from_numpy(rng.random((case["height"], case["width"], 3)))
    return st


def _ok(status):
    if status != ngi.OK:
        raise RuntimeError(ngi.lib().ngi_last_error().decode("utf-8", "replace"))


def run(st):
    kind = st["kind"]
    if kind == "trace":
        hits = st["scene"].trace(st["rays"], any_hit=st["any"])
        if st["any"]:   # an occlusion query says only whether something is hit
            return hits["tri"] != ngi.MISS
        return {"t": hits["t"], "u": hits["u"], "v": hits["v"], "tri": hits["tri"].astype(np.int64)}
    if kind == "trace_device":
        rays, hits = st["rays"], st["hits"]
        _ok(ngi.lib().ngi_trace_device(st["scene"].handle, ctypes.c_void_p(rays.data_ptr()), rays.shape[0], ctypes.c_void_p(hits.data_ptr()),
                                       1 if st["any"] else 0))
        tri = hits[:, 3].view(torch.int32)
        if st["any"]:
            return tri != -1
        return {"t": hits[:, 0], "u": hits[:, 1], "v": hits[:, 2], "tri": tri}
    if kind == "noalloc":
        film = st["film"]
        _ok(ngi.lib().ngi_render_device_noalloc(st["scene"].handle, ctypes.byref(st["params"]), ctypes.c_void_p(film.data_ptr()),
                                                ctypes.byref(st["stats"])))
        return film
    if kind == "render":
        film, stats = ngi.render(st["scene"], st["params"])
        return {"film": film, "samples": stats["samples"]}
    if kind == "session":
        s = st["session"]
        s.reset()
        for _ in range(st["batches"]):
            s.render_batch(st["spp"])
        film, var = s.film(variance=True)
        return {"film": film, "variance": var}
    if kind == "batch":
        b = st["batch"]
        b.render(0)
        b.sync()
        return [b.film(i) for i in range(len(b.scenes))]
    # grad
    st["refl"].grad = st["Le"].grad = None
    img = st["fn"](st["refl"], st["Le"])
    loss = (img - st["target"]).square().mean()
    loss.backward()
    return {"image": img.detach(), "reflectance": st["refl"].grad, "Le": st["Le"].grad}


# A closest-hit query visits about 10 wide nodes (8 boxes of about 14
# operations) and tests about 3 triangles (about 45 operations); a vertex
# takes about 400 operations of shading and random numbers.
RAY_FLOPS = 10 * 8 * 14 + 3 * 45
VERTEX_FLOPS = 400
TRI_BYTES = 48 + 48 + 20   # vertices, normals and the triangle's share of the tree


def _triangles(case):
    if case["scene"] == "field":
        return 20 * 4 ** case["detail"] + (522242 if case["detail"] >= 8 else 2 * 63 * 63)
    return {"cornell": 36, "nave": 76842, "room": max(12, case["detail"])}[case["scene"]]


def _segments(case):
    """Mean number of path segments under the vertex cap and roulette 0.5."""
    most = case["max_vertices"] - 1 if case["max_vertices"] > 0 else 64
    open_ = 0.45 if case.get("scene") == "field" else 0.95   # share of rays that hit something
    n, alive = 0.0, 1.0
    for k in range(1, most + 1):
        n += alive
        alive *= open_ * (0.5 if 0 <= case["rr_depth"] <= k else 1.0)
    return n


def work(case):
    kind = case["kind"]
    if kind == "trace":
        n = case["rays"]
        return {"bytes": n * 48 + min(n * 4, _triangles(case)) * TRI_BYTES, "flops": n * RAY_FLOPS}
    if kind == "batch":   # sides and spp are 0.3 to 1 of the case's, about 0.46 of the pixels and 0.65 of the samples
        pixels = case["scenes"] * 0.46 * case["side"] ** 2
        paths, tris = pixels * case["spp"] * 0.65, case["scenes"] * case["tris"] ** 0.75
    else:
        pixels, tris = case["width"] * case["height"], _triangles(case)
        paths = case["samples"] if case.get("sampling") == "uniform" else pixels * case["spp"] * case.get("batches", 1)
    seg = _segments(case)
    rays = seg * {"pt": 1, "ptdirect": 2, "ltdirect": 2, "bdpt": 2 + seg}[case["renderer"]]
    sides = 2 if kind == "grad" else 1   # the image, then the replay
    return {"bytes": sides * (pixels * 24 + tris * TRI_BYTES), "flops": sides * paths * (rays * RAY_FLOPS + seg * VERTEX_FLOPS)}


def exact(case, seed):
    """Closest hits in 64 bits by testing every triangle (ray queries of at
    most 2e9 ray-triangle pairs); nothing for renders, whose images are
    random estimates."""
    if case["kind"] != "trace" or case["any"] or case["rays"] * _triangles(case) > 2e9:
        return None
    d = _scene(case, seed).desc()
    rays = _rays(case, seed)
    v = torch.from_numpy(d["positions"].astype(np.float32).astype(np.float64)).to(DEVICE)[torch.from_numpy(d["faces"].astype(np.int64)).to(DEVICE)]
    a, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    out = []
    step = max(1, int(2e7 // a.shape[0]))
    for k in range(0, case["rays"], step):
        r = rays[k:k + step]
        o = torch.from_numpy(r["o"].astype(np.float64)).to(DEVICE)[:, None, :]
        w = torch.from_numpy(r["d"].astype(np.float64)).to(DEVICE)[:, None, :]
        tmin = torch.from_numpy(r["tmin"].astype(np.float64)).to(DEVICE)[:, None]
        tmax = torch.from_numpy(r["tmax"].astype(np.float64)).to(DEVICE)[:, None]
        p = torch.linalg.cross(w.expand(-1, a.shape[0], -1), e2[None].expand(w.shape[0], -1, -1))
        det = (p * e1).sum(-1)
        s = o - a
        u = (s * p).sum(-1) / det
        q = torch.linalg.cross(s, e1[None].expand(w.shape[0], -1, -1))
        vv = (w * q).sum(-1) / det
        t = (q * e2).sum(-1) / det
        hit = (det != 0) & (u >= 0) & (vv >= 0) & (u + vv <= 1) & (t > tmin) & (t < tmax)
        t = torch.where(hit, t, torch.full_like(t, math.inf))
        best, i = t.min(dim=1)
        found = torch.isfinite(best)
        pick = lambda x: torch.where(found, x.gather(1, i[:, None])[:, 0], torch.zeros_like(best))
        out.append((torch.where(found, best, tmax[:, 0]), pick(u), pick(vv)))
    t, u, vv = (torch.cat(x) for x in zip(*out))
    to = (lambda x: x) if case["where"] == "device" else (lambda x: x.cpu().numpy())
    return {"t": to(t), "u": to(u), "v": to(vv), "tri": None}
