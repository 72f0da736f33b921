"""Performance cases of the framework: ray queries, renders, adjoint renders
and batches through the package's public entry points.

Scenes (built and finalized once per process, as a program keeps them):
  * "sphere": the Cornell box and ceiling light around a displaced geodesic
    sphere of frequency `freq` (20 freq^2 triangles, per-triangle albedo, 10%
    Phong), freq 16 (5,132 triangles with the box) to 256 (1,310,732);
  * "sky": an open scene (ground, displaced icosphere of `sub` subdivisions,
    a ball, an area light) under a 512 x 256 environment map with a sun;
  * "inverse": the all-diffuse sphere of the inverse-rendering configuration;
  * "soup": `ntri` unconnected small triangles in the unit cube.
A case's seed makes its rays, its render seed and its loss gradient.
"""
import functools
import math

import numpy as np
import torch

import mcrt_amd
from mcrt_amd import scenes

PATH = dict(max_depth=8, rr_start=3, rr_prob=0.8)
BOX_LO, BOX_HI = (1.0, 1.0, 1.0), (54.0, 53.0, 54.0)


def listed():
    return [
        # One ray from host memory, answered before the call returns: picking,
        # or a program written against the reference's Scene::intersect(ray).
        dict(name="pick_host", kind="query", scene="sphere", size=16, rays="incoherent", any=False, host=True, n=1),
        # A short list of device rays inside a simulation step: latency.
        dict(name="closest_small", kind="query", scene="sphere", size=16, rays="incoherent", any=False, host=False,
             n=1000),
        # Visibility tests between points of a mid-size scene (probes,
        # radiosity-like solvers), an odd count.
        dict(name="any_mid", kind="query", scene="sphere", size=71, rays="segments", any=True, host=False, n=500001),
        # The headline query: incoherent closest hit on the 1.3M-triangle mesh.
        dict(name="closest_mesh", kind="query", scene="sphere", size=256, rays="incoherent", any=False, host=False,
             n=1 << 24),
        # The same kind of rays over a BVH larger than the last-level cache.
        dict(name="closest_soup", kind="query", scene="soup", size=1 << 21, rays="incoherent", any=False, host=False,
             n=1 << 23),
        # A sensor or G-buffer frame: coherent primary rays over the soup.
        dict(name="primary_soup", kind="query", scene="soup", size=1 << 21, rays="pinhole", any=False, host=False,
             n=2048 * 2048),
        # A progressive preview's frame: a thumbnail at one sample per pixel.
        dict(name="preview", kind="render", scene="sphere", size=16, w=97, h=61, spp=1, nee=True),
        # The reference's own scale: 256 x 256, 16 spp, 5k triangles.
        dict(name="render_small", kind="render", scene="sphere", size=16, w=256, h=256, spp=16, nee=True),
        # The headline frame: 1024 x 1024, 64 spp, 1.3M triangles.
        dict(name="render_large", kind="render", scene="sphere", size=256, w=1024, h=1024, spp=64, nee=True),
        # An open scene under an environment map with the area light.
        dict(name="render_sky", kind="render", scene="sky", size=6, w=640, h=360, spp=16, nee=True),
        # One step of inverse rendering: film and gradients of 100k triangles.
        dict(name="adjoint_step", kind="adjoint", scene="inverse", size=71, w=512, h=512, spp=32),
        # A batch of uneven scenes replayed as a graph (dataset generation).
        dict(name="batch_uneven", kind="batch", count=12, seed_scenes=21),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "query", "query", "render", "render", "adjoint", "batch"])
    if kind == "query":
        scene = rng.choice(["sphere", "sphere", "soup"])
        any_hit = rng.random() < 0.4
        rays = rng.choice(["incoherent", "segments"] if any_hit else ["incoherent", "pinhole"])
        host = rng.random() < 0.2
        size = _log(rng, 16, 256) if scene == "sphere" else _log(rng, 1 << 12, 1 << 20)
        n = _log(rng, 1, 1 << 16) if host else _log(rng, 64, 1 << 23)
        return dict(kind=kind, scene=scene, size=size, rays=rays, any=any_hit, host=host, n=n)
    if kind == "render":
        scene = rng.choice(["sphere", "sphere", "sky"])
        size = _log(rng, 16, 200) if scene == "sphere" else rng.randint(3, 7)
        return dict(kind=kind, scene=scene, size=size, w=_log(rng, 33, 800), h=_log(rng, 33, 800),
                    spp=_log(rng, 1, 64), nee=rng.random() < 0.8)
    if kind == "adjoint":
        return dict(kind=kind, scene="inverse", size=_log(rng, 16, 120), w=_log(rng, 65, 512), h=_log(rng, 65, 512),
                    spp=_log(rng, 1, 32))
    return dict(kind=kind, count=rng.randint(3, 12), seed_scenes=rng.randint(1, 1 << 20))


@functools.lru_cache(maxsize=1)
def _context():
    return mcrt_amd.Context(0)


@functools.lru_cache(maxsize=16)
def _scene(kind, size, w=0, h=0, noise=7, albedo=11):
    """A finalized scene with its camera; the few a program works with stay."""
    if kind == "soup":
        s = mcrt_amd.Scene(_context())
        grey = s.add_material(mcrt_amd.DIFF, (0.7, 0.7, 0.7))
        s.add(scenes.soup(size), grey)
        s.finalize()
        return s
    if kind == "sky":
        s = scenes.outdoor(sub=size, light=True).to_scene(_context(), w, h)
        s.set_envmap(scenes.sky_envmap(512, 256))
        return s
    if kind == "inverse":
        data, init = scenes.inverse_rendering(freq=size)
        s = data.to_scene(_context(), w, h)
        s.set_material_rgb(init)
        return s
    return scenes.cornell_displaced(geodesic_freq=size, noise_seed=noise, albedo_seed=albedo).to_scene(_context(), w, h)


def _rays(case, seed):
    """The case's rays (n, 8), made on the GPU."""
    g = torch.Generator("cuda").manual_seed(int(seed))
    n = case["n"]
    unit = case["scene"] == "soup"
    lo = torch.tensor((0.0, 0.0, 0.0) if unit else BOX_LO, device="cuda")
    hi = torch.tensor((1.0, 1.0, 1.0) if unit else BOX_HI, device="cuda")

    def points():
        return lo + (hi - lo) * torch.rand(n, 3, device="cuda", generator=g)

    r = torch.empty(n, 8, device="cuda")
    r[:, 3] = 1e-4
    r[:, 7] = math.inf
    if case["rays"] == "pinhole":
        # a square grid from outside the front, jittered by the seed
        side = max(1, math.isqrt(n - 1) + 1)
        i = torch.arange(n, device="cuda")
        jit = torch.rand(n, 2, device="cuda", generator=g)
        x = ((i % side) + jit[:, 0]) / side - 0.5
        y = ((i // side) + jit[:, 1]) / side - 0.5
        mid = 0.5 * (lo + hi)
        eye = mid - torch.tensor((0.0, 0.0, 2.0), device="cuda") * (hi - lo)
        d = torch.stack([0.7 * x, 0.7 * y, torch.ones_like(x)], 1)
        r[:, :3] = eye
        r[:, 4:7] = d / d.norm(dim=1, keepdim=True)
    elif case["rays"] == "segments":
        # between two points: unit direction, tmax the distance
        o, q = points(), points()
        dist = (q - o).norm(dim=1, keepdim=True).clamp_min(1e-3)
        r[:, :3] = o
        r[:, 4:7] = (q - o) / dist
        r[:, 7] = dist[:, 0] - 1e-4
    else:
        d = torch.randn(n, 3, device="cuda", generator=g)
        r[:, :3] = points()
        r[:, 4:7] = d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)
        if case["any"]:
            r[:, 7] = 0.25 * (hi - lo).max()
    return r


def _uneven(case):
    """(frequency, side, spp) of the batch's scenes: triangle counts
    log-uniform in 1k..100k, square films, few to many samples."""
    rng = np.random.default_rng(case["seed_scenes"])
    k = case["count"]
    freq = np.round(np.sqrt(np.exp(rng.uniform(np.log(1e3), np.log(1e5), k)) / 20.0)).astype(int)
    side = rng.choice((96, 128, 256, 384), k)
    spp = rng.choice((4, 8, 16, 32), k)
    return [(int(f), int(s), int(p)) for f, s, p in zip(freq, side, spp)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        parts = _uneven(case)
        ss = [_scene("sphere", f, side, side, albedo=11 + i) for i, (f, side, _) in enumerate(parts)]
        params = [dict(spp=p, max_depth=6, rr_start=3, rr_prob=0.8, seed=int(seed), nee=True) for _, _, p in parts]
        films = [torch.empty(side, side, 3, device="cuda") for _, side, _ in parts]
        return dict(case=case, batch=mcrt_amd.Batch(ss, params, films, graph=True), films=films)
    if kind == "query":
        s = _scene(case["scene"], case["size"])
        rays = _rays(case, seed)
        n = case["n"]
        if case["host"]:
            rays = rays.cpu().numpy()
            out = np.empty(n, np.uint8) if case["any"] else np.empty((n, 4), np.int32)
        else:
            out = torch.empty(n, dtype=torch.uint8, device="cuda") if case["any"] else \
                torch.empty(n, 4, dtype=torch.int32, device="cuda")
        return dict(case=case, scene=s, rays=rays, out=out)
    s = _scene(case["scene"], case["size"], case["w"], case["h"])
    film = torch.empty(case["h"], case["w"], 3, device="cuda")
    st = dict(case=case, scene=s, film=film, seed=int(seed))
    if kind == "adjoint":
        g = torch.Generator("cuda").manual_seed(int(seed))
        # dLoss/dfilm of an L2 loss: small differences of either sign
        st["dfilm"] = torch.randn(case["h"], case["w"], 3, device="cuda", generator=g) * 0.1
        ntri = s.num_triangles()
        st["albedo"] = torch.empty(ntri, 3, device="cuda")
        st["emission"] = torch.empty(ntri, 3, device="cuda")
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "query":
        if case["any"]:
            return state["scene"].occluded(state["rays"], state["out"])
        hits = state["scene"].intersect(state["rays"], state["out"])
        f32 = np.float32 if case["host"] else torch.float32
        return dict(prim=hits[:, 0], tuv=hits[:, 1:].view(f32))
    if kind == "render":
        return state["scene"].render(state["film"], spp=case["spp"], seed=state["seed"], nee=case["nee"], **PATH)
    if kind == "adjoint":
        state["scene"].render_adjoint(state["dfilm"], state["albedo"], state["emission"], state["film"],
                                      spp=case["spp"], seed=state["seed"], max_depth=6, rr_start=3, rr_prob=0.8)
        return dict(albedo=state["albedo"], emission=state["emission"], film=state["film"])
    state["batch"].render()
    return state["films"]


def _ntri(scene, size):
    if scene == "soup":
        return size
    return 20 * 4 ** size + 100 if scene == "sky" else 20 * size * size + 12


def work(case):
    """Bytes: rays, triangles, films and gradients once each.  Flops: per ray
    two box tests (about 40) per doubling of the triangle count and one
    triangle test (about 50); per path vertex two rays and about 300 of
    shading, with four vertices to a path."""
    def ray(ntri):
        return 40.0 * math.log2(ntri) + 50.0

    if case["kind"] == "query":
        ntri = _ntri(case["scene"], case["size"])
        return {"bytes": case["n"] * (32 + (1 if case["any"] else 16)) + 36 * ntri, "flops": case["n"] * ray(ntri)}
    if case["kind"] == "batch":
        parts = _uneven(case)
        return {"bytes": sum(12 * s * s + 84 * _ntri("sphere", f) for f, s, _ in parts),
                "flops": sum(4.0 * s * s * p * (2 * ray(_ntri("sphere", f)) + 300) for f, s, p in parts)}
    ntri = _ntri(case["scene"], case["size"])
    pix = case["w"] * case["h"]
    flops = 4.0 * pix * case["spp"] * (2 * ray(ntri) + 300)
    if case["kind"] == "adjoint":
        return {"bytes": 24 * pix + 108 * ntri, "flops": 2 * flops}
    return {"bytes": 12 * pix + 84 * ntri, "flops": flops}


def exact(case, seed):
    """Closest hits by brute force over every triangle in 64 bits, where that
    is quick; the hit's parameters only (its triangle is a whole number)."""
    if case["kind"] != "query" or case["any"] or case["rays"] == "pinhole":
        return None
    ntri = _ntri(case["scene"], case["size"])
    if case["n"] * ntri > 2e9 or case["scene"] == "soup":
        return None
    tri = scenes.cornell_displaced(geodesic_freq=case["size"]).tris
    tri = torch.from_numpy(tri).cuda().double().reshape(-1, 3, 3)
    v0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    best = []
    for r in _rays(case, seed).double().split(max(1, (1 << 23) // ntri)):
        o, d = r[:, None, :3], r[:, None, 4:7]
        p = torch.linalg.cross(d.expand(-1, ntri, -1), e2.expand(len(r), -1, -1))
        det = (e1 * p).sum(-1)
        s = o - v0
        u = (s * p).sum(-1) / det
        q = torch.linalg.cross(s, e1.expand(len(r), -1, -1))
        v = (d * q).sum(-1) / det
        t = (e2 * q).sum(-1) / det
        ok = (det.abs() >= 1e-6) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > r[:, None, 3]) & (t < r[:, None, 7])
        t = torch.where(ok, t, math.inf)
        k = t.argmin(1, keepdim=True)
        t = t.gather(1, k)
        miss = torch.isinf(t)
        u, v = (torch.where(miss, 0.0, x.gather(1, k)) for x in (u, v))
        best.append(torch.cat([t, u, v], 1))
    return dict(prim=None, tuv=torch.cat(best))
