"""The work a program has this package do on the GPU, as timed cases.

Four kinds of case, each a call a user's program makes on what it keeps
resident (a context and its scenes):

  rays    a batch of ray queries against a resident scene, closest hit or any
          hit: camera rays, scattered rays (bounces, probes) or shadow
          segments, on device arrays or through numpy arrays
  render  one render job, blocking: path or direct-lighting integrator
  serve   jobs of mixed size submitted together to the shared device
  open    a scene described on the host becomes resident (its acceleration
          structure is built) and answers a first query

Scenes are the benchmark's and the tests' procedural ones; they are built
once per size and stay, as a program's scene does, while rays, cameras and
sample streams follow the seed.
"""
import functools
import math

import numpy as np
import torch

from bling_amd import abi, scenes
from bling_amd import transform as T
from bling_amd.runtime import Context, GpuRenderer, GpuScene, Job, JobSpec
from bling_amd.scene import Material, SceneBuilder, View, const, rgb_illum, rgb_refl
from bling_amd.textures import Map3d, Tex

CLOSEST, ANY = "closest", "any"


def listed():
    return [
        # a program asks what lies under a few pixels: the smallest call there is
        _rays("pick_64", "soup", 2200, CLOSEST, "camera", 64, host=True),
        # a script holds its rays in numpy arrays (bling's own closures, batched)
        _rays("numpy_rays_50k", "stack", 100_000, CLOSEST, "scattered", 50_021, host=True),
        # primary visibility of a 2048 x 2048 image: neighbouring rays, hint given
        _rays("camera_rays_4m", "icosphere", 1_310_720, CLOSEST, "camera", 2048 * 2048),
        # the intersection benchmark's scattered rays, every direction and origin
        _rays("scattered_rays_4m", "icosphere", 1_310_720, CLOSEST, "scattered", 4_194_304),
        # shadow segments to an area light over a terrain, a ragged batch
        _rays("shadow_rays_1m", "grid", 1_000_000, ANY, "shadow", 1_000_003),
        # a thumbnail while the user moves the camera: launches and host work
        _render("thumbnail_64", "cornell", 0, 64, 64, 4),
        # the benchmark's Cornell box
        _render("cornell_256", "cornell", 0, 256, 256, 16),
        # a progressive HD-ish terrain with a wide filter and per-pixel variance
        _render("terrain_gauss_641x363", "grid", 1_000_000, 641, 363, 9, passes=2, filt="gauss", variance=True),
        # all BSDF kinds, deep paths, sky map: the divergent benchmark at a preview's size
        _render("divergent_512", "divergent", 600_000, 512, 512, 16, max_depth=16),
        # direct lighting with glass and mirror branches over textured matter
        _render("direct_textured_400x300", "materials", 0, 400, 300, 9, max_depth=5, integrator="direct"),
        # a render service's queue: jobs of several sizes over resident scenes
        {"name": "serve_24", "kind": "serve", "jobs": 24, "max_res": 512, "max_spp": 16, "tris": 400_000},
        # a mesh of a million triangles is opened and queried
        {"name": "open_1m", "kind": "open", "scene": "grid", "tris": 1_000_000, "n": 65_536},
    ]


def draw(rng):
    kind = rng.choice(("rays", "rays", "render", "render", "serve", "open"))
    if kind == "rays":
        scene = rng.choice(("soup", "stack", "icosphere", "grid"))
        tris = {"soup": 2200}.get(scene) or _log_int(rng, 2_000, 1_000_000)
        host = rng.random() < 0.3
        n = _log_int(rng, 1, 200_000 if host else 3_000_000)
        return _rays("", scene, tris, rng.choice((CLOSEST, ANY)), rng.choice(("camera", "scattered", "shadow")), n,
                     host=host)
    if kind == "render":
        scene = rng.choice(("cornell", "stack", "grid", "icosphere", "divergent", "materials"))
        w, h, spp = _log_int(rng, 16, 512), _log_int(rng, 16, 512), rng.choice((1, 4, 9, 16))
        direct = scene in ("cornell", "materials") and rng.random() < 0.4
        return _render("", scene, _log_int(rng, 2_000, 600_000), w, h, spp,
                       max_depth=rng.randint(1, 5) if direct else rng.randint(2, 10),
                       passes=rng.choice((1, 1, 2, 3)) if spp <= 4 else 1,
                       integrator="direct" if direct else "path", variance=rng.random() < 0.3,
                       filt=rng.choice(("box", "box", "gauss", "triangle", "mitchell")))
    if kind == "serve":
        return _nameless({"kind": "serve", "jobs": rng.randint(2, 20), "max_res": rng.choice((128, 256, 512)),
                          "max_spp": rng.choice((4, 9, 16)), "tris": _log_int(rng, 2_000, 400_000)})
    scene = rng.choice(("stack", "grid", "icosphere"))
    return _nameless({"kind": "open", "scene": scene, "tris": _log_int(rng, 500, 900_000),
                      "n": _log_int(rng, 1, 65_536)})


def _rays(name, scene, tris, query, rays, n, host=False):
    return _nameless({"name": name, "kind": "rays", "scene": scene, "tris": tris, "query": query, "rays": rays,
                      "n": n, "host": host})


def _render(name, scene, tris, w, h, spp, max_depth=5, passes=1, integrator="path", variance=False, filt="box"):
    return _nameless({"name": name, "kind": "render", "scene": scene, "tris": tris, "w": w, "h": h, "spp": spp,
                      "max_depth": max_depth, "passes": passes, "integrator": integrator, "variance": variance,
                      "filter": filt})


def _nameless(case):
    if not case.get("name"):
        case.pop("name", None)
    return case


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# ---------------------------------------------------------------- scenes
@functools.lru_cache(maxsize=None)
def _context():
    return Context(0)


@functools.lru_cache(maxsize=16)
def _flat(kind, tris):
    """The host description of a scene of about `tris` triangles."""
    if kind == "cornell":
        return scenes.cornell(256)
    if kind == "soup":  # triangles and every analytic shape kind
        return scenes.small_scene(num_tris=2000, num_spheres=200)
    if kind == "stack":
        return scenes.stack_scene(tris, seed=3)
    if kind == "grid":
        return scenes.grid_scene(tris, seed=1)
    if kind == "icosphere":
        levels = int(np.clip(round(math.log(tris / 20.0, 4.0)), 2, 8))
        return scenes.icosphere_scene(levels=levels, num_spheres=max(20, tris // 131), seed=1, res=256, lit=True)
    if kind == "divergent":
        side = max(8, int(math.sqrt(tris / 4.0)))
        return scenes.divergent_scene(res=256, hm=side, n_tori=10, torus_tris=max(40, tris // 20), n_spheres=100,
                                      sky=(128, 64))
    return _materials()


def _materials():
    """Spheres of the reflective, refractive and textured materials on a
    checkered floor under a quad light and a small sky map."""
    sb = SceneBuilder()
    floor = Material.matte(rgb_refl(0.7, 0.7, 0.7)).textured(0, abi.TEX_CHECKER, (1.0, 1.0, 1.0),
                                                             rgb_refl(0.15, 0.2, 0.5))
    noisy = Material.matte(const(0.5)).textured_inputs(
        spec={0: Tex.blend(Tex.spectrum(rgb_refl(0.8, 0.5, 0.2)), Tex.spectrum(rgb_refl(0.2, 0.3, 0.6)),
                           Tex.scale(0.5, 0.4, Tex.fbm(4, 0.5, Map3d.identity(T.scale((3.0, 3.0, 3.0))))))})
    mats = [Material.matte(rgb_refl(0.7, 0.3, 0.2), sigma=0.4), Material.plastic(rgb_refl(0.2, 0.3, 0.7), const(0.4), 0.02),
            Material.metal(const(0.2), const(3.9), 0.05), Material.glass(1.5, const(1.0), const(1.0)),
            Material.mirror(const(0.9)), Material.substrate(rgb_refl(0.5, 0.2, 0.2), const(0.1), const(0.0), 0.05, 0.1),
            noisy]
    f = sb.material(floor)
    sb.mesh(np.array([[-6, 0, -6], [6, 0, -6], [6, 0, 6], [-6, 0, 6]], np.float32), np.array([[0, 1, 2], [0, 2, 3]]),
            material=f)
    for k in range(21):
        m = sb.material(mats[k % len(mats)])
        r = 0.3 + 0.1 * (k % 3)
        sb.shape(abi.SHAPE_SPHERE, (r,), o2w=T.translate((-2.7 + 0.9 * (k % 7), r, -1.5 + 1.4 * (k // 7))), material=m)
    sb.shape(abi.SHAPE_QUAD, (0.8, 0.8), o2w=T.rotate_x(-90) @ T.translate((0.0, 4.0, 0.0)), material=f,
             emission=rgb_illum(8, 8, 8))
    sb.infinite_light(scenes.sky_gradient(64, 32) * np.float32(0.5), w2l=T.rotate_x(90))
    sb.look(T.look_at((0.0, 3.0, -6.0), (0.0, 0.3, 0.0), (0, 1, 0)), 45.0, 256, 256)
    return sb.build()


_EYE = {"cornell": ((0.5, 0.5, -1.4), (0.5, 0.5, 0.5), 40.0), "soup": ((0.5, 1.0, -3.6), (0.0, 0.0, 0.0), 45.0),
        "stack": ((3.5, 3.0, -4.5), (0.0, 0.6, 0.0), 45.0), "grid": ((0.0, 2.5, -3.5), (0.0, 0.2, 0.0), 50.0),
        "icosphere": ((0.6, 0.9, -3.4), (0.0, 0.0, 0.0), 50.0), "divergent": ((0.0, 2.6, -5.5), (0.0, 0.6, 0.0), 50.0),
        "materials": ((0.0, 3.0, -6.0), (0.0, 0.3, 0.0), 45.0)}
_FILTER = {"box": (abi.FILTER_BOX, (0.0, 0.0, 0.0, 0.0)), "gauss": (abi.FILTER_GAUSS, (2.0, 2.0, 2.0, 0.0)),
           "triangle": (abi.FILTER_TRIANGLE, (1.5, 1.5, 0.0, 0.0)),
           "mitchell": (abi.FILTER_MITCHELL, (2.0, 2.0, 1.0 / 3.0, 1.0 / 3.0))}


def _camera(kind, seed):
    """The scene's eye, moved a little by the seed: (eye, target, fov)."""
    eye, at, fov = _EYE[kind]
    rng = np.random.default_rng(seed)
    return tuple(float(x) for x in np.asarray(eye) + rng.uniform(-0.05, 0.05, 3)), at, fov


class _State:
    """What a program keeps between calls; its scenes are released with it."""

    def __init__(self, case, **kw):
        self.case = case
        self.__dict__.update(kw)

    def __del__(self):
        for s in getattr(self, "resident", ()):
            try:
                s.close()
            except Exception:
                pass


# ------------------------------------------------------------------ rays
def _ray_batch(case, seed):
    """(8, n) float32 on the GPU: ox oy oz dx dy dz tmin tmax."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 17)
    n, kind = case["n"], case.get("rays", "scattered")
    flat = _flat(case["scene"], case["tris"])
    lo, hi = (torch.tensor(x, device="cuda", dtype=torch.float32)[:, None] for x in scenes.scene_bounds(flat))
    rays = torch.empty((8, n), device="cuda")
    rays[6], rays[7] = 0.0, math.inf
    if kind == "camera":  # pixel centres of a square image in row order, jittered
        eye, at, fov = _camera(case["scene"], seed)
        side = max(1, math.isqrt(n - 1) + 1)
        k = torch.arange(n, device="cuda")
        jx, jy = torch.rand((2, n), device="cuda", generator=g)
        x = (((k % side) + jx) / side * 2 - 1) * math.tan(math.radians(fov / 2))
        y = (1 - ((k // side) + jy) / side * 2) * math.tan(math.radians(fov / 2))
        fwd = np.asarray(at) - np.asarray(eye)
        fwd = fwd / np.linalg.norm(fwd)
        right = np.cross((0.0, 1.0, 0.0), fwd)
        right = right / np.linalg.norm(right)
        up = np.cross(fwd, right)
        d = torch.stack([x * float(right[c]) + y * float(up[c]) + float(fwd[c]) for c in range(3)])
        rays[3:6] = d / d.norm(dim=0, keepdim=True)
        rays[0:3] = torch.tensor(eye, device="cuda", dtype=torch.float32)[:, None]
        return rays
    o = lo + (hi - lo) * torch.rand((3, n), device="cuda", generator=g)
    if kind == "shadow":  # toward points of a square light above the scene, up to just before it
        top = hi[1] + 0.5 * (hi - lo).max()
        half = 0.3 * (hi - lo)
        p = (lo + hi) / 2 + half * (2 * torch.rand((3, n), device="cuda", generator=g) - 1)
        p[1] = top
        d = p - o
        dist = d.norm(dim=0)
        rays[3:6] = d / dist
        rays[6] = 1e-3
        rays[7] = dist * 0.999
    else:
        u = 2 * torch.rand(n, device="cuda", generator=g) - 1
        phi = 2 * math.pi * torch.rand(n, device="cuda", generator=g)
        s = (1 - u * u).sqrt()
        rays[3:6] = torch.stack([s * phi.cos(), s * phi.sin(), u])
    rays[0:3] = o
    return rays


def _prepare_rays(case, seed):
    scene = _context().scene(_flat(case["scene"], case["tris"]))
    rays = _ray_batch(case, seed)
    st = _State(case, scene=scene, resident=[scene])
    if case["host"]:
        st.rays = np.ascontiguousarray(rays.t().cpu().numpy())
    else:
        n = case["n"]
        st.rays = rays
        st.t, st.b1, st.b2 = torch.empty((3, n), device="cuda")
        st.prim = torch.empty(n, device="cuda", dtype=torch.int32)
        st.occ = torch.empty(n, device="cuda", dtype=torch.uint8)
    return st


def _run_rays(st):
    case, s = st.case, st.scene
    coherent = case["rays"] == "camera"
    if case["host"]:
        if case["query"] == ANY:
            return {"occluded": s.intersects(st.rays, coherent=coherent)}
        t, b1, b2, prim = s.intersect(st.rays, coherent=coherent)
        return {"t": t, "b1": b1, "b2": b2, "prim": prim}
    ptrs = [r.data_ptr() for r in st.rays]
    if case["query"] == ANY:
        s.intersects_dev(ptrs, case["n"], st.occ.data_ptr(), coherent=coherent)
        return {"occluded": st.occ}
    s.intersect_dev(ptrs, case["n"], [x.data_ptr() for x in (st.t, st.b1, st.b2, st.prim)], coherent=coherent)
    return {"t": st.t, "b1": st.b1, "b2": st.b2, "prim": st.prim}


# --------------------------------------------------------------- renders
def _view(kind, seed, w, h, filt="box"):
    eye, at, fov = _camera(kind, seed)
    f, fp = _FILTER[filt]
    return View.perspective(T.look_at(eye, at, (0, 1, 0)), fov, w, h, filt=f, fparams=fp)


def _spp(n):
    """Square strata, as bling's sampler lays them out without overlap."""
    return math.isqrt(n), math.isqrt(n)


def _prepare_render(case, seed):
    scene = _context().scene(_flat(case["scene"], case["tris"]))
    nu, nv = _spp(case["spp"])
    spec = JobSpec(spp_nu=nu, spp_nv=nv, max_depth=case["max_depth"], sample_depth=3, rr_start_depth=3,
                   passes=case["passes"], seed=seed * 104729 + 1, variance=case["variance"],
                   view=_view(case["scene"], seed, case["w"], case["h"], case["filter"]), integrator=case["integrator"])
    return _State(case, scene=scene, renderer=GpuRenderer(spec), resident=[scene])


def _run_render(st):
    img, sq = st.renderer.render_plain(st.scene)
    out = {"weight": img[..., 0], "xyz": img[..., 1:]}
    if sq is not None:
        out["sq"] = sq
    return out


# The service's queue: job k's scene, edge and samples per pixel.
_SERVED = ("cornell", "stack", "icosphere")


def _served(case):
    edges = [e for e in (128, 256, 512, 192) if e <= case["max_res"]]
    spps = [s for s in (4, 16, 1, 9) if s <= case["max_spp"]]
    for k in range(case["jobs"]):
        yield _SERVED[k % 3], edges[(k * 5 // 3) % len(edges)], spps[(k * 7 // 2) % len(spps)]


def _prepare_serve(case, seed):
    ctx = _context()
    res = {k: ctx.scene(_flat(k, case["tris"] if k != "cornell" else 0)) for k in _SERVED}
    queue = []
    for k, (scene, edge, spp) in enumerate(_served(case)):
        nu, nv = _spp(spp)
        queue.append((res[scene], JobSpec(spp_nu=nu, spp_nv=nv, max_depth=5, sample_depth=3, rr_start_depth=3,
                                          seed=seed * 100003 + k, view=_view(scene, seed, edge, edge))))
    return _State(case, queue=queue, resident=list(res.values()))


def _run_serve(st):
    jobs = [Job(scene, spec) for scene, spec in st.queue]
    images = []
    for j in jobs:
        j.wait()
        images.append(j.poll()[0])
        j.release()
    return {"weight": [i[..., 0] for i in images], "xyz": [i[..., 1:] for i in images]}


# ------------------------------------------------------------------ open
def _prepare_open(case, seed):
    _context()
    flat = _flat(case["scene"], case["tris"])
    return _State(case, flat=flat, rays=np.ascontiguousarray(_ray_batch(case, seed).t().cpu().numpy()))


def _run_open(st):
    scene = GpuScene(_context(), st.flat)
    try:
        t, b1, b2, prim = scene.intersect(st.rays)
    finally:
        scene.close()
    return {"t": t, "b1": b1, "b2": b2, "prim": prim}


# ------------------------------------------------------------- interface
_KINDS = {"rays": (_prepare_rays, _run_rays), "render": (_prepare_render, _run_render),
          "serve": (_prepare_serve, _run_serve), "open": (_prepare_open, _run_open)}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state.case["kind"]][1](state)


def _prims(case, scene=None):
    """(triangles, shapes) of a case's scene, from its declared size."""
    kind, tris = scene or case["scene"], case["tris"]
    if kind == "cornell":
        return 34, 1
    if kind == "soup":
        return 2000, 200
    if kind == "materials":
        return 2, 22
    if kind == "icosphere":
        return 20 * 4 ** int(np.clip(round(math.log(tris / 20.0, 4.0)), 2, 8)), max(20, tris // 131)
    return tris, 100 if kind == "divergent" else 2


def _query_flops(tris, shapes):
    """One ray against a scene: two boxes a level of a balanced tree (18
    operations each), one triangle and one shape test at its end."""
    return 36.0 * (math.log2(tris + 1) + math.log2(shapes + 1)) + 60.0 + 60.0


def _scene_bytes(tris, shapes, touched):
    """Vertices (half as many as triangles) and indices, shapes, as far as
    `touched` queries can need them (a leaf each)."""
    return min(18.0 * tris + 128.0 * shapes, 200.0 * touched)


def work(case):
    if case["kind"] in ("rays", "open"):
        t, s = _prims(case)
        n = case["n"]
        out = 1 if case.get("query") == ANY else 16
        if case["kind"] == "open":  # reads the mesh, writes boxes and links of a tree over it
            return {"bytes": 18.0 * t + 128.0 * s + 64.0 * t + 48.0 * n,
                    "flops": 30.0 * t * math.log2(t + 1) + n * _query_flops(t, s)}
        return {"bytes": (32.0 + out) * n + _scene_bytes(t, s, n), "flops": n * _query_flops(t, s)}
    jobs = ([(s, e, e, p, 1, 5) for s, e, p in _served(case)] if case["kind"] == "serve" else
            [(case["scene"], case["w"], case["h"], case["spp"], case["passes"], case["max_depth"])])
    b = f = 0.0
    for scene, w, h, spp, passes, depth in jobs:
        t, s = _prims(case, scene)
        n = float(w * h * spp * passes)
        # per sample: the camera ray, and at its first vertices a shadow ray,
        # a continuation and 16 bands of light, surface and throughput
        verts = min(depth, 3)
        f += n * (_query_flops(t, s) * (1 + 2 * verts) + verts * (16 * 12 + 400))
        b += 16.0 * w * h + _scene_bytes(t, s, n)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Hits are fixed bit for bit (the reference's binary32 expressions, ties
    to the lowest id).  Film sums take their samples' values in any order."""
    return "exact" if case["kind"] in ("rays", "open") else {"rel": 1e-5}


# ------------------------------------------------------- 64-bit reference
def exact(case, seed):
    if case["kind"] == "render":
        # with the box filter every sample weighs 1 in its own pixel; a
        # Monte Carlo image has no value of its own beside its samples
        if case["filter"] != "box":
            return None
        full = np.full((case["h"], case["w"]), float(case["spp"] * case["passes"]))
        return {"weight": full, "xyz": None, **({"sq": None} if case["variance"] else {})}
    if case["kind"] == "serve":
        jobs = list(_served(case))
        return {"weight": [np.full((e, e), float(p)) for _, e, p in jobs], "xyz": [None] * len(jobs)}
    flat = _flat(case["scene"], case["tris"])
    if case["n"] * float(flat.num_prims) > 1.2e10:
        return None
    rays = _ray_batch(case, seed).double()
    any_hit = case.get("query") == ANY
    t, b1, b2, prim = _brute(flat, rays, any_hit)
    if any_hit:
        return {"occluded": (prim >= 0).cpu().numpy()}
    return {k: v.cpu().numpy() for k, v in (("t", t), ("b1", b1), ("b2", b2), ("prim", prim))}


def _brute(flat, rays, any_hit):
    """Closest hit of every ray over all primitives, in binary64; any_hit:
    a box then also stops rays that start inside it, as bling's does."""
    n = rays.shape[1]
    dev = rays.device
    v = torch.tensor(flat.vertices, device=dev, dtype=torch.float64)
    idx = torch.tensor(flat.indices, device=dev, dtype=torch.long)
    p1, e1, e2 = v[idx[:, 0]], v[idx[:, 1]] - v[idx[:, 0]], v[idx[:, 2]] - v[idx[:, 0]]
    best = torch.full((n,), math.inf, device=dev, dtype=torch.float64)
    b1, b2 = torch.zeros_like(best), torch.zeros_like(best)
    prim = torch.full((n,), -1, device=dev, dtype=torch.int32)
    step = max(1, int(3e7 // max(1, len(p1))))
    for a in range(0, n, step):
        z = min(n, a + step)
        o, d = rays[0:3, a:z].t()[:, None], rays[3:6, a:z].t()[:, None]
        tt, c1, c2 = _triangles(o, d, p1[None], e1[None], e2[None])
        ok = (c1 >= 0) & (c1 <= 1) & (c2 >= 0) & (c1 + c2 <= 1) & (tt >= rays[6, a:z, None]) & (tt <= rays[7, a:z, None])
        tt = torch.where(ok, tt, torch.inf)
        if tt.shape[1]:
            t, k = tt.min(dim=1)
            hit = torch.isfinite(t)
            best[a:z] = torch.where(hit, t, best[a:z])
            b1[a:z] = torch.where(hit, c1.gather(1, k[:, None])[:, 0], b1[a:z])
            b2[a:z] = torch.where(hit, c2.gather(1, k[:, None])[:, 0], b2[a:z])
            prim[a:z] = torch.where(hit, k.int(), prim[a:z])
    for s in range(flat.num_shapes):
        sh = flat.shapes[s]
        m = torch.tensor(list(sh.w2o), device=dev, dtype=torch.float64).view(4, 4)
        o = m[:3, :3] @ rays[0:3] + m[:3, 3:]
        d = m[:3, :3] @ rays[3:6]
        t = _shape(sh.type, list(sh.params), o, d, rays[6], rays[7], any_hit)
        hit = t < best
        best = torch.where(hit, t, best)
        b1, b2 = torch.where(hit, 0.0, b1), torch.where(hit, 0.0, b2)
        prim = torch.where(hit, len(p1) + s, prim).int()
    return torch.where(prim >= 0, best, 0.0), b1, b2, prim


def _dot(a, b):
    return a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1] + a[..., 2] * b[..., 2]


def _cross(a, b):
    return torch.stack(torch.broadcast_tensors(a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1],
                                               a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2],
                                               a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]), dim=-1)


def _triangles(o, d, p1, e1, e2):
    s1 = _cross(d, e2)
    inv = 1.0 / _dot(s1, e1)
    w = o - p1
    s2 = _cross(w, e1)
    return _dot(e2, s2) * inv, _dot(w, s1) * inv, _dot(d, s2) * inv


def _shape(kind, p, o, d, tmin, tmax, any_hit):
    """t of a shape's closest hit in object space, inf on a miss."""
    def pick(t0, t1, ok0, ok1):
        return torch.where(ok0 & (t0 >= tmin) & (t0 <= tmax), t0,
                           torch.where(ok1 & (t1 >= tmin) & (t1 <= tmax), t1, torch.inf))

    def phi_ok(t, most):
        a = torch.atan2(o[1] + t * d[1], o[0] + t * d[0])
        return torch.where(a < 0, a + 2 * math.pi, a) <= most

    if kind == abi.SHAPE_BOX:  # bling's box has its closest hit at its near face only
        near, far = torch.full_like(o[0], -math.inf), torch.full_like(o[0], math.inf)
        for c in range(3):
            a, b = (p[c] - o[c]) / d[c], (p[3 + c] - o[c]) / d[c]
            near, far = torch.maximum(near, torch.minimum(a, b)), torch.minimum(far, torch.maximum(a, b))
        if any_hit:
            near = torch.maximum(near, tmin)
            return torch.where(near <= torch.minimum(far, tmax), near, torch.inf)
        return torch.where((near <= far) & (near >= tmin) & (near <= tmax), near, torch.inf)
    if kind in (abi.SHAPE_QUAD, abi.SHAPE_DISK):
        t = ((p[0] if kind == abi.SHAPE_DISK else 0.0) - o[2]) / d[2]
        x, y = o[0] + t * d[0], o[1] + t * d[1]
        if kind == abi.SHAPE_QUAD:
            ok = (x.abs() <= p[0]) & (y.abs() <= p[1])
        else:
            r2 = x * x + y * y
            ok = (r2 <= p[1] * p[1]) & (r2 >= p[2] * p[2]) & phi_ok(t, p[3])
        return torch.where(ok & (t >= tmin) & (t <= tmax), t, torch.inf)
    k = 3 if kind == abi.SHAPE_SPHERE else 2  # a cylinder is the quadric without z
    a = (d[:k] * d[:k]).sum(0)
    b = 2 * (o[:k] * d[:k]).sum(0)
    c = (o[:k] * o[:k]).sum(0) - p[0] * p[0]
    disc = b * b - 4 * a * c
    real = disc >= 0
    root = disc.clamp(min=0).sqrt()
    t0, t1 = (-b - root) / (2 * a), (-b + root) / (2 * a)
    if kind == abi.SHAPE_SPHERE:
        return pick(t0, t1, real, real)
    ok = [real & (o[2] + t * d[2] > p[1]) & (o[2] + t * d[2] < p[2]) & phi_ok(t, p[3]) for t in (t0, t1)]
    return pick(t0, t1, *ok)
