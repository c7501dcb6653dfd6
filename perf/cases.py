"""The work that users of this framework have it do, as timed cases.

A case is a dict of plain values; its "kind" says which entry point it goes
through:

  query   DeviceScene.query: a batch of rays against a resident scene, closest
          hit or any hit, fast or exact traversal
  render  renderer.render_device: one image of a resident scene, by one of the
          deterministic integrators or the path tracer
  batch   serving.render_batch: many small path-traced jobs of several resident
          scenes in one call

prepare() makes the scene and the rays or render settings from the seed, run()
is one call, work() what that call cannot do without, and exact() the same
result in 64 bits by brute force over the primitives, where that is affordable.
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

from muon_amd import Context, DeviceScene, HostScene, scenes
from muon_amd._lib import RenderParams
from muon_amd.renderer import render_device
from muon_amd.serving import engine_config, render_batch
from muon_amd.workloads import sphere_field_scene

DEVICE = "cuda:0"
DETERMINISTIC = ("normals", "depth", "albedo", "raytracer", "analyticdirect")


def listed():
    """Twelve cases from a single pick to the largest batch and image."""
    return [
        # an editor's pick or a placement probe: a handful of rays, where only latency counts
        dict(name="pick_cornell", kind="query", scene="cornell", size=0, rays=64, any_hit=False, tmax=False,
             exact=False),
        # collision or baking probes: a ragged batch of bounded rays on a mid-sized mesh
        dict(name="probe_icosphere", kind="query", scene="icosphere", size=5, rays=20011, any_hit=False, tmax=True,
             exact=False),
        # the throughput benchmark: incoherent closest hits on the level-7 icosphere
        dict(name="closest_icosphere", kind="query", scene="icosphere", size=7, rays=1 << 24, any_hit=False,
             tmax=False, exact=False),
        # visibility between points of a sphere field
        dict(name="any_spheres", kind="query", scene="spheres", size=10000, rays=3000017, any_hit=True, tmax=True,
             exact=False),
        # callers that need the reference's own hits, ties included
        dict(name="exact_icosphere", kind="query", scene="icosphere", size=6, rays=300007, any_hit=False,
             tmax=False, exact=True),
        # a preview of a mesh
        dict(name="normals_icosphere", kind="render", scene="icosphere", size=6, integrator="normals", width=640,
             height=480, spp=1, depth=5, nee="off", sampling="brdf", roulette=False, lights=1),
        # a Whitted image: shadows and reflections of many spheres, antialiased
        dict(name="raytrace_spheres", kind="render", scene="mirrors", size=500, integrator="raytracer", width=641,
             height=479, spp=4, depth=5, nee="off", sampling="brdf", roulette=False, lights=1),
        # the small path-traced image: the Cornell box
        dict(name="path_cornell", kind="render", scene="cornell", size=0, integrator="pathtracer", width=256,
             height=256, spp=16, depth=5, nee="mis", sampling="brdf", roulette=False, lights=1),
        # path length by roulette alone, several light samples, odd image sides
        dict(name="path_roulette", kind="render", scene="icosphere", size=4, integrator="pathtracer", width=317,
             height=211, spp=25, depth=-1, nee="on", sampling="cosine", roulette=True, lights=4),
        # the ordinary image: a mesh under light and BRDF sampling
        dict(name="path_icosphere", kind="render", scene="icosphere", size=7, integrator="pathtracer", width=512,
             height=512, spp=64, depth=8, nee="mis", sampling="brdf", roulette=False, lights=1),
        # a large image of many materials, without light sampling
        dict(name="path_spheres", kind="render", scene="spheres", size=10000, integrator="pathtracer", width=1024,
             height=1024, spp=32, depth=8, nee="off", sampling="brdf", roulette=False, lights=1),
        # thumbnails of several scenes in one call
        dict(name="batch_small", kind="batch", jobs=48, width=128, spp_lo=4, spp_hi=16, depth=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["query", "query", "query", "render", "render", "path", "path", "batch"])
    if kind == "batch":
        lo = rng.randint(1, 8)
        return dict(kind="batch", jobs=_log(rng, 5, 48), width=rng.randint(40, 128), spp_lo=lo,
                    spp_hi=lo + rng.randint(0, 8), depth=rng.randint(3, 8))
    scene = rng.choice(["cornell", "icosphere", "spheres", "mirrors"])
    size = {"cornell": 0, "icosphere": rng.randint(3, 7), "spheres": _log(rng, 50, 10000),
            "mirrors": _log(rng, 20, 1000)}[scene]
    if kind == "query":
        exact = rng.random() < 0.3
        return dict(kind="query", scene=scene, size=size, rays=_log(rng, 1, 1 << 20 if exact else 1 << 24),
                    any_hit=rng.random() < 0.4, tmax=rng.random() < 0.5, exact=exact)
    if kind == "render":
        integrator = rng.choice(DETERMINISTIC)
        return dict(kind="render", scene=scene, size=size, integrator=integrator, width=_log(rng, 30, 1024),
                    height=_log(rng, 30, 1024), spp=rng.choice([1, 1, rng.randint(2, 9)]), depth=rng.randint(1, 6),
                    nee="off", sampling="brdf", roulette=False, lights=1)
    width, height = _log(rng, 30, 1024), _log(rng, 30, 1024)
    return dict(kind="render", scene=scene, size=size, integrator="pathtracer", width=width, height=height,
                spp=max(1, min(64, _log(rng, 1, 64), (1 << 24) // (width * height))), depth=rng.randint(1, 8),
                nee=rng.choice(["off", "on", "mis"]), sampling=rng.choice(["hemisphere", "cosine", "brdf"]),
                roulette=rng.random() < 0.5, lights=rng.choice([1, 1, 2, 4]))


# ---------------------------------------------------------------- scenes
@functools.lru_cache(maxsize=None)
def _context(use):
    """A program's device context, kept while it runs: one for queries and
    single renders, one for batches."""
    return Context(0)


def _mirrors_text(n, seed):
    """Shiny spheres over a reflecting floor under a point and a directional
    light (and a quad light for the analytic integrator)."""
    rng = np.random.default_rng(seed)
    half = 2.0 * (n / 50.0) ** (1.0 / 3.0)
    lines = [f"camera 0 {half:.6g} {3.2 * half:.6g}  0 0 0  0 1 0  45", "max_depth 5",
             f"point_light {half:.6g} {3 * half:.6g} {2 * half:.6g} 1 1 1", "directional_light 0.3 1 0.4 0.3 0.3 0.3",
             f"quad_light {-0.25 * half:.6g} {1.9 * half:.6g} {-0.25 * half:.6g}  0 0 {0.5 * half:.6g}  "
             f"{0.5 * half:.6g} 0 0  4 4 4",
             "ambient 0.05 0.05 0.05", "specular 0.3 0.3 0.3", "diffuse 0.4 0.4 0.4", "shininess 40",
             f"vertex {-6 * half:.6g} {-1.2 * half:.6g} {-6 * half:.6g}",
             f"vertex {-6 * half:.6g} {-1.2 * half:.6g} {6 * half:.6g}",
             f"vertex {6 * half:.6g} {-1.2 * half:.6g} {6 * half:.6g}",
             f"vertex {6 * half:.6g} {-1.2 * half:.6g} {-6 * half:.6g}", "tri 0 1 2", "tri 0 2 3"]
    for c, r, k in zip(rng.uniform(-half, half, (n, 3)), rng.uniform(0.1, 0.4, n), rng.uniform(0.1, 0.8, (n, 3))):
        lines += ["diffuse %.6g %.6g %.6g" % tuple(k), "sphere %.6g %.6g %.6g %.6g" % (*c, r)]
    return "\n".join(lines) + "\n"


def _host_scene(scene, size, seed, build_on_device=False):
    """The parsed scene. The Cornell box is the same for every seed; the
    others are displaced or placed by it."""
    if scene == "cornell":
        return HostScene.from_text(scenes.cornell_text(seed=seed % 1000))
    if scene == "spheres":
        return HostScene.from_text(scenes.sphere_field_text(n=size, seed=seed))
    if scene == "mirrors":
        return HostScene.from_text(_mirrors_text(size, seed))
    with tempfile.TemporaryDirectory() as tmp:
        text = scenes.icosphere_text(level=size, seed=seed, mesh_file=os.path.join(tmp, "mesh.ply"))
        return HostScene.from_text(text, device_bvh=build_on_device)


def _bounds(host):
    b = host.arrays()["node_bounds"][0]
    return b[:3], b[3:]


def _rays(case, host, seed):
    """Origins uniform in the scene's box (in the mesh's for the icosphere, so
    that rays start inside and outside of it), directions uniform on the
    sphere, bounded rays up to the box's diagonal."""
    n = case["rays"]
    lo, hi = _bounds(host)
    if case["scene"] == "icosphere":
        lo, hi = np.array([-0.42, 0.18, -0.42]), np.array([0.42, 1.02, 0.42])
    gen = torch.Generator(DEVICE)
    gen.manual_seed(seed)
    lo = torch.tensor(lo, dtype=torch.float32, device=DEVICE)
    hi = torch.tensor(hi, dtype=torch.float32, device=DEVICE)
    o = lo + torch.rand(n, 3, generator=gen, device=DEVICE) * (hi - lo)
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=gen, device=DEVICE), dim=1)
    t = None
    if case["tmax"]:
        t = torch.rand(n, generator=gen, device=DEVICE) * float((hi - lo).norm()) + 1e-3
    return o.contiguous(), d.contiguous(), t


NEE = {"off": 0, "on": 1, "mis": 2}
SAMPLING = {"hemisphere": 0, "cosine": 1, "brdf": 2}
INTEGRATOR = {"normals": 0, "albedo": 1, "depth": 2, "raytracer": 3, "analyticdirect": 4, "pathtracer": 5}


def _params(case, host, seed):
    p = RenderParams.from_buffer_copy(host.params)
    if case["scene"] == "icosphere":
        scenes.random_pose(p, "ico", np.random.default_rng(seed), case["width"], case["height"])
    else:
        p.width, p.height = case["width"], case["height"]
        p.tan_fov_x = p.tan_fov_y * np.float32(p.width / p.height)
    p.spp, p.max_depth, p.seed = case["spp"], case["depth"], seed & 0x7FFFFFFF
    p.integrator, p.nee = INTEGRATOR[case["integrator"]], NEE[case["nee"]]
    p.importance_sampling, p.russian_roulette = SAMPLING[case["sampling"]], int(case["roulette"])
    p.light_samples, p.light_stratify = case["lights"], int(case["lights"] == 4)
    return p


def prepare(case, seed):
    """The resident scene, and the rays, the settings or the jobs."""
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    host = _host_scene(case["scene"], case["size"], seed)
    state = {"kind": case["kind"], "scene": DeviceScene(_context("single"), host), "case": dict(case)}
    if case["kind"] == "query":
        state["rays"] = _rays(case, host, seed)
    else:
        state["params"] = _params(case, host, seed)
        state["film"] = torch.empty(case["height"], case["width"], 3, device=DEVICE)
    return state


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    ctx = _context("batch")
    pool = []
    for level in (3, 4):
        host = _host_scene("icosphere", level, seed + level, build_on_device=True)
        pool.append(("ico", host, DeviceScene(ctx, host)))
    for n in (1000, 8000):
        host, dev = sphere_field_scene(ctx, n, seed + n)
        pool.append(("spheres", host, dev))
    jobs = []
    for i in range(case["jobs"]):
        kind, host, dev = pool[i % len(pool)]
        p = RenderParams.from_buffer_copy(host.params)
        scenes.random_pose(p, kind, rng, case["width"], case["width"])
        p.spp = int(rng.integers(case["spp_lo"], case["spp_hi"] + 1))
        p.max_depth, p.seed = case["depth"], int(rng.integers(1 << 31))
        jobs.append((dev, p, i))
    film = 24 * case["width"] ** 2 + 256
    config = engine_config(max_jobs=128, film_budget_bytes=film * case["jobs"] + (1 << 20), iterations_per_poll=4)
    return {"kind": "batch", "context": ctx, "jobs": jobs, "config": config}


def run(state):
    """One call. A render's ray counts (and, for the deterministic
    integrators, test counts) are part of its result."""
    if state["kind"] == "query":
        case = state["case"]
        o, d, t = state["rays"]
        if case["any_hit"]:
            return {"occluded": state["scene"].intersect_any(o, d, t, exact=case["exact"])}
        prim, dist = state["scene"].intersect_closest(o, d, t, exact=case["exact"])
        return {"prim": prim, "t": dist}
    if state["kind"] == "render":
        film, st = render_device(state["scene"], state["params"], state["film"])
        out = {"film": film, "rays": np.array([st.primary_rays, st.secondary_rays, st.shadow_rays], np.int64)}
        if state["case"]["integrator"] != "pathtracer":
            out["tests"] = np.array([st.object_tests, st.object_hits, st.bounds_tests, st.bounds_hits], np.int64)
        return out
    films, _, st = render_batch(state["context"], state["jobs"], state["config"])
    return {"films": films, "rays": np.array([st.primary_rays, st.secondary_rays, st.shadow_rays], np.int64)}


# ---------------------------------------------------------------- work
def _prims(case):
    return {"cornell": 36, "icosphere": 20 * 4 ** case["size"] + 12, "spheres": case["size"] + 8,
            "mirrors": case["size"] + 4}[case["scene"]]


def _ray_flops(prims):
    """A ray needs two slab tests (12 operations) per level of a binary tree
    and one primitive test (60) with its transform (30)."""
    return 24 * math.log2(max(2, prims)) + 90


def work(case):
    """Rays or image once, the primitives once (48 bytes each); path lengths
    are the depth limit's, eight for roulette alone."""
    if case["kind"] == "query":
        n, prims = case["rays"], _prims(case)
        per_ray = 24 + (4 if case["tmax"] else 0) + (1 if case["any_hit"] else 8)
        return {"bytes": n * per_ray + 48 * min(prims, 8 * n), "flops": n * _ray_flops(prims)}
    if case["kind"] == "batch":
        pixels = case["jobs"] * case["width"] ** 2
        samples = pixels * (case["spp_lo"] + case["spp_hi"]) / 2
        return {"bytes": 12 * pixels + 48 * 15000, "flops": samples * 0.5 * case["depth"] * (_ray_flops(4000) + 300)}
    samples = case["width"] * case["height"] * case["spp"]
    prims = _prims(case)
    vertices = 1.0
    if case["integrator"] in ("pathtracer", "raytracer"):
        vertices = 0.5 * (case["depth"] if case["depth"] > 0 else 8) + 0.5
    rays = vertices * (1 + (case["lights"] if case["nee"] != "off" else 0))
    return {"bytes": 12 * case["width"] * case["height"] + 48 * prims,
            "flops": samples * (rays * _ray_flops(prims) + vertices * 150)}


# ---------------------------------------------------------------- 64 bits
MAX_PAIRS = 3e10  # ray-primitive pairs of the brute force


def exact(case, seed):
    """Distances of the closest hits, and from them one-sample depth and
    normals images, by testing every primitive against every ray in float64."""
    if case["kind"] == "query":
        if case["any_hit"] or case["rays"] * _prims(case) > MAX_PAIRS:
            return None
        host = _host_scene(case["scene"], case["size"], seed)
        o, d, t = _rays(case, host, seed)
        dist, _ = _brute_force(host, o.double(), d.double(), None if t is None else t.double())
        return {"prim": None, "t": torch.where(torch.isfinite(dist), dist, 0.0)}
    if case["kind"] != "render" or case["integrator"] not in ("normals", "depth") or case["spp"] != 1:
        return None
    if case["width"] * case["height"] * _prims(case) > MAX_PAIRS:
        return None
    host = _host_scene(case["scene"], case["size"], seed)
    p = _params(case, host, seed)
    o, d = _camera_rays(p)
    dist, prim = _brute_force(host, o, d, None)
    hit = torch.isfinite(dist)
    if case["integrator"] == "depth":
        film = (1 / (1 + dist)).unsqueeze(1).expand(-1, 3)
    else:
        film = _normals(host, prim, o + torch.where(hit, dist, 0.0).unsqueeze(1) * d) * 0.5 + 0.5
    film = torch.where(hit.unsqueeze(1), film, 0.0).reshape(p.height, p.width, 3)
    return {"film": film, "rays": None, "tests": None}


def _camera_rays(p):
    """Pinhole rays through the pixel centres."""
    f = dict(dtype=torch.float64, device=DEVICE)
    y, x = torch.meshgrid(torch.arange(p.height, **f) + 0.5, torch.arange(p.width, **f) + 0.5, indexing="ij")
    a = p.tan_fov_x * (x - p.width / 2) / (p.width / 2)
    b = p.tan_fov_y * (p.height / 2 - y) / (p.height / 2)
    u, v, w, e = (torch.tensor(list(t), **f) for t in (p.cam_u, p.cam_v, p.cam_w, p.eye))
    d = a.reshape(-1, 1) * u + b.reshape(-1, 1) * v - w
    d = d / d.norm(dim=1, keepdim=True)
    return e.expand_as(d).contiguous(), d


def _triangles(host):
    """World vertices of the triangles with their indices; for each its
    object-space normal and M^-1 (what the parallel test looks at)."""
    a = host.arrays()
    idx = np.nonzero(a["prim_type"] == 0)[0]
    g = torch.tensor(a["prim_geom"][idx, :9].astype(np.float64), device=DEVICE).reshape(-1, 3, 3)
    tid = torch.tensor(a["prim_transform"][idx].astype(np.int64), device=DEVICE)
    xf = torch.tensor(a["transforms"].astype(np.float64), device=DEVICE)  # [T, 3, column, row]
    m = xf[:, 0].transpose(1, 2)[tid]
    world = torch.einsum("nij,nkj->nki", m[:, :3, :3], g) + m[:, None, :3, 3]
    obj_n = torch.linalg.cross(g[:, 1] - g[:, 0], g[:, 2] - g[:, 0])
    inv = xf[:, 1].transpose(1, 2)[:, :3, :3]
    return torch.tensor(idx, device=DEVICE), world, obj_n, tid, inv


def _brute_force(host, o, d, tmax):
    """Distance and index of the closest primitive with 0 < distance < tmax;
    infinity and -1 for none. A triangle is missed by rays that its
    unnormalised object-space normal calls parallel (|n . d| < 1e-4)."""
    a = host.arrays()
    n = o.shape[0]
    best = torch.full((n,), math.inf, dtype=torch.float64, device=DEVICE) if tmax is None else tmax.clone()
    who = torch.full((n,), -1, dtype=torch.int64, device=DEVICE)
    idx, tri, obj_n, tid, inv = _triangles(host)
    if len(idx):
        # per triangle the affine map to (u, v, height) coordinates
        e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
        nrm = torch.linalg.cross(e1, e2)
        to = torch.linalg.inv(torch.stack([e1, e2, nrm], dim=2))
        off = -torch.einsum("nij,nj->ni", to, tri[:, 0])
        # n_obj . (M^-1 d / |M^-1 d|) is the height rate times |n_world . e| / ... : a factor per triangle
        rate = torch.einsum("ni,nij,nj->n", obj_n, inv[tid], nrm)
        for at in range(0, n, 1 << 14):
            ro, rd = o[at:at + (1 << 14)], d[at:at + (1 << 14)]
            length = torch.einsum("tij,rj->rti", inv, rd).norm(dim=2)
            for t0 in range(0, len(idx), 4096):
                s = slice(t0, t0 + 4096)
                oz = torch.addmm(off[s, 2], ro, to[s, 2].T)
                dz = rd @ to[s, 2].T
                t = -oz / dz
                u = torch.addmm(off[s, 0], ro, to[s, 0].T).addcmul_(t, rd @ to[s, 0].T)
                v = torch.addmm(off[s, 1], ro, to[s, 1].T).addcmul_(t, rd @ to[s, 1].T)
                ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0)
                ok &= (dz * rate[s]).abs() >= 1e-4 * length[:, tid[s]]
                t.masked_fill_(~ok, math.inf)
                m, k = t.min(dim=1)
                b = best[at:at + (1 << 14)]
                closer = m < b
                best[at:at + (1 << 14)] = torch.where(closer, m, b)
                w = who[at:at + (1 << 14)]
                who[at:at + (1 << 14)] = torch.where(closer, idx[s][k], w)
    sph = np.nonzero(a["prim_type"] == 1)[0]
    if len(sph):
        g = torch.tensor(a["prim_geom"][sph, :4].astype(np.float64), device=DEVICE)
        ids = torch.tensor(sph, device=DEVICE)
        for at in range(0, n, 1 << 14):
            ro, rd = o[at:at + (1 << 14)], d[at:at + (1 << 14)]
            for s0 in range(0, len(sph), 4096):
                c, r = g[s0:s0 + 4096, :3], g[s0:s0 + 4096, 3]
                b = (ro * rd).sum(1, keepdim=True) - rd @ c.T
                cc = (ro * ro).sum(1, keepdim=True) - 2 * ro @ c.T + (c * c).sum(1) - r * r
                root = (b * b - cc).clamp(min=0).sqrt()
                t = torch.where(-b - root >= 0, -b - root, -b + root)
                t.masked_fill_((b * b < cc) | (t <= 0), math.inf)
                m, k = t.min(dim=1)
                old = best[at:at + (1 << 14)]
                closer = m < old
                best[at:at + (1 << 14)] = torch.where(closer, m, old)
                who[at:at + (1 << 14)] = torch.where(closer, ids[s0 + k], who[at:at + (1 << 14)])
    return torch.where(who >= 0, best, math.inf), who


def _normals(host, prim, pos):
    """Face normals of the triangles, radial normals of the spheres."""
    a = host.arrays()
    out = torch.zeros_like(pos)
    idx, tri, _, _, _ = _triangles(host)
    if len(idx):
        table = torch.zeros(len(a["prim_type"]), 3, dtype=torch.float64, device=DEVICE)
        n = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
        table[idx] = n / n.norm(dim=1, keepdim=True)
        out = table[prim.clamp(min=0)]
    sphere = torch.tensor(a["prim_type"] == 1, device=DEVICE)[prim.clamp(min=0)]
    g = torch.tensor(a["prim_geom"][:, :4].astype(np.float64), device=DEVICE)[prim.clamp(min=0)]
    radial = (pos - g[:, :3]) / g[:, 3:4].clamp(min=1e-300)
    return torch.where(sphere.unsqueeze(1), radial, out)
