"""The work a user of the library has it do, as cases that can be timed and compared.

listed() names the cases, draw() makes further ones of the same ranges, prepare() builds what a
program holds before the call (the committed scene, the ray or record buffers, the guide), run()
makes the call through the public entry points (banshee_amd.hip, or the C ABI it loads where a
caller passes device pointers), work() counts what the path cannot do without, and exact() gives
the same outputs in 64-bit arithmetic where plain torch can.

Device buffers are torch tensors handed to the C ABI by pointer. A process keeps one context and
the scenes it has loaded, as a renderer does; what a case's seed changes is the view, the sample
seed, the rays, the maps, the records and the weights.
"""
import functools
import math

import numpy as np
import torch
from ctypes import c_int, c_size_t, c_void_p

from banshee_amd import hip, scenes

# ------------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------------


def listed():
    return [
        # a picking query or a handful of visibility tests from a host loop: the call's latency
        {"name": "pick_cornell", "kind": "rays", "scene": "cornell", "tris": 34, "rays": 1000, "query": "closest",
         "pattern": "camera"},
        # a caller's own integrator (the Intersectable slot) on the full-size terrain: a wavefront of
        # incoherent secondary rays
        {"name": "closest_terrain3M", "kind": "rays", "scene": "terrain", "tris": 3084292, "rays": 2097152,
         "query": "closest", "pattern": "random"},
        # shadow rays of such an integrator in an interior, an odd count
        {"name": "any_room500k", "kind": "rays", "scene": "room", "tris": 500000, "rays": 700001, "query": "any",
         "pattern": "segments"},
        # the Cornell frame of the reference's own unit tests: 256 x 256, 16 samples, depth 5
        {"name": "frame_cornell", "kind": "frame", "scene": "cornell", "tris": 34, "width": 256, "height": 256,
         "grid": 4, "depth": 5},
        # a full production frame: 3.08M triangles at 1080p, 64 samples, depth 8
        {"name": "frame_terrain3M", "kind": "frame", "scene": "terrain", "tris": 3084292, "width": 1920,
         "height": 1080, "grid": 8, "depth": 8},
        # every light and material kind, textures and normal maps: an odd-sized preview frame
        {"name": "frame_maps", "kind": "frame", "scene": "maps", "tris": 36, "width": 637, "height": 361, "grid": 3,
         "depth": 6},
        # many small scenes at once, rendered as one captured batch (thumbnails, data generation)
        {"name": "batch_16", "kind": "batch", "jobs": 16, "max_tris": 200000, "max_res": 384, "max_grid": 4},
        # light-probe baking for a level: a 16^3 grid over 2M triangles, 1024 rays each, 9 coefficients
        {"name": "probes_4096", "kind": "probes", "tris": 2000000, "probes": 4096, "rays": 1024, "lmax": 2,
         "depth": 6},
        # image-based lighting: project a 2K environment map, then irradiance at a frame's normals
        {"name": "env_2048", "kind": "env", "width": 2048, "height": 1024, "lmax": 2, "normals": 262144},
        # guide inference on one pass's vertices
        {"name": "guide_forward", "kind": "guide", "rows": 1048576},
        # a pass's worth of online guide training: ten Adam steps on batches of 2^18 records
        {"name": "guide_train", "kind": "train", "records": 1048576, "batch": 262144, "steps": 10},
        # one guided pass of the progressive renderer, 4 samples at 1024 x 1024, writing records
        {"name": "frame_guided", "kind": "guided", "tris": 500000, "width": 1024, "height": 1024, "grid": 2,
         "depth": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "rays", "frame", "frame", "batch", "probes", "env", "guide", "train", "guided"])
    if kind == "rays":
        scene = rng.choice(["cornell", "room", "terrain", "terrain"])
        tris = 34 if scene == "cornell" else _log(rng, 20000, 500000) if scene == "room" else _log(rng, 2000, 3000000)
        return {"kind": kind, "scene": scene, "tris": tris, "rays": _log(rng, 1, 1 << 22),
                "query": rng.choice(["closest", "any"]), "pattern": rng.choice(["camera", "random", "segments"])}
    if kind == "frame":
        scene = rng.choice(["cornell", "terrain", "terrain", "maps", "materials", "open"])
        w = _log(rng, 17, 1920)
        h = max(9, int(w * rng.uniform(0.5, 1.1)))
        grid = rng.randint(1, 8)
        while w * h * grid * grid > 1 << 24:
            grid = max(1, grid - 1)
            if grid == 1:
                break
        return {"kind": kind, "scene": scene, "tris": _log(rng, 2000, 2000000) if scene == "terrain" else 34,
                "width": w, "height": h, "grid": grid, "depth": rng.randint(1, 10)}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(2, 24), "max_tris": _log(rng, 3000, 200000),
                "max_res": 16 * rng.randint(9, 24), "max_grid": rng.randint(2, 5)}
    if kind == "probes":
        return {"kind": kind, "tris": _log(rng, 2000, 2000000), "probes": _log(rng, 1, 5000),
                "rays": rng.choice([16, 64, 100, 256, 484, 1024]), "lmax": rng.randint(0, 4),
                "depth": rng.randint(1, 8)}
    if kind == "env":
        w = _log(rng, 16, 4096)
        return {"kind": kind, "width": w, "height": max(2, int(w * rng.uniform(0.4, 0.6))), "lmax": rng.randint(0, 4),
                "normals": _log(rng, 1, 1 << 20)}
    if kind == "guide":
        return {"kind": kind, "rows": _log(rng, 1, 1 << 21)}
    if kind == "train":
        batch = _log(rng, 1000, 1 << 18)
        return {"kind": kind, "records": batch * rng.randint(1, 4) + rng.randint(0, 999), "batch": batch,
                "steps": rng.randint(1, 12)}
    w = _log(rng, 48, 1024)
    return {"kind": kind, "tris": _log(rng, 20000, 500000), "width": w, "height": max(16, int(w * rng.uniform(0.5, 1))),
            "grid": rng.randint(1, 2), "depth": rng.randint(2, 8)}


# ------------------------------------------------------------------------------------------------
# what a program holds
# ------------------------------------------------------------------------------------------------


class _Buffer:
    """A torch tensor as the device buffer the library's calls take."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = c_void_p(tensor.data_ptr())
        self.shape = tuple(tensor.shape)


@functools.lru_cache(maxsize=None)
def _context():
    torch.zeros(1, device="cuda")
    return hip.Context(0)


@functools.lru_cache(maxsize=32)
def _scene(kind, tris, seed=1):
    """(scene data, committed scene) of a generator; loaded once, as a program loads its level."""
    if kind == "cornell":
        sc = scenes.cornell_box()
    elif kind == "room":
        sc = scenes.occluded_room(tris)
    elif kind == "terrain":
        sc = scenes.terrain_scene() if tris == 3084292 else scenes.terrain_for_tris(tris, seed)
    elif kind == "maps":
        sc = scenes.normal_mapped_cornell()
    elif kind == "materials":
        sc = scenes.material_scene()
    else:
        sc = scenes.open_scene(scenes.ENV_LIGHT_IS)
    return sc, hip.Scene(_context(), sc)


def _view(sc, seed, width, height):
    """The scene's camera with its eye moved by up to 2 % of the distance to its target."""
    r = np.random.default_rng(seed)
    cam = np.array(sc.camera, np.float64)
    cam[0:3] += r.uniform(-0.02, 0.02, 3) * np.linalg.norm(cam[3:6] - cam[0:3])
    cam[12] = width / height
    return cam


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _unit(n, g):
    d = torch.randn(n, 3, device="cuda", generator=g, dtype=torch.float64)
    return d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _rays(case, sc, seed):
    """[n, 8] rays (origin, tmin, direction, tmax) in the scene's box."""
    n, g = case["rays"], _gen(seed)
    lo = torch.tensor(sc.verts.min(0), device="cuda", dtype=torch.float64)
    hi = torch.tensor(sc.verts.max(0), device="cuda", dtype=torch.float64)

    def inside():
        return lo + (hi - lo) * (0.02 + 0.96 * torch.rand(n, 3, device="cuda", generator=g, dtype=torch.float64))

    tmax = torch.full((n, 1), 1e6, device="cuda", dtype=torch.float64)
    if case["pattern"] == "camera":
        cam = _view(sc, seed, 1, 1)
        eye, at, up = (torch.tensor(cam[k:k + 3], device="cuda") for k in (0, 3, 6))
        f = (at - eye) / (at - eye).norm()
        r = torch.linalg.cross(f, up)
        r = r / r.norm()
        u = torch.linalg.cross(r, f)
        side = max(1, math.isqrt(n - 1) + 1)
        k = torch.arange(n, device="cuda")
        s = math.tan(cam[11] / 2)
        jit = torch.rand(n, 2, device="cuda", generator=g, dtype=torch.float64)
        x = (2 * ((k % side) + jit[:, 0]) / side - 1) * s
        y = (2 * ((k // side) + jit[:, 1]) / side - 1) * s
        d = f + x[:, None] * r + y[:, None] * u
        d = d / d.norm(dim=1, keepdim=True)
        o = eye.expand(n, 3)
    elif case["pattern"] == "random":
        o, d = inside(), _unit(n, g)
    else:
        o = inside()
        d = inside() - o
        tmax = d.norm(dim=1, keepdim=True)
        d = d / tmax.clamp_min(1e-12)
        tmax = tmax - 0.01
    tmin = torch.full((n, 1), 0.01, device="cuda", dtype=torch.float64)
    return torch.cat([o, tmin, d, tmax], 1).float().contiguous()


def _net(seed):
    """A guide's parameters (He-uniform weights, small biases; rows of unused features zero) and
    the Adam moments of a run in progress, from the seed."""
    r = np.random.default_rng(seed)
    parts = []
    for k, n in _LAYERS:
        w = r.uniform(-1, 1, (k, n)) * math.sqrt(6.0 / k)
        if k == 96:
            w[[63, 78, 79, 94, 95]] = 0.0
        parts += [w.ravel(), r.uniform(-0.05, 0.05, n)]
    p = np.concatenate(parts).astype(np.float32)
    m1 = (r.normal(size=p.size) * 1e-3).astype(np.float32)
    m2 = np.exp(r.uniform(math.log(1e-6), math.log(1e-4), p.size)).astype(np.float32)
    return p, m1, m2


_LAYERS = [(96, 64), (64, 64), (64, 64), (64, 64), (64, 48)]
_STEP0 = 200
_LR, _B1, _B2, _EPS = 5e-3, 0.9, 0.99, 1e-8


def _guide(seed):
    g = hip.Guide(_context(), seed=1, lr=_LR, beta1=_B1, beta2=_B2, eps=_EPS, bsdf_fraction=0.5)
    p, m1, m2 = _net(seed)
    g.set_state({"params": p, "m1": m1, "m2": m2, "step": _STEP0})
    return g


def _vertices(n, seed):
    """[n, 8] network inputs: position in the unit box, roughness (1 on diffuse surfaces), normal."""
    g = _gen(seed)
    x = torch.zeros(n, 8, device="cuda")
    x[:, 0:3] = torch.rand(n, 3, device="cuda", generator=g)
    rough = torch.rand(n, device="cuda", generator=g)
    diffuse = torch.rand(n, device="cuda", generator=g) < 0.6
    x[:, 3] = torch.where(diffuse, torch.ones_like(rough), 0.1 + 0.5 * rough)
    x[:, 4:7] = _unit(n, g).float()
    return x


def _records(n, seed):
    """[n, 12] training records: a vertex, a sampled direction and its heavy-tailed weight."""
    g = _gen(seed + 17)
    rec = torch.zeros(n, 12, device="cuda")
    rec[:, 0:7] = _vertices(n, seed)[:, 0:7]
    rec[:, 7] = 1.0
    rec[:, 8:11] = _unit(n, g).float()
    rec[:, 11] = torch.exp(torch.randn(n, device="cuda", generator=g))
    return rec


def _batch_cfgs(case):
    return scenes.batch_jobs(n=case["jobs"], seed=100, max_tris=case["max_tris"], max_res=case["max_res"],
                             max_grid=case["max_grid"])


def prepare(case, seed):
    kind, ctx = case["kind"], _context()
    if kind == "rays":
        sc, s = _scene(case["scene"], case["tris"])
        n = case["rays"]
        rays = _rays(case, sc, seed)
        out = torch.zeros((n, 4) if case["query"] == "closest" else (n,), device="cuda",
                          dtype=torch.float32 if case["query"] == "closest" else torch.int32)
        return {"case": case, "scene": s, "rays": _Buffer(rays), "out": _Buffer(out)}
    if kind == "frame":
        sc, s = _scene(case["scene"], case["tris"])
        acc = torch.zeros(case["height"], case["width"], 8, device="cuda")
        return {"case": case, "scene": s, "accum": _Buffer(acc), "seed": seed,
                "camera": _view(sc, seed, case["width"], case["height"])}
    if kind == "batch":
        jobs, accs = [], []
        for c in _batch_cfgs(case):
            sc, s = _scene("terrain", c["tris"], c["seed"])
            job = hip.BatchJob(s, "render", width=c["res"], height=c["res"], img_grid=c["grid"],
                               max_depth=c["depth"], seed=seed + c["seed"])
            job.accum = _Buffer(torch.zeros(c["res"], c["res"], 8, device="cuda"))
            jobs.append(job)
            accs.append(job.accum.tensor)
        return {"case": case, "jobs": jobs, "accums": accs}
    if kind == "probes":
        sc, s = _scene("terrain", case["tris"])
        side = max(1, math.ceil(case["probes"] ** (1 / 3)))
        p = scenes.probe_grid(sc, side)
        r = np.random.default_rng(seed)
        p = (p + r.uniform(0, 0.05, p.shape))[:case["probes"]].astype(np.float32)
        co = torch.zeros(p.shape[0], (case["lmax"] + 1) ** 2, 3, device="cuda")
        return {"case": case, "scene": s, "probes": p, "coeffs": _Buffer(co), "seed": seed}
    if kind == "env":
        g = _gen(seed)
        h, w = case["height"], case["width"]
        env = torch.from_numpy(scenes.env_map(w, h, seed=seed % 1000)).to("cuda")
        nrm = _unit(case["normals"], g).float().contiguous()
        return {"case": case, "env": env, "normals": nrm,
                "coeffs": torch.zeros((case["lmax"] + 1) ** 2, 3, device="cuda"),
                "irradiance": torch.zeros(case["normals"], 3, device="cuda")}
    if kind == "guide":
        x = _vertices(case["rows"], seed)
        return {"case": case, "guide": _guide(seed), "x": x, "out": torch.zeros(case["rows"], 48, device="cuda")}
    if kind == "train":
        return {"case": case, "guide": _guide(seed), "records": _Buffer(_records(case["records"], seed))}
    sc, s = _scene("room", case["tris"])
    w, h = case["width"], case["height"]
    cap = w * h * case["grid"] ** 2 * 4
    return {"case": case, "scene": s, "guide": _guide(seed), "seed": seed, "camera": _view(sc, seed, w, h),
            "accum": _Buffer(torch.zeros(h, w, 8, device="cuda")),
            "records": _Buffer(torch.zeros(cap, hip.RECORD_FLOATS, device="cuda"))}


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------


def _call(name, *args):
    if getattr(hip.lib(), name)(*args) != 0:
        raise hip.BshError(hip.lib().bsh_last_error().decode())


def _ptr(t):
    return c_void_p(t.data_ptr())


def run(state):
    case = state["case"]
    kind, ctx = case["kind"], _context()
    if kind == "rays":
        n, out = case["rays"], state["out"]
        if case["query"] == "any":
            state["scene"].intersect_any_dev(state["rays"], n, out)
            return {"occluded": out.tensor}
        state["scene"].intersect_closest_dev(state["rays"], n, out)
        return {"prim": out.tensor.view(torch.int32)[:, 0], "hit": out.tensor[:, 1:]}
    if kind == "frame":
        s = state["scene"]
        s.set_camera(state["camera"])
        s.render(case["width"], case["height"], case["grid"], case["depth"], state["seed"], accum=state["accum"],
                 download=False)
        return {"accum": state["accum"].tensor}
    if kind == "batch":
        ctx.batch_run(state["jobs"], tuning={"use_graph": 1})
        return state["accums"]
    if kind == "probes":
        state["scene"].bake_sh(state["probes"], case["rays"], case["lmax"], case["depth"], state["seed"],
                               coeffs=state["coeffs"], download=False)
        return {"coeffs": state["coeffs"].tensor}
    if kind == "env":
        lmax = c_int(case["lmax"])
        _call("bsh_sh_project_env", ctx.h, _ptr(state["env"]), c_int(case["width"]), c_int(case["height"]), lmax,
              _ptr(state["coeffs"]), c_void_p(None))
        _call("bsh_sh_irradiance", ctx.h, lmax, _ptr(state["coeffs"]), _ptr(state["normals"]),
              c_size_t(case["normals"]), _ptr(state["irradiance"]), c_void_p(None))
        return {"coeffs": state["coeffs"], "irradiance": state["irradiance"]}
    if kind == "guide":
        _call("bsh_guide_forward", state["guide"].h, _ptr(state["x"]), c_size_t(case["rows"]), _ptr(state["out"]),
              c_void_p(None))
        return {"out": state["out"]}
    if kind == "train":
        state["guide"].train(state["records"], case["records"], case["steps"], case["batch"])
        return {"params": state["guide"].get_params()}
    s = state["scene"]
    s.set_camera(state["camera"])
    n = s.render_guided(case["width"], case["height"], case["grid"], case["depth"], state["seed"],
                        guide=state["guide"], accum=state["accum"], records=state["records"], download=False)
    return {"accum": state["accum"].tensor, "count": n, "records": state["records"].tensor}


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------


def _ray_flops(tris):
    """Box and triangle tests of one ray: about one 4-wide visit (4 boxes, 12 operations each) and a
    third of a triangle test per halving of the scene."""
    return 60.0 * max(2.0, math.log2(tris))


def _tree_bytes(tris):
    """Triangles (48 B) and 4-wide nodes (64 B for about 3.5 triangles), read once."""
    return tris * (48 + 64 / 3.5)


def work(case):
    kind = case["kind"]
    if kind == "rays":
        return {"bytes": case["rays"] * (36 if case["query"] == "any" else 48) + min(_tree_bytes(case["tris"]),
                                                                                     case["rays"] * 1800.0),
                "flops": case["rays"] * _ray_flops(case["tris"])}
    if kind in ("frame", "guided"):
        samples = case["width"] * case["height"] * case["grid"] ** 2
        rays = samples * (1 + min(case["depth"], 5) * 1.2)
        out = case["width"] * case["height"] * 32
        w = {"bytes": out + _tree_bytes(case["tris"]), "flops": rays * (_ray_flops(case["tris"]) + 400)}
        if kind == "guided":
            w["bytes"] += samples * 2 * 48
            w["flops"] += samples * min(case["depth"], 4) * 0.7 * 43008
        return w
    if kind == "batch":
        b = f = 0.0
        for c in _batch_cfgs(case):
            samples = c["res"] ** 2 * c["grid"] ** 2
            b += c["res"] ** 2 * 32 + _tree_bytes(c["tris"])
            f += samples * (1 + min(c["depth"], 5) * 1.2) * (_ray_flops(c["tris"]) + 400)
        return {"bytes": b, "flops": f}
    if kind == "probes":
        nt = (case["lmax"] + 1) ** 2
        samples = case["probes"] * case["rays"]
        return {"bytes": case["probes"] * 12 * (1 + nt) + min(_tree_bytes(case["tris"]), samples * 1800.0),
                "flops": samples * ((1 + min(case["depth"], 4)) * (_ray_flops(case["tris"]) + 400) + 10 * nt)}
    if kind == "env":
        nt = (case["lmax"] + 1) ** 2
        texels = case["width"] * case["height"]
        return {"bytes": texels * 12 + case["normals"] * 24 + nt * 12,
                "flops": (texels + case["normals"]) * (10.0 * nt + 20)}
    if kind == "guide":
        return {"bytes": case["rows"] * (32 + 192) + 43616, "flops": case["rows"] * 43008.0}
    n, stride = case["records"], max(1, case["records"] // case["batch"])
    rows = sum(min(case["batch"], (n - s % stride + stride - 1) // stride) for s in range(case["steps"]))
    return {"bytes": rows * 48 + case["steps"] * 21808 * 24, "flops": rows * 116736.0}


# ------------------------------------------------------------------------------------------------
# the same in 64 bits
# ------------------------------------------------------------------------------------------------


def _exact_rays(case, seed):
    sc = _scene_data(case)
    rays = _rays(case, sc, seed).double()
    tri = torch.tensor(sc.verts[sc.tri_v], device="cuda", dtype=torch.float64)
    p1, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    out = torch.zeros(rays.shape[0], 3, device="cuda", dtype=torch.float64)
    step = max(1, (1 << 24) // tri.shape[0])
    for k in range(0, rays.shape[0], step):
        o, tmin, d, tmax = (rays[k:k + step, a:b] for a, b in ((0, 3), (3, 4), (4, 7), (7, 8)))
        s1 = torch.linalg.cross(d[:, None].expand(-1, tri.shape[0], 3), e2[None].expand(d.shape[0], -1, 3))
        inv = 1.0 / (s1 * e1).sum(-1)
        dd = o[:, None] - p1
        b1 = (dd * s1).sum(-1) * inv
        s2 = torch.linalg.cross(dd, e1[None].expand_as(dd))
        b2 = (d[:, None] * s2).sum(-1) * inv
        t = (e2 * s2).sum(-1) * inv
        ok = (b1 >= 0) & (b1 <= 1) & (b2 >= 0) & (b1 + b2 <= 1) & (t > tmin) & (t <= tmax)
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, at = t.min(1)
        hit = torch.isfinite(best)
        v = torch.stack([best, b1.gather(1, at[:, None])[:, 0], b2.gather(1, at[:, None])[:, 0]], 1)
        out[k:k + step] = torch.where(hit[:, None], v, torch.zeros_like(v))
    return {"prim": None, "hit": out}


def _scene_data(case):
    return scenes.cornell_box() if case["scene"] == "cornell" else None


def _sh(w, lmax):
    """Real SH of unit directions [n, 3] (z the pole, Condon-Shortley phase, index l l + l + m)."""
    x, y, z = w[:, 0], w[:, 1], w[:, 2]
    r = torch.sqrt((1 - z * z).clamp_min(0))
    safe = r.clamp_min(1e-300)
    phi_c, phi_s = torch.where(r > 0, x / safe, torch.ones_like(x)), torch.where(r > 0, y / safe, torch.zeros_like(y))
    phi = torch.atan2(phi_s, phi_c)
    P = {(0, 0): torch.ones_like(z)}
    for m in range(1, lmax + 1):
        P[(m, m)] = -(2 * m - 1) * r * P[(m - 1, m - 1)]
    for m in range(0, lmax):
        P[(m + 1, m)] = (2 * m + 1) * z * P[(m, m)]
    for m in range(0, lmax + 1):
        for lev in range(m + 2, lmax + 1):
            P[(lev, m)] = ((2 * lev - 1) * z * P[(lev - 1, m)] - (lev + m - 1) * P[(lev - 2, m)]) / (lev - m)
    out = []
    for lev in range(lmax + 1):
        for m in range(-lev, lev + 1):
            k = math.sqrt((2 * lev + 1) / (4 * math.pi) * math.factorial(lev - abs(m)) / math.factorial(lev + abs(m)))
            v = k * P[(lev, abs(m))]
            if m > 0:
                v = v * math.sqrt(2) * torch.cos(m * phi)
            elif m < 0:
                v = v * math.sqrt(2) * torch.sin(-m * phi)
            out.append(v)
    return torch.stack(out, 1)


def _exact_env(case, seed):
    h, w, lmax = case["height"], case["width"], case["lmax"]
    env = torch.from_numpy(scenes.env_map(w, h, seed=seed % 1000)).to("cuda").double()
    th = math.pi / h * (torch.arange(h, device="cuda", dtype=torch.float64) + 0.5)
    ph = 2 * math.pi / w * (torch.arange(w, device="cuda", dtype=torch.float64) + 0.5)
    # the texel a cell reads is floor(k / n * n) in binary32, as the projection defines it
    at = [torch.floor(torch.arange(n, dtype=torch.float32) / n * n).long().to("cuda") for n in (w, h)]
    env = env[at[1]][:, at[0]]
    c = torch.zeros((lmax + 1) ** 2, 3, device="cuda", dtype=torch.float64)
    rows = max(1, (1 << 21) // w)
    for k in range(0, h, rows):
        t, p = torch.meshgrid(th[k:k + rows], ph, indexing="ij")
        d = torch.stack([torch.sin(t) * torch.cos(p), torch.cos(t), torch.sin(t) * torch.sin(p)], -1).reshape(-1, 3)
        wt = (torch.sin(t) * (math.pi / h) * (2 * math.pi / w)).reshape(-1, 1)
        c += (_sh(d, lmax) * wt).T @ env[k:k + rows].reshape(-1, 3)
    conv = [0.8862268925, 1.0233267546, 0.4954159260, 0.0, -0.1107783690]
    scale = torch.cat([torch.full((2 * lev + 1,), conv[lev] * math.sqrt(4 * math.pi / (2 * lev + 1)) * 0.7 / math.pi)
                       for lev in range(lmax + 1)]).to("cuda").double()
    nrm = _unit(case["normals"], _gen(seed)).float().double()
    return {"coeffs": c, "irradiance": _sh(nrm, lmax) @ (c * scale[:, None])}


def _encode(v):
    """[n, 7] raw inputs -> [n, 96]: per band b the sine and cosine of 2^b pi v, then two raw values."""
    blocks = []
    for b in range(6):
        a = v * (math.pi * 2 ** b)
        blocks.append(torch.stack([torch.sin(a), torch.cos(a)], -1).reshape(-1, 14))
        for k in (2 * b, 2 * b + 1):
            blocks.append(v[:, k:k + 1] if k < 7 else torch.zeros_like(v[:, :1]))
    return torch.cat(blocks, 1)


def _unpack(p):
    at, out = 0, []
    for k, n in _LAYERS:
        out.append((p[at:at + k * n].view(k, n), p[at + k * n:at + k * n + n]))
        at += k * n + n
    return out


def _forward(p, v):
    x = _encode(v)
    layers = _unpack(p)
    for k, (w, b) in enumerate(layers):
        x = x @ w + b
        if k + 1 < len(layers):
            x = torch.relu(x)
    return x


def _exact_guide(case, seed):
    p = torch.from_numpy(_net(seed)[0]).to("cuda").double()
    x = _vertices(case["rows"], seed)[:, :7].double()
    return {"out": torch.cat([_forward(p, x[k:k + (1 << 18)]) for k in range(0, x.shape[0], 1 << 18)])}


def _exact_train(case, seed):
    p, m1, m2 = (torch.from_numpy(a).to("cuda").double() for a in _net(seed))
    recs = _records(case["records"], seed).double()
    n, stride = case["records"], max(1, case["records"] // case["batch"])
    for s in range(case["steps"]):
        rec = recs[s % stride::stride][:case["batch"]]
        rows = rec.shape[0]
        wt = (rec[:, 11] * (rows / rec[:, 11].sum())).clamp_max(256.0)
        grad = torch.zeros_like(p)
        for k in range(0, rows, 1 << 16):
            q = p.clone().requires_grad_(True)
            o = _forward(q, rec[k:k + (1 << 16), 0:7])
            mu = torch.nn.functional.normalize(o[:, 8:32].reshape(-1, 8, 3), dim=-1)
            kap = torch.exp(o[:, 32:40].clamp(-2.0, 6.0))
            cosw = (mu * rec[k:k + (1 << 16), None, 8:11]).sum(-1)
            logv = torch.log(kap / (2 * math.pi * -torch.expm1(-2 * kap))) + kap * (cosw - 1)
            logq = torch.logsumexp(torch.log_softmax(o[:, 0:8], 1) + logv, 1)
            (-(wt[k:k + (1 << 16)] * logq).sum() / rows).backward()
            grad += q.grad
        m1 = _B1 * m1 + (1 - _B1) * grad
        m2 = _B2 * m2 + (1 - _B2) * grad * grad
        t = _STEP0 + s + 1
        p = p - _LR * (m1 / (1 - _B1 ** t)) / (torch.sqrt(m2 / (1 - _B2 ** t)) + _EPS)
    return {"params": p}


def exact(case, seed):
    kind = case["kind"]
    if kind == "rays" and case["scene"] == "cornell" and case["query"] == "closest":
        return _exact_rays(case, seed)
    if kind == "env":
        return _exact_env(case, seed)
    if kind == "guide":
        return _exact_guide(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    # path-traced images, and hits in large scenes, have no value that plain torch gives in seconds
    return None
