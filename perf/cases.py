"""Performance cases: what a localisation program has this package do.

Each case is one call, or one filter step, through the public entry points, on
synthetic scenes of tsdf_localization_amd.synth (seeded; ray-cast scans and
particle sets differ from seed to seed, the maps stay, as a robot's map does):

  evaluate  the drop-in call on host arrays (weights normalised in place)
  cloud     the drop-in call on a raw PointCloud2 (x, y, z, ring)
  step      one tracking step of a device-resident filter: odometry, new scan,
            sensor update, resampling, pose and particles read back
  global    sensor update and resampling of particles over the whole map
  raw       raw weights of device-resident inputs, no allocation
  float     update on a map of general float values
  wide      update on a map of the 64-bit form (a campus of buildings)
  batch     many filters in one captured step
  serve     a burst of requests of many robots to the serving loop
  reduce    reduction of a raw scan on the device
  resample  systematic resampling of a host particle array

exact() restates the weights and the pose in double precision with torch.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import tsdf_localization_amd as tsl
from tsdf_localization_amd import _lib, evaluator, synth
from tsdf_localization_amd.server import Server

A_HIT, A_RANGE, A_MAX, MAX_RANGE, SIGMA = 0.9, 0.1, 0.0, 100.0, 0.1
BUILDING_SEED = 0x5EED0002  # the building of synth.building(): 1024 x 1024 x 128 voxels of 0.05 m, 38 % of its blocks
CAMPUS_TILES = (3, 3)
TF = synth.tf_from_xyzrpy(**synth.SCANNER_TF)


def listed():
    return [
        # the smallest filter in use: a converged pose track in one room; launches and host calls count
        {"name": "tiny", "kind": "step", "scene": "room", "particles": 257, "points": 701},
        # the reference node's own call at its usual size: 1,000 particles, a 16-beam scan reduced to 2k points
        {"name": "room", "kind": "evaluate", "scene": "room", "particles": 1000, "points": 2056},
        # the same call with the lidar's raw cloud, reduced on the device first
        {"name": "cloud", "kind": "cloud", "particles": 1000, "beams": 16, "azimuths": 1024},
        # a tracking robot in a large building (odometry step, 64-beam scan)
        {"name": "track", "kind": "step", "scene": "building", "particles": 5000, "points": 10000},
        # a raw scan of a 64-beam lidar (the reduction's most rings) reduced for the update
        {"name": "reduce", "kind": "reduce", "beams": 64, "azimuths": 4096, "points": 250001},
        # the resampler plugin on a host particle array
        {"name": "resample", "kind": "resample", "particles": 100003},
        # a map built elsewhere, with values of its own
        {"name": "float", "kind": "float", "particles": 20000, "points": 5003},
        # global localisation on a campus map, block offsets of 64 bits
        {"name": "wide", "kind": "wide", "particles": 200000, "points": 3989},
        # 64 filters of uneven sizes, one captured step
        {"name": "batch", "kind": "batch", "filters": 64, "max_particles": 50000, "max_points": 30000},
        # 48 robots' requests arriving together
        {"name": "serve", "kind": "serve", "robots": 48, "max_particles": 20000, "max_points": 20000},
        # global localisation: 100,000 particles over the free space, a 20,000-point scan
        {"name": "global", "kind": "global", "particles": 100000, "points": 20000},
        # the same with a million particles and a short scan, weights only
        {"name": "bulk", "kind": "raw", "particles": 1000000, "points": 3989},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "evaluate", "cloud", "global", "raw", "float", "wide", "batch", "serve",
                       "reduce", "resample"])
    if kind == "step":
        scene = rng.choice(["room", "building"])
        if scene == "room":
            return {"kind": kind, "scene": scene, "particles": _log(rng, 100, 3000), "points": _log(rng, 300, 2000)}
        return {"kind": kind, "scene": scene, "particles": _log(rng, 300, 30000), "points": _log(rng, 1000, 15000)}
    if kind == "evaluate":
        scene = rng.choice(["room", "building"])
        top = 2000 if scene == "room" else 15000
        return {"kind": kind, "scene": scene, "particles": _log(rng, 100, 30000), "points": _log(rng, 300, top)}
    if kind == "cloud":
        return {"kind": kind, "particles": _log(rng, 200, 10000), "beams": rng.choice([16, 32, 64]),
                "azimuths": rng.randrange(500, 1100)}
    if kind == "global":
        return {"kind": kind, "particles": _log(rng, 10000, 150000), "points": _log(rng, 2000, 13000)}
    if kind == "raw":
        return {"kind": kind, "particles": _log(rng, 1000, 900000), "points": _log(rng, 700, 4000)}
    if kind == "float":
        return {"kind": kind, "particles": _log(rng, 500, 60000), "points": _log(rng, 700, 12000)}
    if kind == "wide":
        return {"kind": kind, "particles": _log(rng, 10000, 300000), "points": _log(rng, 1500, 9000)}
    if kind == "batch":
        return {"kind": kind, "filters": _log(rng, 3, 64), "max_particles": _log(rng, 1000, 40000),
                "max_points": _log(rng, 3000, 20000)}
    if kind == "serve":
        return {"kind": kind, "robots": _log(rng, 2, 64), "max_particles": _log(rng, 2500, 20000),
                "max_points": _log(rng, 5500, 15000)}
    if kind == "reduce":
        beams, azimuths = rng.choice([16, 32, 64]), rng.randrange(700, 4097)
        return {"kind": kind, "beams": beams, "azimuths": azimuths, "points": int(beams * azimuths * 0.95)}
    return {"kind": "resample", "particles": _log(rng, 500, 800000)}


# ---- scenes ------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _building_scene():
    return synth.campus(BUILDING_SEED, tiles=(1, 1), bases=1).scenes[0]


@functools.lru_cache(maxsize=None)
def _building_map():
    return synth.building(num_particles=1).map


@functools.lru_cache(maxsize=None)
def _campus():
    return synth.campus(0x5EED0005, tiles=CAMPUS_TILES)


@functools.lru_cache(maxsize=None)
def _float_map():
    """The building with a value of its own in every voxel."""
    m = _building_map()
    lut = np.array([tsl.likelihood_value(v, SIGMA) for v in range(-299, 300)], np.float32)
    mm = m.tsdf_mm.astype(np.int32)
    hit = np.abs(mm) < m.truncation_mm
    data = np.where(hit, lut[np.where(hit, mm, 0) + 299], np.float32(m.coef().init_value))
    rng = np.random.default_rng(31)
    data *= rng.uniform(0.999, 1.001, data.shape).astype(np.float32)
    data += rng.uniform(0.0, 1e-4, data.shape).astype(np.float32)
    return tsl.CudaSubVoxelMap(m.coef(), m.grid_occ, data=data)


def _free_pose(scene, rng):
    for _ in range(1000):
        x, y = rng.uniform(2, 49.2), rng.uniform(2, 49.2)
        if scene.sdf([[x, y, 1.0]])[0] > 0.8:
            break
    return np.array([x, y, 1.0, 0.0, 0.0, rng.uniform(-math.pi, math.pi)])


def _raw_scan(seed, beams, azimuths):
    scene, rng = _building_scene(), np.random.default_rng(seed)
    pose = _free_pose(scene, rng)
    pts, rings = scene.raycast(synth.compose_pose(pose, TF), beams, azimuths, -22.5, 22.5, 60.0, 0.01, seed)
    return pose, pts, rings


def _thin(pts, points, rng):
    if pts.shape[0] > points:
        pts = pts[np.sort(rng.choice(pts.shape[0], points, replace=False))]
    return np.ascontiguousarray(pts, np.float32)


def _sizes(count, particles, points):
    """Uneven (particles, points) of `count` filters: log-uniform, uniform."""
    rng = np.random.default_rng(count)
    lo, hi = particles
    return [(int(round(lo * (max(hi, lo) / lo) ** rng.uniform())), int(rng.integers(points[0], points[1] + 1)))
            for _ in range(count)]


def _scan(seed, points):
    """A pose in the building and a reduced scan of `points` points from it."""
    for k in range(50):
        beams = 64 if points <= 10000 else 128
        pose, pts, rings = _raw_scan(seed + 1009 * k, beams, 16 * beams)
        pts, _ = synth.voxel_filter(pts, rings, 0.05, 1.0)
        if pts.shape[0] >= points:
            break
    return pose, _thin(pts, points, np.random.default_rng(seed))


def _around(seed, n, pose):
    return synth.particles_normal(seed, n, pose, [0.2, 0.2, 0.05, math.radians(5), math.radians(1), math.radians(5)])


def _inputs(case, seed):
    """Host inputs of a case on one map: (map, particles, points, tf)."""
    kind, P, N = case["kind"], case["particles"], case.get("points")
    if case.get("scene") == "room":
        w = synth.room(seed=0x5EED0001 + seed, num_particles=P)
        return w.map, w.particles, _thin(w.points, N, np.random.default_rng(seed)), w.tf
    if kind == "wide":
        cp = _campus()
        _, pts = synth.campus_scan(cp, np.random.default_rng(seed), TF, N)
        return cp.map, synth.campus_particles(cp, seed, P, math.radians(3.0)), pts, TF
    pose, pts = _scan(seed, N)
    if kind in ("global", "raw"):
        parts = _building_scene().particles_free(seed, P, (0.5, 0.5, 0.5), (50.7, 50.7, 2.0), 0.3, math.radians(3.0))
    else:
        parts = _around(seed, P, pose)
    return (_float_map() if kind == "float" else _building_map()), parts, pts, TF


def _evaluator(m):
    return tsl.TSDFEvaluator(m, False, A_HIT, A_RANGE, A_MAX, MAX_RANGE)


# ---- prepare -------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind}
    rng = np.random.default_rng(seed)
    if kind == "reduce":
        _, pts, rings = _raw_scan(seed, case["beams"], case["azimuths"])
        n = case["points"]
        st.update(points=pts[:n], rings=rings[:n].astype(np.int16), room=np.empty((n, 3), np.float32),
                  filter=tsl.DeviceFilter(_evaluator(_building_map()), 16))
        return st
    if kind == "cloud":
        pose, pts, rings = _raw_scan(seed, case["beams"], case["azimuths"])
        st.update(ev=_evaluator(_building_map()), particles=_around(seed, case["particles"], pose), points=pts,
                  rings=rings)
        return st
    if kind == "resample":
        n = case["particles"]
        p = rng.uniform(0, 50, (n, 7)).astype(np.float32)
        w = rng.gamma(4.0, 1.0, n)  # the spread of the evaluator's weights: about 0.1 to 4 times their mean
        p[:, 6] = (w / w.sum()).astype(np.float32)
        st.update(room=_room(n), sources=np.zeros(_room(n).shape[0], np.int32), particles=p, u0=np.float32(rng.uniform(0, 1.0 / n)))
        return st
    if kind == "batch":
        ev, stream, filters = _evaluator(_building_map()), tsl.Stream(), []
        sizes = _sizes(case["filters"], (500, case["max_particles"]), (2000, case["max_points"]))
        raws = [_scan(seed + 31 * k, case["max_points"]) for k in range(min(8, len(sizes)))]
        for i, (n, points) in enumerate(sizes):
            pose, pts = raws[i % len(raws)]
            f = tsl.DeviceFilter(ev, n)
            f.set_particles(_around(seed + 7 * i, n, pose))
            f.snapshot()
            f.set_scan(_thin(pts, points, rng), TF)
            filters.append(f)
        b = tsl.Batch(ev, filters)
        b.set_tile(2, 0, 1)
        b.capture(stream, restore=True)
        u0 = np.array([rng.uniform(0, 1.0 / n) for n, _ in sizes], np.float32)
        st.update(ev=ev, filters=filters, batch=b, stream=stream, u0=u0, room=_room(sum(n for n, _ in sizes)))
        return st
    if kind == "serve":
        sizes = _sizes(case["robots"], (2000, case["max_particles"]), (5000, case["max_points"]))
        raws = [_scan(seed + 31 * k, case["max_points"]) for k in range(min(4, len(sizes)))]
        sv = Server(_evaluator(_building_map()), max_robots=len(sizes), max_particles=case["max_particles"],
                    max_batch=64)
        robots = []
        for i, (n, points) in enumerate(sizes):
            pose, pts = raws[i % len(raws)]
            robot = sv.add_robot(_around(seed + 7 * i, n, pose), case["max_points"], TF)
            robots.append((robot, n, _thin(pts, points, rng)))
        st.update(server=sv, robots=robots, seed=seed, passes=0)
        return st
    m, parts, pts, tf = _inputs(case, seed)
    ev = _evaluator(m)
    n = parts.shape[0]
    st.update(ev=ev, particles=parts, points=pts, tf=tf, u0=np.float32(rng.uniform(0, 1.0 / n)))
    if kind == "raw":
        st["d_particles"] = torch.from_numpy(parts).cuda()
        st["d_points"] = torch.from_numpy(pts).cuda()
        st["weights"] = torch.empty(n, dtype=torch.float32, device="cuda")
    elif kind != "evaluate":
        st["room"] = _room(n)
        f = tsl.DeviceFilter(ev, n)
        f.set_particles(parts)
        f.snapshot()
        f.set_scan(pts, tf)
        st.update(filter=f, stream=tsl.Stream(),
                  motion=evaluator.motion_from_odom(0.5, 0.1, 0.1, a=(0.1,) * 12, seed=seed))
    return st


def _room(n):
    """Where a program keeps its particles: resampling n of them can give a few more."""
    return np.zeros((n + 64 + n // 500, 7), np.float32)


# ---- run -----------------------------------------------------------------------


def _pose(p):
    return {"position": np.array(p["position"]), "orientation": np.array(p["orientation"])}


def _into(room, rows):
    """The rows at the head of the program's own array, zeros after them."""
    room[: rows.shape[0]] = rows
    room[rows.shape[0]:] = 0
    return room


def run(st):
    kind = st["kind"]
    if kind == "evaluate":
        parts = st["particles"]
        pose = st["ev"].evaluate(parts, st["points"], st["tf"])
        return {"weights": parts[:, 6], "pose": _pose(pose)}
    if kind == "cloud":
        parts = st["particles"]
        pose = st["ev"].evaluate_cloud(parts, st["points"], st["rings"], TF)
        return {"weights": parts[:, 6], "pose": _pose(pose)}
    if kind == "step":
        f, s = st["filter"], st["stream"]
        f.restore_async(s)
        f.motion_async(st["motion"], s)
        f.set_scan(st["points"], st["tf"])
        f.update_async(s)
        f.resample_async(st["u0"], s)
        pose, n = f.sync(s)
        return {"pose": _pose(pose), "count": n, "particles": _into(st["room"], f.get_particles(n))}
    if kind == "global":
        f, s = st["filter"], st["stream"]
        f.restore_async(s)
        f.update_async(s)
        f.resample_async(st["u0"], s)
        pose, n = f.sync(s)
        return {"pose": _pose(pose), "count": n, "particles": _into(st["room"], f.get_particles(n))}
    if kind in ("float", "wide"):
        f, s = st["filter"], st["stream"]
        f.restore_async(s)
        f.update_async(s)
        pose, n = f.sync(s)
        return {"pose": _pose(pose), "weights": f.get_particles(n)[:, 6]}
    if kind == "raw":
        p, q, w = st["d_particles"], st["d_points"], st["weights"]
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        _lib.check(_lib.lib.tsl_evaluate_raw_noalloc(
            st["ev"].handle, ctypes.c_void_p(p.data_ptr()), p.shape[0], ctypes.c_void_p(q.data_ptr()), q.shape[0],
            ctypes.c_void_p(st["tf"].ctypes.data), ctypes.c_void_p(w.data_ptr()), stream))
        return {"weights": w}
    if kind == "batch":
        b, s = st["batch"], st["stream"]
        b.launch(st["u0"], s)
        poses, counts, status = b.sync(s)
        return {"position": np.array([p["position"] for p in poses]),
                "orientation": np.array([p["orientation"] for p in poses]), "counts": counts, "status": status,
                "particles": _into(st["room"], np.concatenate([f.get_particles(int(n))
                                                              for f, n in zip(st["filters"], counts)]))}
    if kind == "serve":
        sv = st["server"]
        for k, (robot, n, pts) in enumerate(st["robots"]):
            seed = (st["seed"] * 1000003 + st["passes"] * 1009 + k) & 0x7fffffff
            motion = evaluator.motion_from_odom(0.5, 0.1, 0.1, a=(0.1,) * 12, seed=seed)
            u = (seed % 65536 + 0.5) / 65536.0 / (1.05 * n)
            sv.submit(robot, motion, pts, u, request_id=k)
        st["passes"] += 1
        res = sorted(sv.wait(len(st["robots"])), key=lambda r: r["id"])
        return {"position": np.array([r["pose"]["position"] for r in res]),
                "orientation": np.array([r["pose"]["orientation"] for r in res]),
                "counts": np.array([r["count"] for r in res]), "status": np.array([r["status"] for r in res])}
    if kind == "reduce":
        f = st["filter"]
        f.set_scan_raw(st["points"], st["rings"], TF, 0.064)
        return {"points": _into(st["room"], f.get_scan())}
    new, idx = tsl.resample_systematic(st["particles"], st["u0"])
    return {"particles": _into(st["room"], new), "indices": _into(st["sources"], idx)}


# ---- work ----------------------------------------------------------------------

FLOPS_PER_PAIR = 26  # transform 18, offset 3, sub-voxel 3, score and sum 2


def _pairs(case):
    kind = case["kind"]
    if kind == "batch":
        return sum(n * p for n, p in _sizes(case["filters"], (500, case["max_particles"]), (2000, case["max_points"])))
    if kind == "serve":
        return sum(n * p for n, p in _sizes(case["robots"], (2000, case["max_particles"]), (5000, case["max_points"])))
    if kind == "cloud":
        return case["particles"] * case["beams"] * case["azimuths"] * 0.3
    return case["particles"] * case["points"]


def work(case):
    kind = case["kind"]
    if kind == "reduce":
        n = case["points"]
        return {"bytes": 14 * n + 12 * 0.2 * n, "flops": 12 * n}
    if kind == "resample":
        n = case["particles"]
        return {"bytes": (28 + 32) * n, "flops": 2 * n}
    pairs = _pairs(case)
    n = case.get("particles") or pairs / ((5000 + case["max_points"]) / 2)
    voxel = 4 if kind == "float" else 2
    voxels = {"room": 5.4e6}.get(case.get("scene"), 483.5e6 if kind == "wide" else 57.4e6)
    resampled = 28 * n if kind in ("step", "global", "batch", "serve") else 0
    return {"bytes": 28 * n + 4 * n + resampled + 12 * (case.get("points") or 5000) + min(voxel * pairs, voxel * voxels),
            "flops": FLOPS_PER_PAIR * pairs}


# ---- the same in double precision ------------------------------------------------


def _double_map(m, device):
    c = m.coef()
    if m.data is not None:
        values = torch.from_numpy(m.data).to(device)
        lut = None
    else:
        t = m.truncation_mm
        values = torch.from_numpy(m.tsdf_mm).to(device)
        d = torch.arange(-(t - 1), t, dtype=torch.float64, device=device) * 0.001
        lut = (torch.exp(-d * d / SIGMA ** 2 / 2) / math.sqrt(2 * SIGMA ** 2 * math.pi)) ** 3
    return c, torch.from_numpy(np.asarray(m.grid_occ, np.int64)).to(device), values, lut


def _double_weights(m, parts, pts, tf):
    """Sum over the points of a_hit * value + range term, in double, with the
    lookup's conversions: truncation toward zero (offsets in (-1, 0) index
    backwards from block 0) and offsets at or below -1 at sub-index 0."""
    device = "cuda" if torch.cuda.is_available() else "cpu"
    c, grid, values, lut = _double_map(m, device)
    f64 = dict(dtype=torch.float64, device=device)
    p = torch.from_numpy(parts).to(**f64)
    q = torch.from_numpy(pts).to(**f64)
    T = torch.from_numpy(np.asarray(tf).reshape(4, 4)).to(**f64)
    q1 = torch.cat([q, torch.ones_like(q[:, :1])], 1)
    sa, ca, sb, cb, sg, cg = [f(p[:, 3 + a]) for a in range(3) for f in (torch.sin, torch.cos)]
    rows = [[cb * cg, sa * sb * cg - ca * sg, ca * sb * cg + sa * sg, p[:, 0]],
            [cb * sg, sa * sb * sg + ca * cg, ca * sb * sg - sa * cg, p[:, 1]],
            [-sb, sa * cb, ca * cb, p[:, 2]]]
    L = torch.stack([torch.stack(r, 1) for r in rows], 1) @ T
    term = torch.where((q * q).sum(1) < MAX_RANGE ** 2, A_RANGE / MAX_RANGE, A_MAX).sum()
    res, sd = float(c.resolution), int(c.sub_dim)
    dims, ups = (c.dim_x, c.dim_y, c.dim_z), (1, int(c.up_dim_x), int(c.up_dim_2))
    strides = (1, sd, sd * sd)
    out = torch.empty(p.shape[0], **f64)
    step = max(1, int(2e7 // max(1, q.shape[0])))
    for a in range(0, p.shape[0], step):
        up = torch.zeros((), dtype=torch.int64, device=device)
        small, ok = up, torch.ones((), dtype=torch.bool, device=device)
        for ax, lo in enumerate((c.min_x, c.min_y, c.min_z)):
            o = L[a:a + step, ax] @ q1.T - float(lo)
            i = torch.trunc(o)
            neg = o <= -1.0
            ok = ok & (torch.floor(i / res) < dims[ax])
            if ax == 0:
                ok = ok & ~neg
            up = up + i.long() * ups[ax]
            small = small + torch.where(neg, 0.0, torch.trunc((o - i) / res)).long() * strides[ax]
        ok = ok & (up >= 0) & (up < grid.numel())
        s = grid[torch.where(ok, up, 0)]
        ok = ok & (s >= 0)
        idx = s + small
        ok = ok & (idx >= 0) & (idx < int(c.data_size))
        v = values[torch.where(ok, idx, 0)]
        if lut is not None:
            t = m.truncation_mm
            v = v.long()
            ok = ok & (v > -t) & (v < t)
            v = lut[torch.where(ok, v, 0) + t - 1]
        w = torch.where(ok, v.double(), float(c.init_value))
        out[a:a + step] = A_HIT * w.sum(1) + term
    return out


def _double_pose(parts, w):
    p = torch.from_numpy(parts).to(w)
    w = w / w.sum()
    pos = (p[:, :3] * w[:, None]).sum(0)
    r, t, y = [torch.atan2((w * torch.sin(p[:, 3 + a])).sum(), (w * torch.cos(p[:, 3 + a])).sum()).item() / 2
               for a in range(3)]
    cr, sr, cp, sp, cy, sy = math.cos(r), math.sin(r), math.cos(t), math.sin(t), math.cos(y), math.sin(y)
    q = [sr * cp * cy - cr * sp * sy, cr * sp * cy + sr * cp * sy, cr * cp * sy - sr * sp * cy,
         cr * cp * cy + sr * sp * sy]
    return {"position": pos.cpu().numpy(), "orientation": np.array(q)}


def _double_cloud(pts):
    centres = np.floor(pts.astype(np.float64) / 0.064) * 0.064 + 0.032
    return np.unique(centres.astype(np.float32), axis=0)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("reduce", "resample", "step", "batch", "serve"):
        return None  # whole points and indices, or particles moved by noise
    if kind == "cloud":
        pose, pts, _ = _raw_scan(seed, case["beams"], case["azimuths"])
        m, parts, pts, tf = _building_map(), _around(seed, case["particles"], pose), _double_cloud(pts), TF
    else:
        m, parts, pts, tf = _inputs(case, seed)
    w = _double_weights(m, parts, pts, tf)
    if kind == "raw":
        return {"weights": w.cpu().numpy()}
    pose = _double_pose(parts, w)
    if kind == "global":
        return {"pose": pose, "count": None, "particles": None}
    return {"weights": (w / w.sum()).cpu().numpy(), "pose": pose}
