"""Performance cases: what programs on this library have it do.

Every case goes through the public entry points
(latticeboltzmanncuda_amd.capi, the binding of include/lbm.h) and ends with
the read-back that its user needs, on the host.  Kinds of case:

flow       one standard-mode lattice: n steps, then density and velocity
batch      many lattices stepped together: n steps in chunks, then the
           moments of every member
serve      solve requests through the continuous-batching server, velocity
           fields kept
reference  the reference's D3Q27 main loop around an obstacle with the force
           on; "points" cases bring the state in and out as the reference's
           144-byte records, as its load_data / retrieve_data do
geometry   voxelisation of a closed mesh and its reflection tables

The 64-bit values of exact() come from plain torch / numpy code below, which
uses nothing of this repository.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from latticeboltzmanncuda_amd import capi

STORAGE = {"f32": capi.STORE_F32, "f64": capi.STORE_F64,
           "f16": capi.STORE_F16, "bf16": capi.STORE_BF16}
BYTES = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2}
# arithmetic of one node update (moments, equilibria, relaxation)
FLOPS = {9: 140, 19: 300, 27: 420}


def listed():
    return [
        # the smallest lattices that the test configurations run: launches
        # and latency count
        {"name": "cavity2d_128_f32", "kind": "flow", "q": 9, "storage": "f32",
         "bc": "cavity", "nx": 128, "ny": 128, "nz": 1, "solid": 0.0,
         "steps": 1000},
        {"name": "cavity3d_32_f32", "kind": "flow", "q": 19, "storage": "f32",
         "bc": "cavity", "nx": 32, "ny": 32, "nz": 32, "solid": 0.0,
         "steps": 1000},
        # the benchmark's channel through random spheres
        {"name": "channel3d_f32", "kind": "flow", "q": 19, "storage": "f32",
         "bc": "channel", "nx": 256, "ny": 128, "nz": 128, "solid": 0.2,
         "force": 1e-6, "steps": 1000},
        # the same flow on extents that fit no tile, in full precision
        {"name": "channel3d_odd_f64", "kind": "flow", "q": 19,
         "storage": "f64", "bc": "channel", "nx": 121, "ny": 67, "nz": 93,
         "solid": 0.1, "force": 1e-6, "steps": 500},
        # the precision study's vortex, stored in 16 bits
        {"name": "vortex3d_256_f16", "kind": "flow", "q": 19,
         "storage": "f16", "bc": "vortex", "nx": 256, "ny": 256, "nz": 256,
         "solid": 0.0, "steps": 800},
        # one large 2-D lattice streamed from memory, body force (rounds
        # stochastically)
        {"name": "channel2d_4096_f16", "kind": "flow", "q": 9,
         "storage": "f16", "bc": "channel", "nx": 4096, "ny": 4096, "nz": 1,
         "solid": 0.1, "force": 1e-6, "steps": 1000},
        # many 2-D lattices of 32 to 512 nodes a side in one batch
        {"name": "batch2d_f32", "kind": "batch", "mix": "2d",
         "storage": "f32", "count": 256, "lo": 32, "hi": 512, "steps": 500,
         "chunk": 100},
        {"name": "batch2d_f16", "kind": "batch", "mix": "2d",
         "storage": "f16", "count": 256, "lo": 32, "hi": 512, "steps": 500,
         "chunk": 100},
        # a burst of solve requests, half 2-D, half 3-D
        {"name": "serve_mixed_f16", "kind": "serve", "storage": "f16",
         "count": 16, "lo2": 64, "hi2": 512, "lo3": 32, "hi3": 80,
         "steps": 1000, "chunk": 100},
        # the reference's main loop: a small ragged lattice with its records
        # brought in and out, and a large one
        {"name": "reference_points_32", "kind": "reference", "nx": 33,
         "ny": 32, "nz": 31, "radius": 0.2, "steps": 100, "points": True},
        {"name": "reference_128", "kind": "reference", "nx": 128, "ny": 128,
         "nz": 128, "radius": 0.2, "steps": 300, "points": False},
        # setting the obstacle up from a mesh
        {"name": "geometry_96", "kind": "geometry", "nx": 96, "ny": 96,
         "nz": 96, "rings": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "batch", "serve", "reference",
                       "geometry"])
    if kind == "flow":
        q = rng.choice([9, 9, 19, 19, 27])
        storage = rng.choice(["f32", "f32", "f64", "f16", "bf16"])
        bc = rng.choice(["cavity", "channel", "vortex"])
        if q == 9:
            nx, ny, nz = _log_int(rng, 64, 3000), _log_int(rng, 64, 3000), 1
        else:
            nx, ny, nz = (_log_int(rng, 24, 200) for _ in range(3))
        if rng.random() < 0.3:  # whole tiles along the fastest axis
            if q == 9:
                ny = max(64, ny // 64 * 64)
            else:
                nz = max(64, nz // 64 * 64)
        solid = rng.choice([0.0, 0.1, 0.2]) if bc == "channel" else 0.0
        cost = nx * ny * nz * q * BYTES[storage]
        steps = max(50, min(1000, int(2e10 / cost)))
        # a force whose channel would settle at a speed of 0.1
        wide = ny if q == 9 else min(ny, nz)
        return {"kind": kind, "q": q, "storage": storage, "bc": bc, "nx": nx,
                "ny": ny, "nz": nz, "solid": solid, "steps": steps,
                "force": min(1e-6, 0.08 / wide ** 2)}
    if kind == "batch":
        mix = rng.choice(["2d", "2d", "mixed", "3d"])
        hi = rng.randint(100, 512) if mix == "2d" else rng.randint(40, 80)
        return {"kind": kind, "mix": mix,
                "storage": rng.choice(["f32", "f16", "f16", "bf16", "f64"]),
                "count": _log_int(rng, 8, 200 if mix == "2d" else 40),
                "lo": rng.randint(20, 36), "hi": hi,
                "steps": rng.choice([100, 250, 500]),
                "chunk": rng.choice([50, 100])}
    if kind == "serve":
        return {"kind": kind, "storage": rng.choice(["f16", "f16", "f32"]),
                "count": _log_int(rng, 4, 16), "lo2": 64,
                "hi2": rng.randint(128, 512), "lo3": 32,
                "hi3": rng.randint(40, 80), "steps": rng.choice([300, 600]),
                "chunk": 100}
    if kind == "reference":
        n = [_log_int(rng, 20, 140) for _ in range(3)]
        if rng.random() < 0.4:
            n[2] = 64 if n[2] < 100 else 128
        steps = max(20, min(200, int(4e8 / (n[0] * n[1] * n[2]))))
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2],
                "radius": rng.uniform(0.12, 0.3), "steps": steps,
                "points": rng.random() < 0.5}
    return {"kind": kind, "nx": rng.randint(32, 96), "ny": rng.randint(32, 96),
            "nz": rng.randint(32, 96), "rings": rng.randint(4, 20)}


# ------------------------------------------------------------------ inputs
def _spheres(dims, frac, rng):
    """Solid map of random spheres (radius 4 to 8 nodes, smaller in small
    boxes; periodic along x) up to a fraction of the nodes."""
    solid = np.zeros(dims, np.uint8)
    top = max(2.0, min(8.0, min(dims) / 6.0))
    total = 0
    target = frac * solid.size
    while total < target:
        c = rng.random(3) * dims
        r = rng.uniform(top / 2.0, top)
        lo = np.floor(c - r).astype(int)
        hi = np.ceil(c + r).astype(int)
        x = np.arange(lo[0], hi[0] + 1)
        y = np.arange(max(lo[1], 0), min(hi[1] + 1, dims[1]))
        z = np.arange(max(lo[2], 0), min(hi[2] + 1, dims[2]))
        d2 = ((x - c[0]) ** 2)[:, None, None] + \
            ((y - c[1]) ** 2)[None, :, None] + ((z - c[2]) ** 2)[None, None, :]
        at = np.ix_(x % dims[0], y, z)
        old = solid[at]
        new = old | (d2 <= r * r)
        total += int(new.sum()) - int(old.sum())
        solid[at] = new
    return solid.reshape(-1)


def _squares(nx, ny, frac, rng, clear_top=0):
    """Solid map of random squares (side up to an eighth of the lattice, at
    most 64) up to a fraction of the nodes; the rows below a lid stay
    fluid."""
    solid = np.zeros((nx, ny), np.uint8)
    smax = max(2, min(64, min(nx, ny) // 8))
    total = 0
    while total < frac * solid.size:
        s = int(rng.integers(2, smax + 1))
        x0 = int(rng.integers(0, max(1, nx - s + 1)))
        y0 = int(rng.integers(0, max(1, ny - clear_top - s + 1)))
        box = solid[x0:x0 + s, y0:y0 + s]
        total += box.size - int(box.sum())
        box[:] = 1
    return solid.reshape(-1)


def _lattice(q, dims, tau, periodic=(0, 0, 0), lid_face=-1, lid_u=0.0,
             force=0.0, solid=None, rho=None, u=None):
    """A lattice's physics, its numbers rounded to the floats that the
    configuration holds."""
    return {"q": q, "dims": tuple(dims), "tau": float(np.float32(tau)),
            "periodic": periodic, "lid_face": lid_face,
            "lid_u": float(np.float32(lid_u)),
            "force": float(np.float32(force)), "solid": solid, "rho": rho,
            "u": u}


def _config(lat, storage):
    return capi.make_config(*lat["dims"], lattice=lat["q"],
                            storage=STORAGE[storage], tau=lat["tau"],
                            periodic=lat["periodic"],
                            lid_face=lat["lid_face"],
                            lid_u=(lat["lid_u"], 0, 0),
                            force=(lat["force"], 0, 0))


def _flow(case, seed):
    rng = np.random.default_rng(seed)
    dims = (case["nx"], case["ny"], case["nz"])
    jitter = 1.0 + 0.02 * rng.random()
    if case["bc"] == "cavity":
        return _lattice(case["q"], dims, 0.6 * jitter, lid_face=3,
                        lid_u=0.1 * (0.8 + 0.2 * rng.random()))
    if case["bc"] == "channel":
        solid = None
        if case["solid"] > 0:
            solid = (_squares(dims[0], dims[1], case["solid"], rng)
                     if case["q"] == 9 else _spheres(dims, case["solid"], rng))
        return _lattice(case["q"], dims, 0.8 * jitter, periodic=(1, 0, 0),
                        force=case["force"] * (0.8 + 0.2 * rng.random()),
                        solid=solid)
    # Taylor-Green vortex along x and y, shifted by the seed
    nx, ny, nz = dims
    u0 = 0.05 * (0.8 + 0.2 * rng.random())
    kx, ky = 2.0 * math.pi / nx, 2.0 * math.pi / ny
    x = kx * (np.arange(nx) + nx * rng.random())
    y = ky * (np.arange(ny) + ny * rng.random())
    u = np.zeros((3, nx, ny, nz))
    k = max(kx, ky)
    u[0] = (u0 * (ky / k) * np.sin(x)[:, None] * np.cos(y))[:, :, None]
    u[1] = (-u0 * (kx / k) * np.cos(x)[:, None] * np.sin(y))[:, :, None]
    rho = np.empty(dims)
    rho[:] = (1.0 - 0.75 * u0 * u0 * (np.cos(2 * x)[:, None] +
                                      np.cos(2 * y)))[:, :, None]
    return _lattice(case["q"], dims, 0.55 * jitter, periodic=(1, 1, 1),
                    rho=rho.reshape(-1), u=u.reshape(3, -1))


def _members(case, seed):
    """Lattices of a batch: cavities and channels of Reynolds number 100 to
    1000 at speed 0.1, 10 % squares (2-D) or spheres (3-D); a cell Reynolds
    number above 15 is drawn again with a larger viscosity.  Their shapes
    belong to the case, the rest to the seed."""
    shape = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    rng = np.random.default_rng(seed)
    out = []
    for k in range(case["count"]):
        two = case["mix"] == "2d" or (case["mix"] == "mixed" and k % 2 == 0)
        n = np.exp(shape.uniform(math.log(case["lo"]), math.log(case["hi"]),
                                 3)).round().astype(int)
        dims = (int(n[0]), int(n[1]), 1 if two else int(n[2]))
        q = 9 if two else 19
        cavity = bool(shape.random() < 0.5)
        L = dims[0] if cavity else dims[1]
        tau = max(0.52, 0.5 + 3.0 * 0.1 * L / rng.uniform(100.0, 1000.0))
        clear = 2 if cavity else 0
        if two:
            solid = _squares(dims[0], dims[1], 0.1, rng, clear)
        else:
            solid = _spheres(dims, 0.1, rng)
            if cavity:
                solid = solid.reshape(dims)
                solid[:, -clear:, :] = 0
                solid = np.ascontiguousarray(solid).reshape(-1)
        if cavity:
            out.append(_lattice(q, dims, tau, lid_face=3, lid_u=0.1,
                                solid=solid))
        else:
            nu = (tau - 0.5) / 3.0
            out.append(_lattice(q, dims, tau, periodic=(1, 0, 0),
                                force=8.0 * nu * 0.1 / dims[1] ** 2,
                                solid=solid))
    return out


def _requests(case, seed):
    """Body-force channels, half squares in 2-D, half spheres in 3-D, 5 to
    25 % solid.  Their extents belong to the case, the rest to the seed."""
    shape = np.random.default_rng([case["count"], case["hi2"], case["hi3"]])
    rng = np.random.default_rng(seed)
    out = []
    for k in range(case["count"]):
        two = k % 2 == 0
        lo, hi = (case["lo2"], case["hi2"]) if two else (case["lo3"],
                                                         case["hi3"])
        n = int(round(math.exp(shape.uniform(math.log(lo), math.log(hi)))))
        frac = rng.uniform(0.05, 0.25)
        tau = rng.uniform(0.55, 1.0)
        force = 8.0 * (tau - 0.5) / 3.0 * 0.05 / (n * n)
        if two:
            out.append(_lattice(9, (n, n, 1), tau, periodic=(1, 0, 0),
                                force=force, solid=_squares(n, n, frac, rng)))
        else:
            out.append(_lattice(19, (n, n, n), tau, periodic=(1, 0, 0),
                                force=force,
                                solid=_spheres((n, n, n), frac, rng)))
    return out


# D3Q27 velocities in the library's order, its inverse map, 1/|e|^2
E27 = np.array([[0, 0, 0], [-1, 0, 0], [0, -1, 0], [0, 0, -1], [0, 0, 1],
                [0, 1, 0], [1, 0, 0], [-1, -1, 0], [-1, 0, -1], [-1, 0, 1],
                [-1, 1, 0], [0, -1, -1], [0, -1, 1], [0, 1, -1], [0, 1, 1],
                [1, -1, 0], [1, 0, -1], [1, 0, 1], [1, 1, 0], [-1, -1, -1],
                [-1, -1, 1], [-1, 1, -1], [-1, 1, 1], [1, -1, -1],
                [1, -1, 1], [1, 1, -1], [1, 1, 1]])
INV27 = np.array([int(np.where((E27 == -e).all(1))[0][0]) for e in E27])
SPLIT27 = np.array([0.0] + [float(np.float32(1.0) / np.float32(e @ e))
                            for e in E27[1:]])


def _sphere_tables(dims, centre, radius):
    """Flags and reflection records of a spherical obstacle: every link of
    an inside node to an outside one is turned about the sphere's normal and
    shared among the three best aligned directions that lead outside."""
    grid = np.stack(np.meshgrid(*(np.arange(n) for n in dims),
                                indexing="ij"), -1).reshape(-1, 3)
    inside = ((grid - centre) ** 2).sum(1) <= radius ** 2
    box = np.zeros([n + 2 for n in dims], bool)  # outside nodes, padded
    box[1:-1, 1:-1, 1:-1] = ~inside.reshape(dims)
    ids = np.where(inside)[0]
    pos = grid[ids]
    free = np.stack([box[tuple((pos + e + 1).T)] for e in E27], 1)
    ids, pos, free = (a[free.any(1)] for a in (ids, pos, free))
    n = len(ids)
    length = np.maximum(np.sqrt((E27 ** 2).sum(1)), 1.0)
    unit = E27 / length[:, None]
    dirs = np.zeros((n, 14), np.uint32)
    weights = np.zeros((n, 81), np.float32)
    for k in range(1, 27):
        rows = np.where(free[:, k])[0]
        if not len(rows):
            continue
        normal = pos[rows] + 0.5 * E27[k] - centre
        normal /= np.linalg.norm(normal, axis=1)[:, None]
        v = 2.0 * (normal @ unit[k])[:, None] * normal - unit[k]
        score = 2.0 - np.linalg.norm(v[:, None, :] - unit[None], axis=2)
        score[~free[rows]] = -1.0
        best = np.argsort(-score, axis=1, kind="stable")[:, :3]
        s = np.take_along_axis(score, best, 1)
        s = np.where(s > 0.0, s, 0.0)
        s /= s.sum(1)[:, None]
        for r in range(3):
            slot = int(INV27[k]) * 3 + r
            d = np.where(s[:, r] > 0.0, best[:, r], 0).astype(np.uint32)
            dirs[rows, slot // 6] |= d << np.uint32(5 * (slot % 6))
            weights[rows, slot] = s[:, r]
    flags = np.where(inside, np.uint8(1), np.uint8(0))
    flags[ids] |= 2
    return flags, ids.astype(np.int32), dirs, weights


def _reference(case, seed):
    rng = np.random.default_rng(seed)
    dims = (case["nx"], case["ny"], case["nz"])
    radius = case["radius"] * min(dims)
    centre = np.array(dims) * 0.5 + rng.uniform(-0.5, 0.5, 3)
    induced = np.full(27, 0.001, np.float32)
    induced[6] = 0.002
    n = dims[0] * dims[1] * dims[2]
    f = (induced[:, None] * (1.0 + 0.05 * rng.random((27, n)))).astype(
        np.float32)
    return dims, _sphere_tables(dims, centre, radius), induced, f


REF_TAU = 0.6


def _ball_mesh(rings, centre, radius):
    """Closed triangle mesh of a ball: rings of latitude, twice as many
    meridians."""
    m = 2 * rings
    t = np.pi * np.arange(1, rings) / rings
    p = 2.0 * np.pi * np.arange(m) / m
    v = np.stack([np.sin(t)[:, None] * np.cos(p), np.sin(t)[:, None] *
                  np.sin(p), np.repeat(np.cos(t)[:, None], m, 1)], -1)
    v = np.concatenate([v.reshape(-1, 3), [[0, 0, 1.0], [0, 0, -1.0]]])
    top, bottom = len(v) - 2, len(v) - 1
    faces = []
    for j in range(m):
        k = (j + 1) % m
        faces.append((top, j, k))
        faces.append((bottom, (rings - 2) * m + k, (rings - 2) * m + j))
        for i in range(rings - 2):
            a, b = i * m + j, i * m + k
            faces.append((a, a + m, b))
            faces.append((b, a + m, b + m))
    return ((v * radius + centre).astype(np.float32),
            np.array(faces, np.int32))


# ------------------------------------------------------------------ passes
def prepare(case, seed):
    kind = case["kind"]
    if kind == "flow":
        lat = _flow(case, seed)
        ctx = capi.Context(_config(lat, case["storage"]))
        if lat["solid"] is not None:
            ctx.upload_solid(lat["solid"])
        ctx.init_equilibrium(lat["rho"], lat["u"])
        return {"case": case, "ctx": ctx}
    if kind == "batch":
        batch = capi.Batch(STORAGE[case["storage"]])
        members = [batch.add(_config(lat, case["storage"]), lat["solid"])
                   for lat in _members(case, seed)]
        batch.autotune(steps=10)
        for m in members:  # tuning steps the members
            m.init_equilibrium()
        return {"case": case, "batch": batch, "members": members}
    if kind == "serve":
        reqs = [{"cfg": _config(lat, case["storage"]), "solid": lat["solid"],
                 "arrival_s": 0.0, "max_steps": case["steps"], "tol": 1e-9}
                for lat in _requests(case, seed)]
        return {"case": case, "requests": reqs}
    if kind == "reference":
        dims, (flags, node, dirs, weights), induced, f = _reference(case, seed)
        ctx = capi.Context(capi.make_config(
            *dims, lattice=capi.D3Q27, mode=capi.MODE_REFERENCE, tau=REF_TAU))
        state = {"case": case, "ctx": ctx}
        ctx.upload_flags(flags)
        ctx.upload_reflections(node, dirs, weights)
        ctx.set_flow(capi.FLOW_PLANE, [0, 0], induced)
        if case["points"]:
            pts = np.zeros(f.shape[1], capi.POINT_DTYPE)
            pts["f"] = f.T
            pts["isInternal"] = flags & 1
            pts["isReflected"] = flags >> 1
            state["points"] = pts
        else:
            ctx.set_populations(f.reshape(-1))
        return state
    rng = np.random.default_rng(seed)
    dims = np.array([case["nx"], case["ny"], case["nz"]])
    spacing = 0.0125
    verts, faces = _ball_mesh(
        case["rings"], spacing * (0.5 * dims + rng.uniform(-0.5, 0.5, 3)),
        spacing * 0.3 * dims.min() * rng.uniform(0.9, 1.0))
    ctx = capi.Context(capi.make_config(
        *(int(d) for d in dims), lattice=capi.D3Q27,
        mode=capi.MODE_REFERENCE, tau=REF_TAU))
    # room for the records of a ball of that size (about two layers of nodes)
    most = 200 + int(4 * 4 * math.pi * (0.3 * dims.min()) ** 2)
    return {"case": case, "ctx": ctx, "verts": verts, "faces": faces,
            "spacing": spacing, "most": most}


def _build_reflections(ctx, verts, faces, spacing, most):
    """lbm_build_reflections into zeroed arrays of `most` records."""
    import ctypes as C
    node = np.zeros(most, np.int32)
    dirs = np.zeros((most, 14), np.uint32)
    weights = np.zeros((most, 81), np.float32)
    count = C.c_int32(0)
    capi.check(capi.load().lbm_build_reflections(
        ctx.h, verts.ctypes.data, len(verts), faces.ctypes.data, len(faces),
        spacing, most, node.ctypes.data, dirs.ctypes.data,
        weights.ctypes.data, C.byref(count)), "lbm_build_reflections")
    return count.value, node, dirs, weights


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "flow":
        state["ctx"].step(case["steps"])
        rho, u = state["ctx"].moments()
        return {"rho": rho, "u": u}
    if kind == "batch":
        state["batch"].step(case["steps"], case["chunk"])
        got = [m.moments() for m in state["members"]]
        return {"rho": np.concatenate([r for r, _ in got]),
                "u": np.concatenate([u.reshape(-1) for _, u in got])}
    if kind == "serve":
        _, results = capi.serve(state["requests"],
                                storage=STORAGE[case["storage"]],
                                chunk=case["chunk"], keep_results=True)
        return {"u": np.concatenate([r["u"].reshape(-1) for r in results]),
                "steps": np.array([r["steps"] for r in results]),
                "status": np.array([r["status"] for r in results])}
    ctx = state["ctx"]
    if kind == "reference":
        if case["points"]:
            ctx.upload_points(state["points"])
        ctx.set_force([0, 0, 0])
        ctx.step_reference(case["steps"], with_force=True)
        if case["points"]:
            return {"f": ctx.download_points()["f"], "force": ctx.force()}
        rho, u = ctx.moments()
        return {"rho": rho, "u": u, "force": ctx.force()}
    inside = capi.voxelize_mesh(ctx, state["verts"], state["faces"],
                                state["spacing"])
    ctx.upload_flags(inside)
    k, node, dirs, weights = _build_reflections(
        ctx, state["verts"], state["faces"], state["spacing"], state["most"])
    flags = inside.copy()
    flags[node[:k]] |= capi.FLAG_REFLECTED
    ctx.upload_flags(flags)
    ctx.upload_reflections(node[:k], dirs[:k], weights[:k])
    return {"inside": inside, "records": k, "node": node,
            "dirs": dirs.view(np.int32), "weights": weights}


def work(case):
    """Every population is read and written once in a pass (a pass of many
    steps needs no more than that from memory), every velocity field is
    written once; each node update's arithmetic is done for each step."""
    kind = case["kind"]
    if kind in ("flow", "reference"):
        n = case["nx"] * case["ny"] * case["nz"]
        q = case.get("q", 27)
        size = BYTES[case.get("storage", "f32")]
        out = 288.0 if case.get("points") else 16.0
        return {"bytes": n * (2.0 * q * size + out),
                "flops": 1.0 * n * case["steps"] * FLOPS[q]}
    if kind == "geometry":
        n = case["nx"] * case["ny"] * case["nz"]
        # a node map out and in, the records of the surface's nodes
        surface = 4 * math.pi * (0.3 * min(case["nx"], case["ny"],
                                           case["nz"])) ** 2
        return {"bytes": 3.0 * n + 2 * 384.0 * surface,
                "flops": 27 * 60.0 * surface + 10.0 * n}
    size = BYTES[case["storage"]]
    lats = (_members(dict(case), 0) if kind == "batch"
            else _requests(case, 0))
    total, flops = 0.0, 0.0
    for lat in lats:
        n = lat["dims"][0] * lat["dims"][1] * lat["dims"][2]
        total += n * (2.0 * lat["q"] * size + 16.0)
        flops += 1.0 * n * case["steps"] * FLOPS[lat["q"]]
    return {"bytes": total, "flops": flops}


# ------------------------------------------------------- values in 64 bits
E19 = E27[:19]
E9 = np.array([[0, 0, 0], [-1, 0, 0], [0, -1, 0], [0, 1, 0], [1, 0, 0],
               [-1, -1, 0], [-1, 1, 0], [1, -1, 0], [1, 1, 0]])
VELOCITIES = {9: E9, 19: E19, 27: E27}
SHELLS = {9: (4 / 9, 1 / 9, 1 / 36), 19: (1 / 3, 1 / 18, 1 / 36),
          27: (8 / 27, 2 / 27, 1 / 54, 1 / 216)}


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _bgk64(lats, steps):
    """The BGK lattices of one velocity set in one pool of nodes: density
    and velocity of each after `steps` steps, in float64."""
    dev = _device()
    q = lats[0]["q"]
    E = VELOCITIES[q]
    w = [SHELLS[q][int(np.abs(e).sum())] for e in E]
    inv = [int(np.where((E == -e).all(1))[0][0]) for e in E]
    total = sum(int(np.prod(a["dims"])) for a in lats)
    one = dict(dtype=torch.float64, device=dev)
    omega, force = torch.empty(total, **one), torch.empty(total, **one)
    solid = torch.zeros(total, dtype=torch.bool, device=dev)
    rho, u = torch.ones(total, **one), torch.zeros(3, total, **one)
    pull = [torch.empty(total, dtype=torch.int32, device=dev) for _ in E]
    lids = any(a["lid_face"] >= 0 for a in lats)
    lid = [None] * q
    at = 0
    for a in lats:
        dims, n = a["dims"], int(np.prod(a["dims"]))
        s = slice(at, at + n)
        omega[s], force[s] = 1.0 / a["tau"], a["force"]
        if a["solid"] is not None:
            solid[s] = torch.from_numpy(a["solid"].astype(bool)).to(dev)
        if a["rho"] is not None:
            rho[s] = torch.from_numpy(a["rho"]).to(dev)
            u[:, s] = torch.from_numpy(a["u"]).to(dev)
        node = torch.arange(n, dtype=torch.int64, device=dev)
        c = [node // (dims[1] * dims[2]), node // dims[2] % dims[1],
             node % dims[2]]
        for i, e in enumerate(E):
            out = torch.zeros(n, dtype=torch.bool, device=dev)
            src = torch.zeros(n, dtype=torch.int64, device=dev)
            for ax in range(3):
                k = c[ax] - int(e[ax])
                if not a["periodic"][ax]:
                    out |= (k < 0) | (k >= dims[ax])
                src = src * dims[ax] + k % dims[ax]
            if a["solid"] is not None:
                out |= solid[s][src]
            pull[i][s] = torch.where(out, inv[i] * total + at + node,
                                     i * total + at + src).to(torch.int32)
            if lids:
                if lid[i] is None:
                    lid[i] = torch.zeros(total, **one)
                if a["lid_face"] >= 0 and e[1] == -1:  # the upper y face
                    lid[i][s] = torch.where(
                        c[1] == dims[1] - 1,
                        6.0 * w[i] * float(e[0]) * a["lid_u"], 0.0)
        at += n
    forced = bool((force != 0).any())

    def dot(e, v):
        t = None
        for ax in range(3):
            if e[ax]:
                x = v[ax] if e[ax] > 0 else -v[ax]
                t = x if t is None else t + x
        return torch.zeros_like(v[0]) if t is None else t

    def equilibrium(i, r, v, usq):
        eu = dot(E[i], v)
        return w[i] * r * (1.0 + 3.0 * eu + 4.5 * eu * eu - 1.5 * usq), eu

    f = torch.empty(q, total, **one)
    usq = (u * u).sum(0)
    for i in range(q):
        f[i] = equilibrium(i, rho, u, usq)[0]
    new = torch.empty_like(f)

    def moments(g):
        r = g.sum(0)
        j = torch.zeros(3, total, **one)
        for i in range(1, q):
            for ax in range(3):
                if E[i][ax]:
                    j[ax] += g[i] if E[i][ax] > 0 else -g[i]
        return r, j

    for _ in range(steps):
        flat = f.reshape(-1)
        for i in range(q):
            torch.index_select(flat, 0, pull[i], out=new[i])
            if lid[i] is not None:
                new[i] += lid[i]
        r, j = moments(new)
        j[0] += 0.5 * force
        v = j / r
        usq = (v * v).sum(0)
        for i in range(q):
            eq, eu = equilibrium(i, r, v, usq)
            new[i] += omega * (eq - new[i])
            if forced:
                ex = float(E[i][0])
                new[i] += (1.0 - 0.5 * omega) * w[i] * force * (
                    3.0 * (ex - v[0]) + 9.0 * eu * ex)
            new[i].masked_fill_(solid, w[i])
        f, new = new, f
    r, j = moments(f)
    j[0] -= 0.5 * force
    v = j / r
    r.masked_fill_(solid, 0.0)
    v.masked_fill_(solid, 0.0)
    r, v = r.cpu().numpy(), v.cpu().numpy()
    out, at = [], 0
    for a in lats:
        n = int(np.prod(a["dims"]))
        out.append((r[at:at + n], v[:, at:at + n]))
        at += n
    return out


def _pools(lats, steps):
    """_bgk64 of lattices of several velocity sets, in their order."""
    got = [None] * len(lats)
    for q in VELOCITIES:
        at = [k for k, a in enumerate(lats) if a["q"] == q]
        if at:
            for k, v in zip(at, _bgk64([lats[k] for k in at], steps)):
                got[k] = v
    return got


def _reference64(case, seed):
    """The reference's main loop (stream, reflect, collide, inject) in
    float64: populations and force."""
    dev = _device()
    dims, (flags, node, dirs, weights), induced, f = _reference(case, seed)
    n = f.shape[1]
    f = torch.from_numpy(f).double().to(dev).reshape(27, *dims)
    induced = torch.from_numpy(induced).double().to(dev)
    inside = torch.from_numpy((flags & 1).astype(bool)).to(dev)
    tau = float(np.float32(REF_TAU))
    w = [SHELLS[27][int(np.abs(e).sum())] for e in E27]
    node64 = node.astype(np.int64)
    slots = []
    plane = np.array([dims[1] * dims[2], dims[2], 1])
    for s in range(1, 81):
        d = (dirs[:, s // 6] >> np.uint32(5 * (s % 6))) & 31
        at = np.where(d > 0)[0]
        if len(at):
            d = d[at].astype(np.int64)
            ts = E27[s] * SPLIT27[s] if s < 27 else np.zeros(3)
            push = E27[d] * SPLIT27[d][:, None] - ts
            slots.append((s // 3, torch.from_numpy(node64[at]).to(dev),
                          torch.from_numpy(d * n + node64[at] +
                                           E27[d] @ plane).to(dev),
                          torch.from_numpy(weights[at, s]).double().to(dev),
                          torch.from_numpy(push).to(dev)))
    force = torch.zeros(3, dtype=torch.float64, device=dev)

    def part(e, size):
        return (slice(max(e, 0), size + min(e, 0)),
                slice(max(-e, 0), size + min(-e, 0)))

    for _ in range(case["steps"]):
        g = torch.zeros_like(f)
        for i, e in enumerate(E27):
            to, frm = zip(*(part(int(e[a]), dims[a]) for a in range(3)))
            g[i][to] = f[i][frm]
        flat = g.reshape(-1)
        for k, src, dst, weight, push in slots:
            val = flat[k * n + src] * weight
            flat.index_add_(0, dst, val)
            force += (val[:, None] * push).sum(0)
        g = g.reshape(27, n)
        g[:, inside] = 0.0
        rho, u = _split_moments(g)
        usq = (u * u).sum(0)
        for i, e in enumerate(E27):
            c = float(e[0]) * u[0] + float(e[1]) * u[1] + float(e[2]) * u[2]
            eq = w[i] * rho * (1.0 + 3.0 * c + 4.5 * c * c - 1.5 * usq)
            g[i] += (eq - g[i]) / tau
        f = g.reshape(27, *dims)
        f[:, 0] += induced[:, None, None]
    return f.reshape(27, n), force


def _split_moments(g):
    rho = g.sum(0)
    u = torch.zeros(3, g.shape[1], dtype=g.dtype, device=g.device)
    for i, e in enumerate(E27):
        for a in range(3):
            if e[a]:
                u[a] += g[i] * (float(e[a]) * SPLIT27[i])
    return rho, torch.where(rho != 0, u / torch.where(rho != 0, rho, 1.0), u)


def exact(case, seed):
    kind = case["kind"]
    if kind == "flow":
        (rho, u), = _bgk64([_flow(case, seed)], case["steps"])
        return {"rho": rho, "u": u}
    if kind == "batch":
        got = _pools(_members(case, seed), case["steps"])
        return {"rho": np.concatenate([r for r, _ in got]),
                "u": np.concatenate([u.reshape(-1) for _, u in got])}
    if kind == "serve":
        steps = -(-case["steps"] // case["chunk"]) * case["chunk"]
        got = _pools(_requests(case, seed), steps)
        return {"u": np.concatenate([u.reshape(-1) for _, u in got]),
                "steps": None, "status": None}
    if kind == "reference":
        f, force = _reference64(case, seed)
        force = force.cpu().numpy()
        if case["points"]:
            return {"f": f.T.contiguous().cpu().numpy(), "force": force}
        rho, u = _split_moments(f)
        return {"rho": rho.cpu().numpy(), "u": u.cpu().numpy(),
                "force": force}
    # the ranking of a reflected direction's targets has ties that rounding
    # decides: the tables have no value of their own in 64 bits
    return None
