"""Geometry set-up on the GPU at the places where its short cuts could go
wrong: the line counts of the voxeliser against the rule that it documents,
on a face or winding number above 1/2, with all solid angles summed in numpy
(the oracle's ray parity is another rule where shells overlap; meshes with vertices, edges and faces on lattice lines, several shells,
faces turned inside out, meshes that do not close), reflection rays that
leave the faces near their node, and the receiver tables for records in any
order."""
import ctypes as C
import sys

import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi
from oracle import oracle as O
from test_voxel_gpu import gpu_inside, icosphere, read_obj, write_obj

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def box_mesh(lo, hi):
    v = np.array([[x, y, z] for x in (lo[0], hi[0]) for y in (lo[1], hi[1])
                  for z in (lo[2], hi[2])], np.float32)
    f = [(0, 1, 3), (0, 3, 2), (4, 6, 7), (4, 7, 5), (0, 4, 5), (0, 5, 1),
         (2, 3, 7), (2, 7, 6), (0, 2, 6), (0, 6, 4), (1, 5, 7), (1, 7, 3)]
    return v, np.array(f, np.int32)


def joined(*meshes):
    v, f, at = [], [], 0
    for a, b in meshes:
        v.append(a)
        f.append(b + at)
        at += len(a)
    return np.concatenate(v), np.concatenate(f)


def octahedron(c, r):
    v = np.array([[r, 0, 0], [-r, 0, 0], [0, r, 0], [0, -r, 0], [0, 0, r],
                  [0, 0, -r]], np.float32) + np.float32(c)
    f = [(0, 2, 4), (2, 1, 4), (1, 3, 4), (3, 0, 4), (2, 0, 5), (1, 2, 5),
         (3, 1, 5), (0, 3, 5)]
    return v, np.array(f, np.int32)


H = 0.125  # exact in binary: lattice lines run through vertices and edges
MESHES = {
    # corners on nodes: lines along the box's edges, nodes on its faces
    "box on nodes": box_mesh((2 * H, 2 * H, 2 * H), (9 * H, 7 * H, 8 * H)),
    "box between nodes": box_mesh((0.3, 0.28, 0.33), (1.1, 0.9, 1.02)),
    # lines through the tips and the edges of all faces
    "octahedron": octahedron((6 * H, 6 * H, 6 * H), 4 * H),
    "octahedron inside out": (octahedron((6 * H, 6 * H, 6 * H), 4 * H)[0],
                              octahedron((0, 0, 0), 1)[1][:, ::-1].copy()),
    # W = 2 in the inner shell; 0 where it is turned round
    "two shells": joined(box_mesh((H, H, H), (10 * H, 10 * H, 10 * H)),
                         octahedron((5 * H, 5 * H, 5 * H), 3 * H)),
    "hollow": joined(box_mesh((H, H, H), (10 * H, 10 * H, 10 * H)),
                     (octahedron((5 * H, 5 * H, 5 * H), 3 * H)[0],
                      octahedron((0, 0, 0), 1)[1][:, ::-1])),
    "ball": icosphere(2, (0.7, 0.71, 0.69), 0.5),
    # do not close: every node takes the sum of solid angles
    "open box": (box_mesh((0.3, 0.28, 0.33), (1.1, 0.9, 1.02))[0],
                 box_mesh((0, 0, 0), (1, 1, 1))[1][:10]),
    "one face turned": (octahedron((6 * H, 6 * H, 6 * H), 4 * H)[0],
                        np.concatenate([octahedron((0, 0, 0), 1)[1][:7],
                                        [[3, 0, 5]]]).astype(np.int32)),
    # a face without area closes it all the same
    "flat face": (octahedron((6 * H, 6 * H, 6 * H), 4 * H)[0],
                  np.concatenate([octahedron((0, 0, 0), 1)[1],
                                  [[0, 0, 2]]]).astype(np.int32)),
}


def winding_inside(verts, faces, dims, h):
    x = [np.arange(n).astype(np.float32) * np.float32(h) for n in dims]
    p = np.stack(np.meshgrid(*x, indexing="ij"), -1).reshape(-1, 3).astype(
        np.float64)
    on = np.zeros(len(p), bool)
    omega = np.zeros(len(p))
    for f in faces:
        a, b, c = (verts[k].astype(np.float64) for k in f)
        n = np.cross(b - a, c - a)
        nn = np.linalg.norm(n)
        if nn:
            off = np.abs((p - a) @ n)
            scale = nn * (np.linalg.norm(p - a, axis=1) +
                          np.linalg.norm(b - a))
            hit = off <= 1e-12 * scale
            for u, v in ((a, b), (b, c), (c, a)):
                hit &= np.cross(v - u, p - u) @ n >= -1e-12 * nn * nn
            on |= hit
        r = [q - p for q in (a, b, c)]
        la, lb, lc = (np.linalg.norm(q, axis=1) for q in r)
        num = (r[0] * np.cross(r[1], r[2])).sum(1)
        den = la * lb * lc + (r[0] * r[1]).sum(1) * lc + \
            (r[1] * r[2]).sum(1) * la + (r[2] * r[0]).sum(1) * lb
        omega += 2.0 * np.arctan2(num, den)
    box = ((p >= verts.min(0)) & (p <= verts.max(0))).all(1)
    w = np.abs(omega / (4 * np.pi))
    # a mesh that does not close can have W = 1/2 itself at a node: rounding
    # decides there, for either side
    tie = ~on & (np.abs(w - 0.5) < 1e-9)
    return (box & (on | (w > 0.5))).astype(np.uint8), tie


@pytest.mark.parametrize("name", MESHES)
@pytest.mark.parametrize("dims", [(12, 13, 11), (11, 12, 70)])
def test_voxelize_lines(tmp_path, name, dims):
    verts, faces = MESHES[name]
    path = str(tmp_path / "mesh.obj")
    write_obj(path, verts, np.asarray(faces))
    verts, faces = read_obj(path)
    say(f"case: voxelise {name} {dims}")
    g = gpu_inside(verts, faces, dims, H)
    o, tie = winding_inside(verts, faces, dims, H)
    say(f"  inside {int(g.sum())} (solid angles {int(o.sum())}), "
        f"{int(tie.sum())} ties")
    assert tie.sum() <= 1 and o.any()
    assert np.array_equal(g[~tie], o[~tie])


def build(ctx, verts, faces, spacing, most):
    node = np.zeros(most, np.int32)
    dirs = np.zeros((most, 14), np.uint32)
    w = np.zeros((most, 81), np.float32)
    k = C.c_int32(0)
    v, f = np.ascontiguousarray(verts), np.ascontiguousarray(faces)
    capi.check(capi.load().lbm_build_reflections(
        ctx.h, v.ctypes.data, len(v), f.ctypes.data, len(f), spacing, most,
        node.ctypes.data, dirs.ctypes.data, w.ctypes.data, C.byref(k)),
        "lbm_build_reflections")
    return node[:k.value], dirs[:k.value], w[:k.value]


@pytest.mark.parametrize("shift", [0, 2])
def test_reflection_tables_any_flags(tmp_path, shift):
    # shift 2: the flagged block lies two nodes beside the mesh, so most
    # rays meet no face on their link (the next face along the ray, or none)
    verts, faces = icosphere(2, (0.75, 0.75, 0.75), 0.4)
    path = str(tmp_path / "ball.obj")
    write_obj(path, verts, faces)
    verts, faces = read_obj(path)
    dims = (13, 12, 14)
    mesh = O.Mesh(path)
    ok, inside = mesh.insert(dims, H)
    assert ok
    inside = np.roll(inside.reshape(dims), shift, 0).reshape(-1)
    say(f"case: reflection tables, flags shifted by {shift}")
    flags, (node, dirs, w) = mesh.preprocess(dims, H, inside * O.FLAG_INTERNAL)
    with capi.Context(capi.make_config(*dims, lattice=27,
                                       mode=capi.MODE_REFERENCE)) as c:
        c.upload_flags(inside)
        gn, gd, gw = build(c, verts, faces, H, int(inside.sum()))
    assert len(node) and np.array_equal(gn, node)
    assert np.array_equal(gd, dirs) and np.array_equal(gw, w)


def ref_setup(dims=(20, 18, 21)):
    verts, faces = icosphere(2, (1.2, 1.1, 1.3), 0.6)
    ctx = capi.Context(capi.make_config(*dims, lattice=27,
                                        mode=capi.MODE_REFERENCE, tau=0.6))
    flags = capi.voxelize_mesh(ctx, verts, faces, H)
    ctx.upload_flags(flags)
    node, dirs, w = build(ctx, verts, faces, H, int(flags.sum()))
    flags[node] |= capi.FLAG_REFLECTED
    ctx.upload_flags(flags)
    induced = np.full(27, 0.001, np.float32)
    induced[6] = 0.002
    ctx.set_flow(capi.FLOW_PLANE, [0, 0], induced)
    n = ctx.n
    f = (induced[:, None] * (1 + 0.1 * np.random.default_rng(3).random(
        (27, n)))).astype(np.float32)
    return ctx, flags, node, dirs, w, f


def run(ctx, f, steps=6):
    ctx.set_populations(f.reshape(-1))
    ctx.set_force([0, 0, 0])
    ctx.step_reference(steps, True)
    return ctx.populations(), ctx.force()


def test_receivers_in_any_record_order():
    say("case: records shuffled, fewer, and staged")
    ctx, flags, node, dirs, w, f = ref_setup()
    with ctx:
        order = np.random.default_rng(1).permutation(len(node))
        ctx.upload_reflections(node, dirs, w)
        a, fa = run(ctx, f)
        ctx.upload_reflections(node[order], dirs[order], w[order])
        b, fb = run(ctx, f)
        assert np.array_equal(a, b) and np.array_equal(fa, fb)
        # some records only, and nodes flagged reflecting without one
        some = order[:len(order) // 3]
        ctx.upload_reflections(node[some], dirs[some], w[some])
        b, _ = run(ctx, f)
        ctx.set_populations(f.reshape(-1))
        for _ in range(6):
            ctx.stream()
            ctx.reflect(False)
            ctx.collide(0.6)
            ctx.flow()
        assert np.array_equal(b, ctx.populations())
        assert not np.array_equal(a, b)
        # no records, then no flags at all
        ctx.upload_reflections(node[:0], dirs[:0], w[:0])
        b, fb = run(ctx, f)
        assert np.isfinite(b).all() and not fb.any()
        ctx.upload_flags(np.zeros_like(flags))
        c, _ = run(ctx, f)
        assert not np.array_equal(b, c)


def test_receivers_follow_uploaded_points():
    say("case: flags through upload_points")
    ctx, flags, node, dirs, w, f = ref_setup()
    with ctx:
        ctx.upload_reflections(node, dirs, w)
        want, _ = run(ctx, f)
        pts = np.zeros(ctx.n, capi.POINT_DTYPE)
        pts["f"] = f.T
        pts["isInternal"] = flags & 1
        pts["isReflected"] = flags >> 1
        for _ in range(2):  # unchanged flags
            ctx.upload_points(pts)
            ctx.step_reference(6, True)
            assert np.array_equal(ctx.populations(), want)
        other = pts.copy()
        other["isReflected"][node[::2]] = 0
        ctx.upload_points(other)
        ctx.step_reference(6, True)
        assert not np.array_equal(ctx.populations(), want)
        ctx.upload_points(pts)
        ctx.step_reference(6, True)
        assert np.array_equal(ctx.populations(), want)


def test_refused_geometries():
    say("case: geometries that the reflection cannot run")
    ctx, flags, node, dirs, w, f = ref_setup()
    with ctx:
        twice = np.concatenate([node, node[5:6]])
        with pytest.raises(capi.LbmError,
                           match=f"two reflection records for node {node[5]}"):
            ctx.upload_reflections(twice, np.concatenate([dirs, dirs[5:6]]),
                                   np.concatenate([w, w[5:6]]))
        bad = flags.copy()
        bad[node[7]] = capi.FLAG_REFLECTED
        ctx.upload_flags(bad)
        with pytest.raises(capi.LbmError,
                           match=f"reflecting node {node[7]} is not internal"):
            ctx.upload_reflections(node, dirs, w)
        # a target that is flagged: the node that slot 3 k + r of the first
        # record's first used slot leads to
        s = next(s for s in range(3, 81) if O.slot_dir(dirs[0], s))
        e = O.std_tables(27)[0][O.slot_dir(dirs[0], s)]
        nx, ny, nz = ctx.dims
        t = int(node[0]) + int(e[2]) + nz * (int(e[1]) + ny * int(e[0]))
        bad = flags.copy()
        bad[t] = capi.FLAG_INTERNAL
        ctx.upload_flags(bad)
        with pytest.raises(capi.LbmError,
                           match=f"reflection target {t} is a flagged node"):
            ctx.upload_reflections(node, dirs, w)
        ctx.upload_flags(flags)
        ctx.upload_reflections(node, dirs, w)
        got, _ = run(ctx, f)
        assert np.isfinite(got).all()
