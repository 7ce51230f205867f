"""GPU mesh voxelisation (lbm_voxelize_mesh) against the oracle's
point-in-mesh loop: identical inside maps for the reference tests' cubes
and for a 1280-face sphere mesh, at several lattice sizes and spacings."""
import os
import sys
import time

import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DATA = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                    "dataFiles")


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def read_obj(path):
    verts, faces = [], []
    with open(path) as fh:
        for line in fh:
            tok = line.split()
            if not tok:
                continue
            if tok[0] == "v":
                verts.append([float(t) for t in tok[1:4]])
            elif tok[0] == "f":
                faces.append([int(t.split("/")[0]) - 1 for t in tok[1:4]])
    return np.array(verts, np.float32), np.array(faces, np.int32)


def icosphere(level, center, radius):
    t = (1.0 + 5 ** 0.5) / 2.0
    v = [(-1, t, 0), (1, t, 0), (-1, -t, 0), (1, -t, 0), (0, -1, t), (0, 1, t),
         (0, -1, -t), (0, 1, -t), (t, 0, -1), (t, 0, 1), (-t, 0, -1), (-t, 0, 1)]
    v = [np.array(p, float) / np.linalg.norm(p) for p in v]
    f = [(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9),
         (5, 11, 4), (11, 10, 2), (10, 7, 6), (7, 1, 8), (3, 9, 4), (3, 4, 2),
         (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11), (6, 2, 10),
         (8, 6, 7), (9, 8, 1)]
    for _ in range(level):
        mid = {}

        def m(a, b):
            key = (min(a, b), max(a, b))
            if key not in mid:
                p = v[a] + v[b]
                v.append(p / np.linalg.norm(p))
                mid[key] = len(v) - 1
            return mid[key]
        nf = []
        for a, b, c in f:
            ab, bc, ca = m(a, b), m(b, c), m(c, a)
            nf += [(a, ab, ca), (b, bc, ab), (c, ca, bc), (ab, bc, ca)]
        f = nf
    verts = (np.array(v) * radius + np.array(center)).astype(np.float32)
    return verts, np.array(f, np.int32)


def write_obj(path, verts, faces):
    with open(path, "w") as fh:
        for p in verts:
            fh.write("v %.9g %.9g %.9g\n" % tuple(float(c) for c in p))
        for a, b, c in faces:
            fh.write(f"f {a + 1} {b + 1} {c + 1}\n")


def oracle_inside(path, dims, spacing):
    mesh = O.Mesh(path)
    ok, internal = mesh.insert(dims, spacing)
    assert ok
    return internal.astype(np.uint8)


def gpu_inside(verts, faces, dims, spacing):
    with capi.Context(capi.make_config(*dims, lattice=27,
                                       mode=capi.MODE_REFERENCE)) as c:
        return capi.voxelize_mesh(c, verts, faces, spacing)


@pytest.mark.parametrize("name", ["cube.obj", "compat_cube.obj",
                                  "cube_angled.obj"])
@pytest.mark.parametrize("dims,spacing", [((32, 32, 32), 0.05),
                                          ((40, 36, 30), 0.03),
                                          ((10, 10, 10), 0.1)])
def test_voxelize_reference_meshes(name, dims, spacing):
    path = os.path.join(DATA, name)
    verts, faces = read_obj(path)
    b = np.array([verts.min(0), verts.max(0)])
    in_box = not ((b[0] < 0).any() or (b[1] > np.array(dims) * spacing).any())
    say(f"case: voxelise {name} {dims} spacing {spacing} in box {in_box}")
    g = gpu_inside(verts, faces, dims, spacing)
    if in_box:
        o = oracle_inside(path, dims, spacing)
    else:
        # insertModel ignores a mesh that leaves the box (Lattice.cpp:236-244);
        # the voxeliser still answers for every node: the oracle's inside
        # test node by node, at the same float coordinates x * spacing
        mesh = O.Mesh(path)
        ok, internal = mesh.insert(dims, spacing)
        assert not ok and not internal.any()
        sp = np.float32(spacing)
        o = np.array([mesh.inside(float(np.float32(x) * sp),
                                  float(np.float32(y) * sp),
                                  float(np.float32(z) * sp))
                      for x in range(dims[0]) for y in range(dims[1])
                      for z in range(dims[2])], np.uint8)
    say(f"  inside {int(g.sum())} (oracle {int(o.sum())})")
    assert np.array_equal(g, o)


def test_voxelize_sphere_mesh(tmp_path):
    verts, faces = icosphere(3, (0.6, 0.6, 0.6), 0.45)
    path = str(tmp_path / "sphere.obj")
    write_obj(path, verts, faces)
    verts, faces = read_obj(path)  # the floats the OBJ holds
    dims, spacing = (48, 48, 48), 0.025
    say(f"case: voxelise sphere ({len(faces)} faces) {dims}")
    t0 = time.perf_counter()
    g = gpu_inside(verts, faces, dims, spacing)
    t1 = time.perf_counter()
    o = oracle_inside(path, dims, spacing)
    t2 = time.perf_counter()
    say(f"  inside {int(g.sum())}  gpu {t1 - t0:.3f} s (incl. setup)  "
        f"oracle {t2 - t1:.3f} s")
    assert np.array_equal(g, o)
    # the sphere's volume within the lattice resolution
    expect = 4.0 / 3.0 * np.pi * 0.45 ** 3 / spacing ** 3
    assert abs(g.sum() - expect) < 0.05 * expect


BIN = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "latticeboltzmanncuda_amd", "bin")


def dump(tmp_path, mesh_path, dims, spacing, gpu):
    import subprocess
    out = tmp_path / ("gpu.bin" if gpu else "host.bin")
    cmd = [os.path.join(BIN, "GeometryDump"), mesh_path, *map(str, dims),
           repr(spacing), str(out)] + (["--gpu"] if gpu else [])
    r = subprocess.run(cmd, timeout=300, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out.read_bytes()


@pytest.mark.parametrize("mesh,dims,spacing", [
    ("cube_angled.obj", (3, 3, 3), 0.5),
    ("compat_cube.obj", (32, 32, 32), 0.05),
    ("cube_angled.obj", (32, 32, 32), 0.05),
    ("cube_angled.obj", (24, 20, 28), 0.045),
    ("sphere", (40, 40, 40), 0.03),
])
def test_gpu_reflection_tables_equal_host_builder(tmp_path, mesh, dims,
                                                  spacing):
    # the GPU voxeliser + reflection-table builder against the host
    # builders (which match the oracle): the same bytes -- flags, record
    # nodes, direction words and weights
    if mesh == "sphere":
        verts, faces = icosphere(2, (0.6, 0.6, 0.6), 0.4)
        path = str(tmp_path / "sphere.obj")
        write_obj(path, verts, faces)
    else:
        path = os.path.join(DATA, mesh)
    say(f"case: reflection tables {mesh} {dims} spacing {spacing}")
    t0 = time.perf_counter()
    host = dump(tmp_path, path, dims, spacing, False)
    t1 = time.perf_counter()
    gpu = dump(tmp_path, path, dims, spacing, True)
    t2 = time.perf_counter()
    n = int(np.prod(dims))
    nrec = int(np.frombuffer(host[n:n + 4], np.int32)[0])
    say(f"  records {nrec}  host {t1 - t0:.2f} s  gpu {t2 - t1:.2f} s "
        "(process wall time)")
    assert nrec > 0
    assert len(host) == len(gpu)
    assert host == gpu


def test_mesh_outside_the_lattice_costs_its_upload():
    # no node in the mesh's box: the faces' edges are not looked at (20,480
    # faces: 0.2 ms more)
    verts, faces = icosphere(5, (10.0, 10.0, 10.0), 2.0)
    say(f"case: {len(faces)} faces beside the lattice")
    took = {}
    with capi.Context(capi.make_config(24, 20, 16, lattice=27,
                                       mode=capi.MODE_REFERENCE)) as c:
        for name, move in (("beside", (40.0, 0.0, 0.0)),
                           ("above", (0.0, 0.0, 30.0)), ("in", (0, 0, 0))):
            v = np.ascontiguousarray(verts + np.float32(move), np.float32)
            best = 1e9
            for _ in range(8):
                t0 = time.perf_counter()
                got = capi.voxelize_mesh(c, v, faces, 1.0)
                best = min(best, time.perf_counter() - t0)
            took[name] = best
            assert bool(np.any(got)) == (name == "in")
    say(f"  {({k: round(1e6 * t) for k, t in took.items()})} us")
    assert took["beside"] < 0.75 * took["in"]
    assert took["above"] < 0.75 * took["in"]
