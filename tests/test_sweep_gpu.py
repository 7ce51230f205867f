"""Several steps of D2Q9 lattices in one pass over memory (the sweep, which
large lattices and large batches take): the same bytes as one step at a
time, for rows that fill a wavefront's strip in part, exactly or in several
strips, for one or several x-chunks per wavefront, periodic and walled
axes, a moving wall, a body force, solid nodes, every storage type and
every number of steps that the passes divide differently."""
import os
import sys

import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi

pytestmark = pytest.mark.gpu

F32, F64, F16, BF16 = (capi.STORE_F32, capi.STORE_F64, capi.STORE_F16,
                       capi.STORE_BF16)
STEPS = (2, 3, 4, 5, 7, 1, 8)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


# nx, ny around a strip's 64 lanes (56 of them stored between two others),
# and rows that share a wavefront with other chunks (ny <= 32)
DIMS = [(70, 64), (9, 65), (33, 200), (5, 57), (130, 56), (3, 121), (64, 32),
        (40, 9), (2, 300), (1, 1), (1, 128), (50, 24), (37, 25), (120, 120)]


def small_lattices(storage):
    rng = np.random.default_rng(17)
    k = 0
    for nx, ny in DIMS:
        for per in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0)):
            kw = dict(tau=0.7, periodic=per)
            if k % 2 and not per[1]:
                kw.update(lid_face=3, lid_u=(0.05, 0, 0))
            if k % 3 != 1:
                kw.update(force=(2e-5, 1e-6, 0))
            solid = None
            if k % 4 != 3:
                solid = (rng.random(nx * ny) < 0.15).astype(np.uint8)
            k += 1
            n = nx * ny
            u = 0.02 * (rng.random((3, n)) - 0.5)
            u[2] = 0
            yield (capi.make_config(nx, ny, 1, lattice=capi.D2Q9,
                                    storage=storage, **kw), solid,
                   1.0 + 0.01 * rng.random(n), u)


@pytest.mark.parametrize("storage", [F32, F64, F16, BF16])
def test_batch_sweep_equals_single_steps(storage):
    # a large member makes the batch take the sweep; the small ones, alone,
    # are stepped one step at a time
    side = 2300 if storage in (F16, BF16) else 800
    say(f"case: batch sweep, storage {storage}, {len(DIMS) * 4} shapes")
    lattices = list(small_lattices(storage))
    with capi.Batch(storage) as b:
        big = b.add(capi.make_config(side, side, 1, lattice=capi.D2Q9,
                                     storage=storage, tau=0.8, lid_face=3,
                                     lid_u=(0.05, 0, 0)))
        members = []
        for cfg, solid, rho, u in lattices:
            members.append(b.add(cfg, solid))
            members[-1].init_equilibrium(rho, u)
        for n in STEPS:
            b.step(n)
        b.step(24, 6)
        b.synchronize()
        got = [m.populations(np.float64) for m in members]
        rho, _ = big.moments()
    assert np.isfinite(rho).all()
    for (cfg, solid, rho, u), g in zip(lattices, got):
        with capi.Context(cfg) as c:
            c.upload_solid(solid)
            c.init_equilibrium(rho, u)
            c.step(sum(STEPS) + 24)
            want = c.populations(np.float64)
        assert np.array_equal(g, want), (cfg.nx, cfg.ny, list(cfg.periodic))


@pytest.mark.parametrize("dims,per,storage", [
    ((700, 301), (1, 0, 0), F32),    # odd rows, six strips
    ((5000, 50), (0, 1, 0), F32),    # one strip with its halo, periodic
    ((333, 777), (1, 1, 0), F64),
    ((2801, 2701), (0, 0, 0), F16),
    ((2800, 2702), (1, 1, 0), BF16)])
def test_large_lattice_sweep_equals_single_steps(dims, per, storage):
    say(f"case: sweep {dims} periodic {per} storage {storage}")
    n = dims[0] * dims[1]
    rng = np.random.default_rng(5)
    solid = (rng.random(n) < 0.1).astype(np.uint8)
    kw = dict(lid_face=3, lid_u=(0.05, 0, 0)) if not per[1] else {}
    cfg = capi.make_config(*dims, 1, lattice=capi.D2Q9, storage=storage,
                           tau=0.8, periodic=per, force=(1e-5, 0, 0), **kw)
    got = []
    for single in (False, True):
        if single:
            os.environ["LBM_GROUP_STEP"] = "0"
        try:
            with capi.Context(cfg) as c:
                c.upload_solid(solid)
                c.init_equilibrium()
                for k in STEPS:
                    c.step(k)
                got.append(c.populations())
        finally:
            os.environ.pop("LBM_GROUP_STEP", None)
    assert np.array_equal(*got)


# above the sizes that are stepped in boxes, and rows of 8 to 16 nodes
@pytest.mark.parametrize("dims,per,storage", [
    ((1201, 701), (0, 0, 0), F32),     # strips with a remainder
    ((17001, 50), (0, 1, 0), F32),     # one strip with its halo, periodic
    ((4001, 233), (1, 0, 0), F32),
    ((62501, 16), (1, 0, 0), F32),     # several chunks a wavefront
    ((2, 400000), (1, 1, 0), F32),     # two rows
    ((901, 777), (1, 1, 0), F64),
    ((250001, 8), (0, 0, 0), F64),
    ((23, 30011), (0, 0, 0), F64)])
def test_sweep_above_the_boxes_equals_single_steps(dims, per, storage):
    say(f"case: sweep above the boxes {dims} periodic {per} storage {storage}")
    n = dims[0] * dims[1]
    rng = np.random.default_rng(6)
    solid = (rng.random(n) < 0.1).astype(np.uint8)
    kw = dict(lid_face=3, lid_u=(0.05, 0, 0)) if not per[1] else {}
    cfg = capi.make_config(*dims, 1, lattice=capi.D2Q9, storage=storage,
                           tau=0.8, periodic=per, force=(1e-5, 0, 0), **kw)
    assert capi.step_route(cfg, 8) == (capi.STEP_SWEEP, {4: 2})
    rho = 1.0 + 0.01 * rng.random(n)
    u = 0.02 * (rng.random((3, n)) - 0.5)
    u[2] = 0
    with capi.Context(cfg) as c:
        c.upload_solid(solid)
        got = []
        for steps in ((3, 4, 6, 8, 1, 11), [1] * 33):
            c.init_equilibrium(rho, u)
            for s in steps:
                c.step(s)
            got.append(c.populations(np.float64))
    assert np.isfinite(got[0]).all()
    assert np.array_equal(*got)
