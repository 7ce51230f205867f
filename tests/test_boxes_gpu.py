"""Several steps of small D2Q9 lattices in one launch (boxes in LDS): the same
bytes as one step at a time, for sizes around a box's side and rim, lattices
smaller than a rim on periodic and walled axes, the largest lattice of each
kind of box, a moving wall, a body force, solid nodes, every storage type and
step counts that the passes divide differently."""
import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi

pytestmark = pytest.mark.gpu

F32, F64, F16, BF16 = (capi.STORE_F32, capi.STORE_F64, capi.STORE_F16,
                       capi.STORE_BF16)
STEPS = (2, 3, 4, 5, 7, 1, 8, 9, 16, 21, 31)
DIMS = [(8, 8), (7, 9), (16, 17), (15, 16), (1, 1), (2, 3), (1, 40), (31, 5),
        (33, 64), (100, 41), (150, 160), (152, 160), (283, 283), (300, 434),
        (361, 362)]


def lattice(nx, ny, storage, k):
    rng = np.random.default_rng(100 * nx + ny)
    n = nx * ny
    per = ((0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0))[k % 4]
    kw = dict(tau=0.7, periodic=per)
    if k % 3 != 1 and not per[1]:
        kw.update(lid_face=3, lid_u=(0.05, 0, 0))
    if k % 5 != 2:
        kw.update(force=(2e-5, 1e-6, 0))
    solid = (rng.random(n) < 0.15).astype(np.uint8) if k % 7 != 3 else None
    u = 0.02 * (rng.random((3, n)) - 0.5)
    u[2] = 0
    cfg = capi.make_config(nx, ny, 1, lattice=capi.D2Q9, storage=storage, **kw)
    return cfg, solid, 1.0 + 0.01 * rng.random(n), u


def populations(member, rho, u, steps):
    member.init_equilibrium(rho, u)
    for n in steps:
        member.step(n)
    return member.populations(np.float64)


@pytest.mark.parametrize("storage", [F32, F64, F16, BF16])
def test_boxes_equal_single_steps(storage):
    for k in range(2 * len(DIMS)):
        nx, ny = DIMS[k // 2]
        print(f"case: boxes {nx} x {ny}, storage {storage}, variant {k}",
              flush=True)
        cfg, solid, rho, u = lattice(nx, ny, storage, k)
        with capi.Context(cfg) as c:
            if solid is not None:
                c.upload_solid(solid)
            got = populations(c, rho, u, STEPS)
            want = populations(c, rho, u, [1] * sum(STEPS))
        assert np.array_equal(got, want)
