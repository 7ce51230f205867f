"""Two steps of large D3Q19 lattices in one pass (FP32 and FP64): the same
bytes as one step at a time, for rows that are whole tiles, rows that start
anywhere, rows cut into strips, bands and chunks with remainders, periodic
and walled axes, moving walls on two axes, a body force, solid nodes and step
counts that the passes divide differently."""
import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi

pytestmark = pytest.mark.gpu

STEPS = (4, 1, 5, 2, 7, 11, 6)
# nx, ny, nz, periodic axes, moving face (or -1), force
CASES = [
    ((110, 60, 64), (1, 0, 0), -1, True),    # whole tiles, one strip
    ((61, 64, 128), (1, 1, 1), -1, False),
    ((121, 67, 93), (0, 1, 0), 5, True),     # odd; lid on the upper z face
    ((97, 61, 65), (0, 0, 0), 3, False),     # cavity
    ((73, 90, 61), (0, 0, 1), 1, True),      # lid on the upper x face
    ((50, 41, 300), (1, 0, 1), -1, True),    # strips
    ((47, 37, 259), (0, 0, 0), 5, False),
    ((200, 25, 120), (0, 1, 1), 0, False),   # few rows
    ((181, 77, 30), (1, 1, 0), 4, True),     # short rows
    ((150, 140, 130), (1, 0, 0), -1, True),  # above two million nodes
]


@pytest.mark.parametrize("storage", [capi.STORE_F32, capi.STORE_F64])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_march_equals_single_steps(k, storage):
    dims, per, lid, forced = CASES[k]
    print(f"case: march {dims} periodic {per} lid {lid} storage {storage}",
          flush=True)
    rng = np.random.default_rng(k)
    n = dims[0] * dims[1] * dims[2]
    kw = {}
    if lid >= 0:
        kw.update(lid_face=lid, lid_u=(0.03, 0.02, -0.01))
    if forced:
        kw.update(force=(1e-5, -2e-6, 3e-6))
    cfg = capi.make_config(*dims, lattice=19, storage=storage, tau=0.7,
                           periodic=per, **kw)
    solid = (rng.random(n) < 0.12).astype(np.uint8) if k % 3 else None
    rho = 1.0 + 0.01 * rng.random(n)
    u = 0.02 * (rng.random((3, n)) - 0.5)
    with capi.Context(cfg) as c:
        if solid is not None:
            c.upload_solid(solid)
        got = []
        for steps in (STEPS, [1] * sum(STEPS)):
            c.init_equilibrium(rho, u)
            for s in steps:
                c.step(s)
            got.append(c.populations(np.float64))
    assert np.isfinite(got[0]).all()
    assert np.array_equal(*got)


# shapes whose FP32 plan is the march (most of those above take it in FP64
# only): rows of whole tiles, which are stored past the caches, rows that
# start anywhere, rows cut into strips
F32_CASES = [
    ((40, 120, 128), (1, 0, 0), -1, True),
    ((96, 96, 64), (0, 0, 1), 3, True),
    ((64, 80, 192), (1, 1, 1), -1, False),
    ((100, 100, 100), (0, 1, 0), 4, True),
    ((200, 100, 40), (1, 0, 1), 2, False),
    ((60, 60, 400), (1, 0, 0), -1, True),    # strips
    ((90, 70, 350), (0, 1, 1), 0, False),    # strips across a periodic end
    ((30, 101, 448), (0, 0, 0), 5, True),    # strips of whole tiles
]


@pytest.mark.parametrize("k", range(len(F32_CASES)))
def test_f32_march_equals_single_steps(k):
    dims, per, lid, forced = F32_CASES[k]
    print(f"case: FP32 march {dims} periodic {per} lid {lid}", flush=True)
    rng = np.random.default_rng(20 + k)
    n = dims[0] * dims[1] * dims[2]
    kw = {}
    if lid >= 0:
        kw.update(lid_face=lid, lid_u=(0.03, 0.02, -0.01))
    if forced:
        kw.update(force=(1e-5, -2e-6, 3e-6))
    cfg = capi.make_config(*dims, lattice=19, storage=capi.STORE_F32, tau=0.7,
                           periodic=per, **kw)
    assert capi.step_route(cfg, 7) == (capi.STEP_MARCH, {1: 3, 2: 2})
    solid = (rng.random(n) < 0.12).astype(np.uint8) if k % 3 else None
    rho = 1.0 + 0.01 * rng.random(n)
    u = 0.02 * (rng.random((3, n)) - 0.5)
    with capi.Context(cfg) as c:
        if solid is not None:
            c.upload_solid(solid)
        got = []
        for steps in ((4, 1, 7), [1] * 12):
            c.init_equilibrium(rho, u)
            for s in steps:
                c.step(s)
            got.append(c.populations())
    assert np.isfinite(got[0]).all()
    assert np.array_equal(*got)
