"""C4 batching: lattices stepped together by one persistent kernel (plain
launches and hipGraph chunks) give the same populations as each lattice
stepped alone; admission honours the HBM budget; residuals are right."""
import sys
import time

import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi, workloads

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def mixed_specs():
    rng = np.random.default_rng(11)
    specs = []
    # D2Q9 cavities and channels with squares
    for (nx, ny), kind in [((40, 33), "cavity"), ((97, 64), "channel"),
                           ((32, 200), "cavity"), ((150, 41), "channel")]:
        solid = workloads.random_squares(nx, ny, 0.1, rng)
        if kind == "cavity":
            cfg = capi.make_config(nx, ny, 1, lattice=9, tau=0.7, lid_face=3,
                                   lid_u=(0.1, 0, 0))
        else:
            cfg = capi.make_config(nx, ny, 1, lattice=9, tau=0.8,
                                   periodic=(1, 0, 0), force=(1e-5, 0, 0))
        specs.append((cfg, solid))
    # D3Q19 channel with spheres and a cavity
    solid, _ = capi.random_spheres((48, 24, 20), 3, 0.15, 3.0, 5.0, True)
    specs.append((capi.make_config(48, 24, 20, lattice=19, tau=0.8,
                                   periodic=(1, 0, 0), force=(1e-5, 0, 0)),
                  solid))
    specs.append((capi.make_config(20, 20, 20, lattice=19, tau=0.6,
                                   lid_face=3, lid_u=(0.1, 0, 0)), None))
    return specs


def run_alone(cfg, solid, steps):
    with capi.Context(cfg) as c:
        c.upload_solid(solid)
        c.init_equilibrium()
        c.step(steps)
        return c.populations()


@pytest.mark.parametrize("chunk", [0, 10])
def test_batch_equals_alone(chunk):
    say(f"case: batch of 6 mixed lattices, chunk={chunk}")
    specs = mixed_specs()
    steps = 37  # odd: exercises the buffer parity bookkeeping
    with capi.Batch(capi.STORE_F32) as b:
        members = [b.add(cfg, solid) for cfg, solid in specs]
        b.set_launch(128, 64)
        b.step(steps, chunk)
        b.synchronize()
        got = [m.populations() for m in members]
    for (cfg, solid), g in zip(specs, got):
        ref = run_alone(cfg, solid, steps)
        assert np.array_equal(g, ref)


def test_batch_launch_shapes_and_autotune_agree():
    say("case: batch launch shapes + autotune")
    specs = mixed_specs()
    outs = []
    for shape in [(64, 0), (256, 16), (512, 1000), None]:
        with capi.Batch(capi.STORE_F16) as b:
            members = [b.add(capi.make_config(
                cfg.nx, cfg.ny, cfg.nz, lattice=cfg.lattice,
                storage=capi.STORE_F16, tau=cfg.tau,
                periodic=tuple(cfg.periodic), lid_face=cfg.lid_face,
                lid_u=tuple(cfg.lid_u), force=tuple(cfg.force)), solid)
                for cfg, solid in specs]
            if shape is None:
                block, grid = b.autotune(steps=4, use_cache=False)
                say(f"  autotuned block {block} grid {grid}")
                # autotuning stepped the members: start again from rest
                for m in members:
                    m.init_equilibrium()
            else:
                b.set_launch(*shape)
            b.step(24, 12)
            b.synchronize()
            outs.append([m.populations() for m in members])
    for o in outs[1:]:
        for a, c in zip(outs[0], o):
            assert np.array_equal(a, c)


def test_batch_add_remove_between_chunks():
    say("case: admit / evict between graph chunks")
    specs = mixed_specs()
    with capi.Batch(capi.STORE_F32) as b:
        m0 = b.add(*specs[0])
        m1 = b.add(*specs[1])
        b.step(20, 10)
        m2 = b.add(*specs[2])  # joins late
        b.step(20, 10)
        b.remove(m1)           # leaves early
        b.step(20, 10)
        b.synchronize()
        g0, g2 = m0.populations(), m2.populations()
    assert np.array_equal(g0, run_alone(*specs[0], 60))
    assert np.array_equal(g2, run_alone(*specs[2], 40))


def test_batch_budget_admission():
    say("case: HBM budget admission")
    cfg = capi.make_config(64, 64, 1, lattice=9, tau=0.7)
    need = capi.Batch.estimate_bytes(cfg)
    with capi.Batch(capi.STORE_F32, budget_bytes=3 * need + 4096) as b:
        b.add(cfg)
        b.add(cfg)
        with pytest.raises(capi.LbmError) as e:
            for _ in range(3):
                b.add(cfg)
        assert e.value.code == 6  # LBM_ERR_BUDGET
        nlat, _, used = b.info()
        assert nlat >= 2 and used <= 3 * need + 4096


def test_batch_residuals_match_host():
    say("case: batch residuals vs host computation")
    specs = mixed_specs()[:3]
    with capi.Batch(capi.STORE_F32) as b:
        members = [b.add(cfg, solid, track_residual=True)
                   for cfg, solid in specs]
        b.step(50)
        r0 = b.residuals()  # against the zero snapshot: 1 for moving flow
        u_prev = [m.moments()[1].astype(np.float64) for m in members]
        b.step(20)
        r1 = b.residuals()
        for m, up, (cfg, solid) in zip(members, u_prev, specs):
            _, u = m.moments()
            fl = solid == 0
            d = (u.astype(np.float64) - up)[:, fl]
            ref = np.sqrt((d ** 2).sum() / (u.astype(np.float64)[:, fl] ** 2).sum())
            assert abs(r0[m.slot] - 1.0) < 1e-9
            assert abs(r1[m.slot] - ref) <= 1e-6 * ref + 1e-12


def test_batch_member_parameter_change_between_chunks():
    say("case: tau / force of a member changed between chunks")
    cfg, solid = mixed_specs()[1]  # D2Q9 channel with squares
    with capi.Batch(capi.STORE_F32) as b:
        m = b.add(cfg, solid)
        b.step(20, 10)
        m.set_tau(0.65)
        m.set_body_force((2e-5, 0.0, 0.0))
        b.step(20, 10)
        b.synchronize()
        got = m.populations()
    with capi.Context(capi.make_config(
            cfg.nx, cfg.ny, cfg.nz, lattice=cfg.lattice, tau=cfg.tau,
            periodic=tuple(cfg.periodic), force=tuple(cfg.force))) as c:
        c.upload_solid(solid)
        c.init_equilibrium()
        c.step(20)
        c.set_tau(0.65)
        c.set_body_force((2e-5, 0.0, 0.0))
        c.step(20)
        ref = c.populations()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("calls", [[(9, 0)], [(10, 0), (35, 0)],
                                   [(45, 10), (100, 100), (12, 6), (7, 2)]])
def test_classes_side_by_side_equal_alone(calls):
    # D2Q9, D3Q19 and D3Q27 members step on streams of their own; a member
    # read between two calls is complete, and one that leaves and one that
    # joins find no step under way
    say(f"case: three lattice types side by side, calls {calls}")
    specs = mixed_specs()
    specs.append((capi.make_config(30, 17, 22, lattice=27, tau=0.7,
                                   periodic=(1, 1, 0)), None))
    with capi.Batch(capi.STORE_F32) as b:
        members = [b.add(cfg, solid) for cfg, solid in specs]
        done = 0
        for n, chunk in calls:
            b.step(n, chunk)
            done += n
            for k in (0, 4, 6):
                assert np.array_equal(members[k].populations(),
                                      run_alone(*specs[k], done))
        b.remove(members[1])
        late = b.add(*specs[5])
        b.step(40, 20)
        assert np.array_equal(late.populations(), run_alone(*specs[5], 40))
        assert np.array_equal(members[6].populations(),
                              run_alone(*specs[6], done + 40))


@pytest.mark.parametrize("storage,side", [(capi.STORE_F32, 1400),
                                          (capi.STORE_F64, 1400),
                                          (capi.STORE_F16, 2500)])
def test_autotuner_times_the_kernel_whose_shape_it_chooses(storage, side):
    # large D2Q9 batches take several steps a launch in a kernel of one shape;
    # the tuner's shape is for the other one, so its 19 candidates take at
    # least as long as single steps
    say(f"case: autotuner on a batch of sweeps, storage {storage}")
    steps = 60
    cfg = capi.make_config(side, side, 1, lattice=9, storage=storage, tau=0.7,
                           periodic=(1, 0, 0), force=(1e-6, 0, 0))
    with capi.Batch(storage) as b:
        m = b.add(cfg)
        b.step(10)
        b.synchronize()
        t0 = time.perf_counter()
        b.autotune(steps, use_cache=False)
        tuning = time.perf_counter() - t0
        single = 1e9
        for _ in range(3):
            t0 = time.perf_counter()
            for _ in range(steps // 2):
                b.step(2)
            b.synchronize()
            single = min(single, (time.perf_counter() - t0) / steps)
        b.step(30)
        b.synchronize()
        got = m.populations()
    say(f"  tuning {tuning * 1e3:.1f} ms, a single step {single * 1e6:.1f} us")
    assert tuning > 0.85 * 19 * steps * single
    total = 10 + 19 * (steps + 2) + 3 * steps + 30
    assert np.array_equal(got, run_alone(cfg, None, total))


def test_many_members_step_and_change(tmp_path):
    # more lattices than the sweep has places for: a call after an odd number
    # of steps brings their descriptors up to date and no more (it planned
    # every sweep anew: 49 ms); members that change parameters, or by a
    # snapshot their periodic axes, are stepped with what they have now
    say("case: 3500 lattices and a long one, odd calls")
    small = capi.make_config(16, 16, 1, lattice=9, tau=0.7, lid_face=3,
                             lid_u=(0.05, 0, 0))
    long = capi.make_config(4000, 64, 1, lattice=9, tau=0.8,
                            periodic=(1, 0, 0), force=(1e-5, 0, 0))
    other = capi.make_config(16, 16, 1, lattice=9, tau=0.9,
                             periodic=(0, 1, 0), force=(0, 1e-5, 0))
    path = str(tmp_path / "other.snap")
    with capi.Context(other) as c:
        c.init_equilibrium()
        c.step(5)
        c.save(path)
    with capi.Batch(capi.STORE_F32) as b:
        members = [b.add(small) for _ in range(3500)]
        big = b.add(long)
        took = []
        for n in (1, 1, 3, 1, 1, 1, 5, 1):
            b.synchronize()
            t0 = time.perf_counter()
            b.step(n)
            b.synchronize()
            took.append(time.perf_counter() - t0)
        say(f"  {[round(1e3 * t, 2) for t in took]} ms")
        assert sorted(took)[4] < 8e-3
        members[7].set_tau(0.65)
        members[9].load(path)
        b.step(7)
        b.step(10, 2)
        b.synchronize()
        got = [m.populations() for m in (members[0], members[3499], big,
                                         members[7], members[9])]
    assert np.array_equal(got[0], run_alone(small, None, 31))
    assert np.array_equal(got[1], got[0])
    assert np.array_equal(got[2], run_alone(long, None, 31))
    with capi.Context(small) as c:
        c.init_equilibrium()
        c.step(14)
        c.set_tau(0.65)
        c.step(17)
        assert np.array_equal(got[3], c.populations())
    with capi.Context(other) as c:
        c.load(path)
        c.step(17)
        assert np.array_equal(got[4], c.populations())


def test_short_chunks_of_several_types_cost_no_more_than_their_launches():
    # chunks of two steps hold all lattice types in one graph: with one graph
    # per type and chunk they took up to 1.4 times as long
    say("case: short chunks of two lattice types")
    specs = [(capi.make_config(90, 80 + k, 1, lattice=9, tau=0.7, lid_face=3,
                               lid_u=(0.05, 0, 0)), None) for k in range(6)]
    specs += [(capi.make_config(20, 22, 20 + k, lattice=19, tau=0.7,
                                periodic=(1, 0, 0), force=(1e-5, 0, 0)), None)
              for k in range(6)]

    def members(select):
        b = capi.Batch(capi.STORE_F32)
        ms = [b.add(*s) for s in specs if select(s[0].lattice)]
        b.step(20, 2)
        b.synchronize()
        return b, ms

    def took(b):
        best = 1e9
        for _ in range(5):
            t0 = time.perf_counter()
            for _ in range(20):
                b.step(20, 2)
            b.synchronize()
            best = min(best, (time.perf_counter() - t0) / 20)
        return best

    both, ms = members(lambda q: True)
    flat, _ = members(lambda q: q == 9)
    deep, _ = members(lambda q: q == 19)
    t = [took(b) * 1e6 for b in (both, flat, deep)]
    say(f"  20 steps by twos: both {t[0]:.0f} us, D2Q9 {t[1]:.0f}, D3Q19 "
        f"{t[2]:.0f}")
    assert t[0] < 0.92 * (t[1] + t[2])
    got = [m.populations() for m in ms]
    for b in (both, flat, deep):
        b.close()
    for (cfg, solid), g in list(zip(specs, got))[::5]:
        assert np.array_equal(g, run_alone(cfg, solid, 20 + 5 * 20 * 20))


def test_short_and_long_calls_in_turn_equal_alone():
    # a call of 8 steps captures one graph of both types, one of 16 a graph
    # per type, which the short calls after it take too
    say("case: short and long calls in chunks of 8, two lattice types")
    specs = [(capi.make_config(90, 80 + k, 1, lattice=9, tau=0.7, lid_face=3,
                               lid_u=(0.05, 0, 0)), None) for k in range(2)]
    specs += [(capi.make_config(28, 27, 28 + k, lattice=19, tau=0.7,
                                periodic=(1, 0, 0), force=(1e-5, 0, 0)), None)
              for k in range(2)]
    calls = [8, 8, 16, 8, 35, 4, 800, 9]
    with capi.Batch(capi.STORE_F32) as b:
        ms = [b.add(*s) for s in specs]
        for n in calls:
            b.step(n, 8)
        b.synchronize()
        got = [m.populations() for m in ms]
    for s, g in zip(specs, got):
        assert np.array_equal(g, run_alone(*s, sum(calls)))
