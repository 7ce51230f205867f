"""Copies between host arrays and the GPU through the pinned slots: what goes
up comes down unchanged, for sizes around the direct copy's limit, one chunk,
the ring of slots and the threaded copies, from several threads at once, and
the moments' two arrays (which share their chunks) equal the direct
read-back's."""
import ctypes
import sys
import threading
import time

import numpy as np
import pytest

from latticeboltzmanncuda_amd import capi

pytestmark = pytest.mark.gpu

# nodes of a D3Q27 FP32 lattice (108 bytes each): 64 KiB, 512 KiB, 8 chunks of
# 512 KiB, 8 MiB, 32 MiB, each from both sides
NODES = [1, 606, 607, 4854, 4855, 38836, 38837, 77672, 77673, 310689, 310690,
         500009]


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def round_trip(n, seed):
    f = np.random.default_rng(seed).random(27 * n, np.float32)
    with capi.Context(capi.make_config(n, 1, 1, lattice=27,
                                       mode=capi.MODE_REFERENCE)) as c:
        c.set_populations(f)
        assert np.array_equal(c.populations(), f)
        pts = c.download_points()
        assert np.array_equal(pts["f"], f.reshape(27, n).T)
        pts["f"] += 1
        c.upload_points(pts)
        again = c.download_points()
        assert np.array_equal(again["f"], pts["f"])


@pytest.mark.parametrize("n", NODES)
def test_round_trip(n):
    say(f"case: transfer round trip, {n} nodes")
    round_trip(n, n)


def test_round_trips_of_several_threads():
    say("case: transfers of 4 threads")
    errors = []

    def work(k):
        try:
            for n in (5000 + k, 90000 + k, 1000 + k, 40000 + k):
                round_trip(n, k)
        except BaseException as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("dims", [(3, 1000), (31, 1057), (700, 751),
                                  (1500, 1301)])
def test_moments_pieces(dims):
    say(f"case: moments in pieces {dims}")
    n = dims[0] * dims[1]
    with capi.Context(capi.make_config(*dims, 1, lattice=capi.D2Q9, tau=0.8,
                                       periodic=(1, 1, 0))) as c:
        rng = np.random.default_rng(1)
        u = 0.02 * (rng.random((3, n)) - 0.5)
        u[2] = 0
        c.init_equilibrium(1.0 + 0.01 * rng.random(n), u)
        c.step(3)
        rho, vel = c.moments()
        r2 = np.zeros(n, np.float32)
        v2 = np.zeros(3 * n, np.float32)
        capi.check(c.lib.lbm_moments_noalloc(c.h, r2.ctypes.data,
                                             v2.ctypes.data), "noalloc")
        assert np.array_equal(rho, r2) and np.array_equal(vel.ravel(), v2)
        v3 = np.zeros(3 * n, np.float32)
        capi.check(c.lib.lbm_moments(c.h, None, v3.ctypes.data), "moments")
        assert np.array_equal(v2, v3)


def hip():
    """The HIP runtime that the library runs on."""
    capi.load()
    with open("/proc/self/maps") as fh:
        path = next(l.split()[-1] for l in fh if "libamdhip64" in l)
    return ctypes.CDLL(path)


def flat(nbytes):
    """A lattice whose moments fill so many bytes."""
    return capi.make_config(1024, nbytes // 16 // 1024, 1, lattice=capi.D2Q9,
                            tau=0.8, periodic=(1, 1, 0))


@pytest.mark.parametrize("kind", ["pinned", "managed"])
def test_memory_of_the_runtime_is_copied_directly(kind):
    # a result (and an upload) in pinned memory takes as long as the runtime's
    # own copy of it, not the detour through the library's pinned slots
    say(f"case: {kind} host memory")
    rt, nbytes = hip(), 256 << 20
    p = ctypes.c_void_p()
    size = ctypes.c_size_t(nbytes)
    if kind == "pinned":
        assert rt.hipHostMalloc(ctypes.byref(p), size, 0) == 0
    else:
        assert rt.hipMallocManaged(ctypes.byref(p), size, 1) == 0
    try:
        with capi.Context(flat(nbytes)) as c:
            c.init_equilibrium(1.0 + 0.01 * np.random.default_rng(3).random(c.n))
            c.step(2)
            want = c.moments()
            got = np.frombuffer((ctypes.c_float * (4 * c.n)).from_address(
                p.value), np.float32)
            got[:] = 0  # the CPU holds its pages
            best = 1e9
            for _ in range(4):
                c.synchronize()
                t0 = time.perf_counter()
                capi.check(c.lib.lbm_moments(c.h, p, p.value + 4 * c.n),
                           "moments")
                best = min(best, time.perf_counter() - t0)
            assert np.array_equal(got[:c.n], want[0])
            assert np.array_equal(got[c.n:].reshape(3, -1), want[1])
            if kind == "pinned":
                d = ctypes.c_void_p()
                assert rt.hipMalloc(ctypes.byref(d), size) == 0
                direct = 1e9
                for _ in range(4):
                    t0 = time.perf_counter()
                    assert rt.hipMemcpy(p, d, size, 2) == 0
                    direct = min(direct, time.perf_counter() - t0)
                rt.hipFree(d)
                say(f"  moments {best * 1e3:.2f} ms, copy alone "
                    f"{direct * 1e3:.2f}")
                assert best < 1.35 * direct + 3e-4
        f = np.frombuffer((ctypes.c_float * (nbytes // 4)).from_address(
            p.value), np.float32)
        n = nbytes // 108
        f[:27 * n] = np.random.default_rng(4).random(27 * n, np.float32)
        with capi.Context(capi.make_config(n, 1, 1, lattice=27,
                                           mode=capi.MODE_REFERENCE)) as c:
            capi.check(c.lib.lbm_set_populations_f32(c.h, p), "populations")
            assert np.array_equal(c.populations(), f[:27 * n])
    finally:
        (rt.hipHostFree if kind == "pinned" else rt.hipFree)(p)


def test_threads_sleep_while_the_gpu_steps():
    # a result behind queued steps: the copy's threads touch its pages and
    # sleep until its first chunk is there (they kept six CPUs busy)
    say("case: CPU time of a read-back behind queued steps")
    with capi.Context(flat(256 << 20)) as c:
        c.init_equilibrium()
        c.step(40)
        want = c.moments()
        c.step(2400)
        t0, p0 = time.perf_counter(), time.process_time()
        got = c.moments()
        wall, cpu = time.perf_counter() - t0, time.process_time() - p0
    say(f"  {cpu:.3f} s of CPU in {wall:.3f} s")
    assert wall > 0.1  # the steps were still under way
    assert cpu < 2.5 * wall
    assert np.array_equal(got[0], want[0])  # rest stays at rest


@pytest.mark.parametrize("nbytes", [200 << 10, 9 << 20])
def test_more_threads_than_slots(nbytes):
    say(f"case: 12 threads read {nbytes >> 10} KiB each")
    cs = [capi.Context(flat(nbytes)) for _ in range(12)]
    want, errors = [], []
    for k, c in enumerate(cs):
        c.init_equilibrium(np.full(c.n, 1.0 + 0.001 * k))
        want.append(np.float32(c.moments()[0][0]))

    def work(k):
        try:
            for _ in range(6):
                rho, u = cs[k].moments()
                assert (rho == want[k]).all() and (u == 0).all()
        except BaseException as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(12)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for c in cs:
        c.close()
    assert not errors, errors
