"""The moment calls' way to the host: a small lattice's planes cross in one
copy, and what a call keeps on the device is bounded."""
import gc
import threading
import time

import numpy as np
import pytest

from chemsim_amd import Context, Lattice, Params, capi
from chemsim_amd import workloads as W
from chemsim_amd.batch import Batch

pytestmark = pytest.mark.gpu


def _median_us(call, n=300):
    call()
    t = []
    for _ in range(n):
        t0 = time.perf_counter()
        call()
        t.append(time.perf_counter() - t0)
    return 1e6 * float(np.median(t))


def test_small_planes_take_one_copy(ctx):
    """Three planes of 16 x 16 cost about what one costs (25 us; with a copy
    and its latency per plane they took twice as long)."""
    n = 16
    ptr = lambda a: a.ctypes.data_as(capi.C.c_void_p)  # noqa: E731
    f32, f64 = np.empty((3, n, n), np.float32), np.empty((3, n, n))
    with Lattice(ctx, n, n, "f32", Params(tau=0.8)) as lat, Batch(ctx, [(n, n)], "f32") as b:
        lat.init_equilibrium(*W.rest_state(n, n))
        b.init_equilibrium(0, *W.rest_state(n, n))
        one = _median_us(lambda: capi.call("cs_lattice_density", lat.handle, ptr(f32[0])))
        three = _median_us(lambda: capi.call("cs_lattice_moments_f64", lat.handle, *(ptr(p) for p in f64)))
        batch = _median_us(lambda: capi.call("cs_batch_moments", b.handle, 0, *(ptr(p) for p in f32)))
    print(f"one plane {one:.1f} us, three {three:.1f} us, of a batch {batch:.1f} us")
    assert three < 1.5 * one and batch < 1.5 * one


@pytest.mark.parametrize("n", [1, 255, 256, 257, 313, 443, 512])
def test_planes_together_or_one_by_one(ctx, n):
    """Either side of the bytes up to which planes cross together: every plane
    lands in its own array, in the f32 and in the f64 calls."""
    rng = np.random.default_rng(5)
    rho = (1 + 0.01 * rng.standard_normal((n, n))).astype(np.float32)
    u = (0.03 * rng.standard_normal((2, n, n))).astype(np.float32)
    with Lattice(ctx, n, n, "f32", Params(tau=0.8)) as lat, Batch(ctx, [(n, n)], "f32") as b:
        lat.init_equilibrium(rho, u[0], u[1])
        b.init_equilibrium(0, rho, u[0], u[1])
        f64 = lat.moments_f64()
        ux, uy = lat.velocity()
        for got in ((lat.density(), ux, uy), b.moments(0), (lat.density(), *b.velocity(0))):
            for g, ref in zip(got, f64):
                np.testing.assert_array_equal(g, ref.astype(np.float32))
    np.testing.assert_allclose(f64[0], rho, rtol=1e-5)
    np.testing.assert_allclose(f64[1:], u, atol=1e-6)


def _free_bytes():
    free, total = capi.C.c_size_t(), capi.C.c_size_t()
    hip = capi.C.CDLL("libamdhip64.so")
    assert hip.hipMemGetInfo(capi.C.byref(free), capi.C.byref(total)) == 0
    return free.value


def test_calls_keep_bounded_buffers_per_context(ctx):
    """Reading 40 lattices of 1024 x 512 and a batch keeps at most the 64 MiB
    that one context's handles share (12.6 MB for each would be 500 MB), and
    gives it back with the last handle."""
    w, h = 1024, 512
    other = Context(0)
    lats = [Lattice(other, w, h, "f32", Params(tau=0.8)) for _ in range(40)]
    batch = Batch(other, [(w, h)] * 3, "f32")
    rest = W.rest_state(w, h)
    for lat in lats:
        lat.init_equilibrium(*rest)
    for i in range(3):
        batch.init_equilibrium(i, *rest)
    lats[0].sync()
    gc.collect()
    before = _free_bytes()
    for lat in lats:
        lat.moments_f64()
    for i in range(3):
        batch.moments(i)
    kept = before - _free_bytes()
    print(f"kept {kept / 2**20:.1f} MiB")
    assert kept <= (64 + 4) << 20  # and the allocator's granularity
    big = Lattice(other, 2200, 2200, "f32", Params(tau=0.8))  # 116 MB of planes: allocated for the call
    with_big = _free_bytes()
    big.moments_f64()
    assert with_big - _free_bytes() <= 4 << 20
    for x in (*lats, batch, big):
        x.close()
    assert _free_bytes() >= before + 40 * 2 * 9 * 4 * w * h


def test_moment_calls_from_several_threads(ctx):
    """Lattices of one context read from several threads at once, each call from a
    buffer of its own."""
    n, sides = 6, [64, 200, 333, 128, 512, 257]
    lats, want = [], []
    rng = np.random.default_rng(9)
    for s in sides:
        lat = Lattice(ctx, s, s, "f32", Params(tau=0.8))
        lat.init_equilibrium((1 + 0.01 * rng.standard_normal((s, s))).astype(np.float32),
                             *(0.03 * rng.standard_normal((2, s, s))).astype(np.float32))
        lats.append(lat)
        want.append((lat.density(), *lat.velocity(), *lat.moments_f64()))
    errors = []

    def read(k):
        try:
            for _ in range(40):
                got = (lats[k].density(), *lats[k].velocity(), *lats[k].moments_f64())
                for g, r in zip(got, want[k]):
                    np.testing.assert_array_equal(g, r)
        except BaseException as e:  # reported below
            errors.append((k, repr(e)[:300]))

    threads = [threading.Thread(target=read, args=(k,)) for k in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for lat in lats:
        lat.close()
    assert not errors, errors


def test_threads_do_not_allocate_per_call(ctx):
    """Six threads that read their own lattices again and again find their buffers
    kept: the device's free memory never grows meanwhile (with one kept buffer for
    all, the other five allocated and freed theirs in every call)."""
    n, side = 6, 512
    other = Context(0)
    lats = [Lattice(other, side, side, "f32", Params(tau=0.8)) for _ in range(n)]
    rest = W.rest_state(side, side)
    for lat in lats:
        lat.init_equilibrium(*rest)
        lat.velocity()
    gc.collect()  # handles that earlier tests dropped free their memory now
    start, stop = threading.Barrier(n), threading.Event()
    seen = [_free_bytes()]

    def read(k):
        start.wait()
        for _ in range(200):
            lats[k].velocity()

    def watch():
        while not stop.is_set():
            seen.append(_free_bytes())

    watcher = threading.Thread(target=watch)
    watcher.start()
    threads = [threading.Thread(target=read, args=(k,)) for k in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    stop.set()
    watcher.join()
    for lat in lats:
        lat.close()
    assert len(seen) > 20
    assert all(b <= a for a, b in zip(seen, seen[1:])), sorted(set(seen))
