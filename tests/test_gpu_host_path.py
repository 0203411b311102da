"""The host-buffer entry points (cfft_fwd_host, cfft_inv_host,
cfft_fwd_monomial_host, cfft128_*_host) against the device-buffer ones, bit
for bit.  Calls of at most 64 KiB run their kernels on the pinned staging
buffer itself, larger ones copy through a device buffer, and batches above
64 MiB run in chunks; the cases sit on both sides of each limit."""
import numpy as np
import pytest

from cfft_amd import DeviceBuffer, fft128, ordered, unordered
from cfft_amd.ordered import FftAlgo


def _rand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _both(plan, x, fwd):
    h = x.copy()
    (plan.fwd if fwd else plan.inv)(h)
    d = DeviceBuffer.from_host(x)
    (plan.fwd if fwd else plan.inv)(d)
    return h, d.download()


@pytest.mark.gpu
@pytest.mark.parametrize("n,base_n,batch", [
    (1024, 1024, 1),     # 16 KiB: on the pinned buffer
    (1024, 1024, 4),     # 64 KiB: the largest call on the pinned buffer
    (1024, 1024, 5),     # through a device buffer
    (4096, 512, 1),      # two-level plan on the pinned buffer
    (65536, 1024, 1),    # 1 MiB through a device buffer
    (1024, 1024, 4100),  # 64 MiB + 64 KiB: two chunks
])
def test_unordered_host_equals_device(cfft, n, base_n, batch):
    print("host path: unordered n=%d base=%d batch=%d" % (n, base_n, batch), flush=True)
    plan = unordered.Plan(n, unordered.Method.UserProvided(FftAlgo.Dif16, base_n))
    rng = np.random.default_rng(n + batch)
    x = _rand(rng, batch, n) if batch > 1 else _rand(rng, n)
    for fwd in (True, False):
        h, d = _both(plan, x, fwd)
        assert np.array_equal(h.view(np.uint64), d.view(np.uint64))


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(256, 1), (1024, 8), (16384, 1)])
def test_ordered_host_equals_device(cfft, n, batch):
    print("host path: ordered n=%d batch=%d" % (n, batch), flush=True)
    plan = ordered.Plan(n, ordered.Method.UserProvided(FftAlgo.Dit4), large=True)
    rng = np.random.default_rng(n)
    x = _rand(rng, batch, n) if batch > 1 else _rand(rng, n)
    for fwd in (True, False):
        h, d = _both(plan, x, fwd)
        assert np.array_equal(h.view(np.uint64), d.view(np.uint64))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1024, 8192])
def test_fwd_monomial_host_equals_device(cfft, n):
    print("host path: fwd_monomial n=%d" % n, flush=True)
    plan = unordered.Plan(n, unordered.Method.UserProvided(FftAlgo.Dif4, min(n, 1024)))
    for degree in (0, 1, n // 3, n - 1):
        m = np.full(n, np.nan, dtype=np.complex128)  # every point is written
        plan.fwd_monomial(degree, m)
        d = DeviceBuffer.from_host(np.zeros(n, dtype=np.complex128))
        plan.fwd_monomial(degree, d)
        assert np.array_equal(m.view(np.uint64), d.download().view(np.uint64))


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(1024, 1), (1024, 3), (4096, 2)])
def test_fft128_host_equals_device(cfft, n, batch):
    print("host path: fft128 n=%d batch=%d" % (n, batch), flush=True)
    plan = fft128.Plan(n)
    rng = np.random.default_rng(n * batch)
    shape = (batch, n) if batch > 1 else (n,)
    hi = [rng.standard_normal(shape) for _ in range(2)]
    lo = [h * 2.0 ** -60 * rng.standard_normal(shape) for h in hi]
    arrs = [hi[0], lo[0], hi[1], lo[1]]
    for fwd in (True, False):
        h = [a.copy() for a in arrs]
        (plan.fwd if fwd else plan.inv)(*h)
        d = [DeviceBuffer.from_host(a.copy()) for a in arrs]
        (plan.fwd if fwd else plan.inv)(*d)
        for a, b in zip(h, d):
            assert np.array_equal(a.view(np.uint64), b.download().view(np.uint64))


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(64, 1), (64, 7), (64, 512), (64, 513), (128, 5), (256, 3),
                                     (512, 2), (1024, 1), (1024, 64), (1024, 65), (1024, 256),
                                     (1024, 257), (8192, 3)])
@pytest.mark.parametrize("algo", list(FftAlgo))
def test_polled_host_calls_equal_device(cfft, n, batch, algo):
    """Host calls of up to 4 MiB: groups of transforms partly filled, the most
    workgroups that report to the polling host (64: 512 transforms of 64 points,
    64 of 1024) and one transform more, the largest call on the pinned buffer
    (256 transforms of 1024 points) and one through a device buffer; several
    calls in a row on one slot; both directions."""
    print("host path: polled n=%d batch=%d %s" % (n, batch, algo.name), flush=True)
    plan = ordered.Plan(n, ordered.Method.UserProvided(algo), large=True)
    rng = np.random.default_rng(n + batch)
    for fwd in (True, False, True):
        x = _rand(rng, batch, n)
        h, d = _both(plan, x, fwd)
        assert np.array_equal(h.view(np.uint64), d.view(np.uint64))


@pytest.mark.gpu
def test_polled_host_calls_from_threads(cfft):
    """Threads sharing a plan each poll a slot of their own."""
    import threading
    print("host path: threads", flush=True)
    plan = unordered.Plan(1024, unordered.Method.UserProvided(FftAlgo.Dif16, 512))
    rng = np.random.default_rng(5)
    xs = [_rand(rng, 3, 1024) for _ in range(4)]
    want = [_both(plan, x, True)[1] for x in xs]
    bad = []

    def work(x, w):
        for _ in range(50):
            h = x.copy()
            plan.fwd(h)
            if not np.array_equal(h.view(np.uint64), w.view(np.uint64)):
                bad.append(1)

    ts = [threading.Thread(target=work, args=a) for a in zip(xs, want)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
