"""cfft_external_product_noalloc through the C ABI: the same bits as
cfft_external_product on two calls in a row (the second smaller), batches
that need several passes over the fixed 32 MiB scratch (where the split form
runs: the one-launch form, k1 = 2 ... 4 on Dif16 plans, uses none of it), no
device memory taken by the calls, and a GLWE too large for the scratch
refused."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

M = 2**64
K1, LEVELS, BASE_LOG = 2, 3, 8


def _setup(N, algo, base_n, seed, k1=K1):
    from cfft_amd import products
    from cfft_amd.device import DeviceBuffer
    from cfft_amd.unordered import FftAlgo, Method, Plan
    rng = np.random.default_rng(seed)
    plan = Plan(N // 2, Method.UserProvided(FftAlgo(algo), base_n))
    key = rng.integers(0, M, (k1 * LEVELS, k1, N), dtype=np.uint64)
    dk = DeviceBuffer.from_host(key)
    kf = DeviceBuffer((k1 * LEVELS, k1, N // 2), np.complex128)
    products.ggsw_to_fourier(plan, dk, k1, LEVELS, kf)
    return rng, plan, kf


def _both(plan, kf, glwe, stream):
    """(noalloc result, cfft_external_product result) for the same GLWEs."""
    from cfft_amd import check, lib
    from cfft_amd.device import DeviceBuffer
    batch, k1 = glwe.shape[:2]
    dg = DeviceBuffer.from_host(glwe)
    o1 = DeviceBuffer(glwe.shape, np.uint64)
    o2 = DeviceBuffer(glwe.shape, np.uint64)
    check(lib.cfft_external_product_noalloc(plan.handle, kf.dptr, k1, LEVELS, BASE_LOG, dg.dptr,
                                            o1.dptr, batch, stream.handle))
    stream.synchronize()
    r1 = o1.download()
    check(lib.cfft_external_product(plan.handle, kf.dptr, k1, LEVELS, BASE_LOG, dg.dptr, o2.dptr,
                                    batch, stream.handle))
    stream.synchronize()
    return r1, o2.download()


@pytest.mark.parametrize("N,algo,base_n,first,second,k1", [
    (4096, 6, 1024, 400, 37, 2),  # the one-launch form: one pass each
    (2048, 6, 1024, 700, 5, 2),
    (1024, 6, 512, 9, 3, 2),
    (2048, 2, 64, 50, 7, 2),      # generic split kernels (Dif4 plan): one pass each
    (4096, 6, 1024, 200, 37, 5),  # wave-local split kernels, 68 GLWEs per pass: 3 passes, then 1
    (2048, 6, 1024, 700, 5, 1),   # 682 per pass: 2 passes, then 1
    (1024, 6, 512, 600, 3, 5),    # 273 per pass: 3 passes, then 1
    (2048, 2, 64, 700, 7, 2),     # generic split kernels, 341 per pass: 3 passes, then 1
])
def test_noalloc_equals_allocating_entry_point(cfft, N, algo, base_n, first, second, k1):
    from cfft_amd import lib
    from cfft_amd.device import Stream
    assert lib.cfft_noalloc_scratch_bytes() == 32 << 20
    rng, plan, kf = _setup(N, algo, base_n, N + first, k1)
    s = Stream()
    for batch in (first, second):
        glwe = rng.integers(0, M, (batch, k1, N), dtype=np.uint64)
        got, want = _both(plan, kf, glwe, s)
        assert np.array_equal(got, want), (N, batch, int(np.sum(got != want)))


@pytest.mark.parametrize("k1,batch", [(2, 600), (5, 240)])  # one launch; split, 4 passes
def test_noalloc_takes_no_device_memory(cfft, k1, batch):
    from cfft_amd import check, lib
    from cfft_amd.device import DeviceBuffer, Stream, mem_info
    rng, plan, kf = _setup(4096, 6, 1024, 5, k1)
    s = Stream()
    glwe = rng.integers(0, M, (batch, k1, 4096), dtype=np.uint64)
    dg = DeviceBuffer.from_host(glwe)
    do = DeviceBuffer(glwe.shape, np.uint64)
    # first call on this device resolves the scratch's address
    check(lib.cfft_external_product_noalloc(plan.handle, kf.dptr, k1, LEVELS, BASE_LOG, dg.dptr,
                                            do.dptr, 1, s.handle))
    s.synchronize()
    free0, _ = mem_info()
    for _ in range(3):
        check(lib.cfft_external_product_noalloc(plan.handle, kf.dptr, k1, LEVELS, BASE_LOG,
                                                dg.dptr, do.dptr, batch, s.handle))
    s.synchronize()
    free1, _ = mem_info()
    # a scratch-cache entry would take at least 32 MiB
    assert free1 >= free0 - (4 << 20), (free0, free1)


def test_noalloc_refuses_oversized_glwe(cfft):
    from cfft_amd import CfftPanic, check, lib
    from cfft_amd.device import DeviceBuffer
    from cfft_amd.unordered import FftAlgo, Method, Plan
    plan = Plan(8192, Method.UserProvided(FftAlgo.Dif16, 1024))
    k1, levels = 64, 5  # 64 * 5 * 8192 * 16 bytes = 40 MiB of spectra per GLWE
    d = DeviceBuffer((16,), np.uint64)
    with pytest.raises(CfftPanic, match="scratch"):
        check(lib.cfft_external_product_noalloc(plan.handle, d.dptr, k1, levels, 8, d.dptr,
                                                d.dptr, 1, None))
