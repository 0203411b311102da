"""CPU check: a device buffer's batch is counted in whole numbers of any size,
also where its shape holds 32-bit numpy integers."""
import ctypes

import numpy as np
import pytest


class _Calls:
    """Stands in for the library: answers fft_size, records the batch."""

    def __init__(self, n):
        self.n, self.batch = n, []

    def cfft_plan_fft_size(self, handle, out):
        ctypes.cast(out, ctypes.POINTER(ctypes.c_size_t))[0] = self.n
        return 0

    def _transform(self, *args):
        self.batch.append(args[2])
        return 0

    def _transform128(self, *args):
        self.batch.append(args[5])
        return 0

    cfft_fwd = cfft_inv = _transform
    cfft128_fwd = cfft128_inv = _transform128


def _buffer(shape, dtype):
    from cfft_amd.device import DeviceBuffer
    b = DeviceBuffer.__new__(DeviceBuffer)
    b.shape, b.dtype, b.dptr = shape, np.dtype(dtype), 0
    return b


@pytest.mark.parametrize("shape", [(1 << 21, 2048), (np.int32(1 << 21), np.int32(2048)),
                                   (np.int32(1 << 16), np.int32(1 << 16)), (3, np.int16(2048))])
def test_batch_of_a_device_buffer(monkeypatch, shape):
    from cfft_amd import fft128, ordered
    want = int(shape[0]) * int(shape[1]) // 2048
    calls = _Calls(2048)
    monkeypatch.setattr(ordered, "lib", calls)
    monkeypatch.setattr(fft128, "lib", calls)
    plan = ordered._PlanBase()
    plan.handle = 1
    plan.fwd(_buffer(shape, np.complex128))
    plan128 = fft128.Plan.__new__(fft128.Plan)
    plan128.handle = 1
    plan128.inv(*[_buffer(shape, np.float64)] * 4)
    plan.handle = plan128.handle = None  # nothing to destroy
    assert calls.batch == [want, want]
