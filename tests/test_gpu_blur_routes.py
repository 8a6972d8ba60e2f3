"""The blur's two routes and the sweep's segments of several column blocks.

A stack of many frames leaves a workgroup several 32-column blocks, whose ring
of columns wraps and is refilled; a frame by itself is cut into one block each.
Both make the same sums, and the route does not depend on the number of
frames, so that a frame's result is the same to the bit.  The oracle bounds it
as in test_gpu_prefilter.py: 1e-12 of the frame's maximum in FP64.

A kernel wide enough takes the GEMMs whatever the frame's size; a narrower one
takes them or the sweep, whichever is less work, and so never takes much
longer.  Medians of calls of 60 to 120 us differ by a few percent: bound at a
fifth.  (The sweep of 48x48 and 65x65 frames at 6 takes 1.5 times as long.)"""
import ctypes
import time

import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import prefilter as P
from steadyscan_amd import _native as N

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,n,sigma,dtype", [
    (64, 300, 1040, 0.7, np.float32),   # one segment of 10 blocks, the last one of 12 columns
    (40, 170, 1040, 4.0, np.float32),   # a ring wider than the rows' tile
    (64, 300, 400, 1.0, np.float64),    # two segments of 5 blocks
    (130, 200, 150, 6.0, np.float64),   # three strips, 4 + 3 blocks
    (65, 257, 256, 6.9, np.float64),    # 61 taps a side
    (64, 300, 400, 2.0, np.uint16),
    (48, 48, 300, 6.0, np.float64),     # by the GEMMs
])
def test_a_frame_alone_and_in_a_stack(h, w, n, sigma, dtype):
    rng = np.random.default_rng(h + w)
    a = np.asfortranarray(np.round(200 + 800 * rng.random((h, w, n), dtype=np.float32)).astype(dtype))
    got = ssa.prefilter_foralignment(a, sigma, False)
    for f in (0, n // 2, n - 1):
        ref = P.prefilter_foralignment(a[:, :, f], sigma, False)
        assert np.array_equal(got[:, :, f], ssa.prefilter_foralignment(a[:, :, f], sigma, False)), f
        if dtype == np.float64:
            assert np.abs(got[:, :, f] - ref).max() <= 1e-12 * np.abs(a).max()
        elif dtype == np.float32:
            assert np.all(np.abs(got[:, :, f] - ref) <= np.spacing(np.abs(ref)))
        else:
            d = np.abs(got[:, :, f].astype(np.int64) - ref.astype(np.int64))
            assert d.max() <= 1 and np.count_nonzero(d) <= 2


@pytest.mark.parametrize("dtype,sigma", [(np.uint16, 0.9), (np.int16, 2.4), (np.uint16, 6.9)])
def test_integers_round_half_away_from_zero(dtype, sigma):
    """Both are the same doubles to FP64 rounding: at most a tie differs."""
    a = (np.round(1000 * np.random.default_rng(5).standard_normal((150, 130, 3))).astype(dtype)
         if dtype == np.int16 else np.round(800 * np.random.default_rng(5).random((150, 130, 3))).astype(dtype))
    d = ssa.prefilter_foralignment(a, sigma, False).astype(np.int64) - P.prefilter_foralignment(a, sigma, False)
    assert np.abs(d).max() <= 1 and np.count_nonzero(d) <= 2


@pytest.mark.parametrize("size", [48, 65, 100])
def test_a_narrower_kernel_takes_no_longer(handle, size):
    n = 512
    a = np.random.default_rng(6).integers(0, 1000, (n, size * size), dtype=np.uint16)
    src, dst = DeviceBuffer(a.nbytes), DeviceBuffer(a.nbytes)
    src.upload(a)

    def median(sigma):
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            assert N.lib().ss_prefilter(handle.ptr, N.SS_U16, ctypes.c_void_p(src.ptr.value),
                                        ctypes.c_void_p(dst.ptr.value), size, size, n, sigma, 0, 1) == 0
            t.append(time.perf_counter() - t0)
        return sorted(t)[len(t) // 2]

    widest = median(40.0)
    times = {s: median(s) for s in (1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 10.0)}
    print(f"{size}: sigma 40 {widest * 1e6:.0f} us,", {s: round(t * 1e6) for s, t in times.items()}, flush=True)
    src.free(), dst.free()
    assert max(times.values()) <= 1.2 * widest
