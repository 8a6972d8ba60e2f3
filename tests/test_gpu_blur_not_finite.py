"""Blurred stacks of which some frames hold a NaN or an infinity: the full
circular convolution spreads a NaN over its frame, and an infinity over all
outputs whose tap is not 0 (NaN where it is), and leaves the other frames of
the stack alone.  The reference is the convolution's two circulant matrix
products in numpy, bounds as in test_gpu_prefilter.py: 1e-12 of the frame's
maximum in FP64, one rounding in FP32.

A stack in which every frame is like that costs what its arithmetic costs.
The sweep takes about 1.3 us a 512x512 float32 frame, storing NaNs less than
one, the products 21 us: bounds of 4 and 50 times the finite stack's time hold
with a factor of 2 to spare.  (Blurred one frame at a time it is 170 times.)"""
import ctypes
import math
import time

import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import prefilter as P
from steadyscan_amd import _native as N

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu


def circulant(n, sigma):
    """n x n matrix of the wrapped Gaussian on the padded period."""
    s = n + P.gauss_pad(sigma)
    d = np.minimum(np.arange(s), s - np.arange(s)).astype(float)
    g = np.exp(-d * d / (2 * sigma ** 2))
    return (g / g.sum())[np.subtract.outer(np.arange(n), np.arange(n)) % s]


def blurred(a, sigma):
    with np.errstate(invalid="ignore"):
        rows = (circulant(a.shape[0], sigma)[:, :, None] * a[None, :, :]).sum(axis=1)
        return (rows[:, None, :] * circulant(a.shape[1], sigma)[None, :, :]).sum(axis=2)


def stack(h, w, dtype, seed):
    a = (200 + 800 * np.random.default_rng(seed).random((h, w, 9))).astype(dtype)
    a[h // 2, w // 3, 1] = np.nan
    a[0, 0, 2] = np.inf
    a[h - 1, w - 1, 4] = -np.inf
    a[3, 4, 5], a[3, 5, 5] = np.inf, -np.inf
    a[5, 6, 6], a[6, 5, 6] = np.nan, np.inf
    a[:, :, 8] = np.nan
    return np.asfortranarray(a)


def check(got, a, sigma):
    for f in range(a.shape[2]):
        ref = blurred(a[:, :, f].astype(np.float64), sigma)
        assert np.array_equal(np.isnan(got[:, :, f]), np.isnan(ref)), f
        assert np.array_equal(np.isinf(got[:, :, f]), np.isinf(ref)), f
        ok = np.isfinite(ref)
        d = np.abs(got[:, :, f][ok] - ref[ok])
        assert d.size == 0 or np.all(d <= (1e-9 if a.dtype == np.float64 else 1e-9 + np.spacing(np.abs(got[:, :, f][ok]))))
        inf = np.isinf(ref)
        assert np.array_equal(got[:, :, f][inf], ref[inf]), f


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("h,w,sigma", [(70, 45, 1.0), (130, 100, 0.6)])
def test_mixed_stack(h, w, sigma, dtype):
    a = stack(h, w, dtype, 1)
    check(ssa.prefilter_foralignment(a, sigma, False), a, sigma)


def test_mixed_stack_on_the_device(handle):
    a = stack(70, 45, np.float32, 2)
    flat = a.ravel(order="F")
    src, dst = DeviceBuffer(flat.nbytes), DeviceBuffer(flat.nbytes)
    src.upload(flat)
    for out in (dst, src):  # out of place, then in place
        assert N.lib().ss_prefilter(handle.ptr, N.SS_F32, ctypes.c_void_p(src.ptr.value),
                                    ctypes.c_void_p(out.ptr.value), 70, 45, 9, 1.0, 0, 1) == 0
        check(out.download(np.float32, flat.size).reshape(a.shape, order="F"), a, 1.0)
    src.free(), dst.free()


def test_median_of_a_mixed_stack():
    a = stack(40, 50, np.float64, 3)
    got = ssa.prefilter_foralignment(a, 1.0, True)
    for f in range(a.shape[2]):
        if np.isnan(a[:, :, f]).any():
            assert np.isnan(got[:, :, f]).all()
        elif np.isfinite(a[:, :, f]).all():
            ref = P.prefilter_foralignment(a[:, :, f], 1.0, True)
            assert np.abs(got[:, :, f] - ref).max() <= 1e-12 * np.abs(ref).max()
        else:
            ref = blurred(a[:, :, f], 1.0)
            med = np.nan if np.isnan(ref).any() else np.median(ref)
            with np.errstate(invalid="ignore"):
                assert np.array_equal(np.isnan(got[:, :, f]), np.isnan(ref / med))


@pytest.mark.parametrize("bad,factor", [(math.nan, 4), (math.inf, 50)])
def test_time_of_a_stack_without_finite_frames(handle, bad, factor):
    n, size = 100, 512
    a = (200 + 800 * np.random.default_rng(4).random((n, size * size), dtype=np.float32))
    src, dst = DeviceBuffer(a.nbytes), DeviceBuffer(a.nbytes)

    def best():
        t = []
        for _ in range(4):
            t0 = time.perf_counter()
            assert N.lib().ss_prefilter(handle.ptr, N.SS_F32, ctypes.c_void_p(src.ptr.value),
                                        ctypes.c_void_p(dst.ptr.value), size, size, n, 1.0, 0, 1) == 0
            t.append(time.perf_counter() - t0)
        return min(t)

    src.upload(a)
    finite = best()
    a[:, 1000] = bad
    src.upload(a)
    t = best()
    print(f"finite {finite * 1e6:.0f} us, {bad} in every frame {t * 1e6:.0f} us", flush=True)
    src.free(), dst.free()
    assert t <= factor * finite
