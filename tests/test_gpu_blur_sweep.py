"""The one-sweep blur of ss_prefilter at the edges of its tiles and of its
rule: frames of a few rows and columns, where the taps cover the whole padded
period, sizes around the 64-row strips and 32-column blocks, the widest
kernel that it takes and the first that the GEMMs take, in place and out of
place, and frames with a NaN or an infinity.  Bounds as in
test_gpu_prefilter.py: 1e-12 of the frame's maximum in FP64, one rounding of
the class otherwise."""
import ctypes

import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import prefilter as P
from steadyscan_amd import _native as N

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu


def frames(shape, dtype, seed):
    a = 200 + 800 * np.random.default_rng(seed).random(shape)
    return (np.round(a) if np.issubdtype(np.dtype(dtype), np.integer) else a).astype(dtype)


@pytest.mark.parametrize("shape,sigma", [
    ((1, 1, 1), 1.0), ((2, 3, 2), 1.5), ((8, 40, 1), 4.0), ((63, 33, 2), 0.5), ((64, 32, 1), 1.0), ((65, 31, 3), 2.0),
    ((129, 64, 1), 6.0), ((200, 97, 2), 6.7), ((200, 97, 2), 7.5), ((40, 300, 1), 3.3), ((512, 70, 1), 1.0),
])
def test_sizes_f64(shape, sigma):
    a = frames(shape, np.float64, 1)
    err = np.abs(ssa.prefilter_foralignment(a, sigma, False) - P.prefilter_foralignment(a, sigma, False)).max()
    print(f"{shape} sigma {sigma}: {err / np.abs(a).max():.2e}", flush=True)
    assert err <= 1e-12 * np.abs(a).max()


@pytest.mark.parametrize("dtype", [np.float32, np.uint16, np.int16])
def test_classes(dtype):
    a = frames((70, 45, 2), dtype, 2)
    got, ref = ssa.prefilter_foralignment(a, 2.4, False), P.prefilter_foralignment(a, 2.4, False)
    if dtype == np.float32:
        assert np.all(np.abs(got - ref) <= np.spacing(np.abs(ref)))
    else:
        assert np.abs(got.astype(np.int64) - ref.astype(np.int64)).max() <= 1


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_frames_that_are_not_finite(bad):
    a = frames((70, 45, 3), np.float64, 3)
    a[3, 4, 1] = bad
    got = ssa.prefilter_foralignment(a, 1.0, False)
    ref = P.prefilter_foralignment(a[:, :, ::2], 1.0, False)
    assert not np.isfinite(got[:, :, 1]).any()
    assert np.abs(got[:, :, ::2] - ref).max() <= 1e-12 * 1000


def test_in_place_on_the_device(handle):
    a = np.asfortranarray(frames((100, 80, 2), np.float32, 4))
    ref = ssa.prefilter_foralignment(a, 1.3, False, handle=handle)
    flat = a.ravel(order="F")
    src, dst = DeviceBuffer(flat.nbytes), DeviceBuffer(flat.nbytes)
    src.upload(flat)
    for out in (dst, src):
        assert N.lib().ss_prefilter(handle.ptr, N.SS_F32, ctypes.c_void_p(src.ptr.value),
                                    ctypes.c_void_p(out.ptr.value), 100, 80, 2, 1.3, 0, 1) == 0
        assert np.array_equal(out.download(np.float32, flat.size), ref.ravel(order="F"))
