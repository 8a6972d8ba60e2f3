"""Gap filling at the edges of what a workgroup holds: up to 19456 missing
pixels run in LDS and registers, larger regions stream the rest.  The oracle's
sparse direct solve bounds the result as in test_gpu_prefilter.py: 1e-9 of
the frame's maximum in FP64, one rounding in FP32."""
import ctypes

import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import prefilter as P
from steadyscan_amd import _native as N

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu


def frame(h, w, first, count, seed=1):
    """Pixels first .. first + count of the column-major frame are missing."""
    a = 200 + 800 * np.random.default_rng(seed).random(h * w)
    a[first:first + count] = np.nan
    return np.asfortranarray(a.reshape((h, w), order="F"))


@pytest.mark.parametrize("count", [1, 63, 1024, 1025, 8192, 19455, 19456, 19457, 20481, 23000])
def test_sizes(count):
    a = frame(160, 200, 1611, count)
    got, ref = ssa.imgapfill_leastsquares(a), P.imgapfill_leastsquares(a)
    err = np.abs(got - ref).max() / 1000
    print(f"{count} missing: {err:.2e}", flush=True)
    assert np.isfinite(got).all() and err <= 1e-9


def test_sizes_in_one_call_in_place(handle):
    """Frames of every size in one launch, filled in place and out of place
    on the device, equal each frame filled alone."""
    counts = [0, 300, 19456, 19500]
    f = [frame(160, 200, 1611, c, seed=c).astype(np.float32) for c in counts]
    alone = np.concatenate([ssa.imgapfill_leastsquares(x).ravel(order="F") for x in f])
    flat = np.concatenate([x.ravel(order="F") for x in f])
    src, dst = DeviceBuffer(flat.nbytes), DeviceBuffer(flat.nbytes)
    src.upload(flat)
    for out in (dst, src):
        assert N.lib().ss_fill_gaps(handle.ptr, N.SS_F32, ctypes.c_void_p(src.ptr.value),
                                    ctypes.c_void_p(out.ptr.value), 160, 200, len(f), 1) == 0
        assert np.array_equal(out.download(np.float32, flat.size), alone)
