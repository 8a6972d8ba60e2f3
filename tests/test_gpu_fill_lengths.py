"""Gap filling where a frame's entries per thread step into the next loop: one
workgroup of 1024 threads takes 1, 2, 4, 8 or up to 19 entries a thread.  The
missing pixels are scattered (no thread's entries are its neighbours'), in
frames of one call.  The oracle's sparse direct solve bounds the result as in
test_gpu_prefilter.py: 1e-9 of the frame's maximum in FP64."""
import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import prefilter as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1, 31, 1023), (1024, 1025, 2047), (2048, 2049, 4095), (4096, 4097, 5000),
                                    (8191, 8192, 8193)])
def test_lengths(counts):
    rng = np.random.default_rng(11)
    a = 200 + 800 * rng.random((110, 130, len(counts)))
    for f, n in enumerate(counts):
        gone = rng.permutation(110 * 130)[:n]
        a[gone % 110, gone // 110, f] = np.nan
    got, ref = ssa.imgapfill_leastsquares(a), P.imgapfill_leastsquares(a)
    err = np.abs(got - ref).max(axis=(0, 1)) / 1000
    print(f"{counts}: {err}", flush=True)
    assert np.isfinite(got).all() and err.max() <= 1e-9
