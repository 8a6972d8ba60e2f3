"""Edges of the pixel kernels that the tests of their row loops leave out: the
correlation of frames of 1024 image columns and more (four runs of rows per
thread), pixels that are not finite before and behind a column's first row
outside the template, and the BF16 gradients in the general row loop."""
import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import oracle as O
from steadyscan_amd import workloads as W

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu


def group(w, lines, dtype, flags, n=4, motion=(6.0, 0.5), seed=71):
    h = 3 * lines
    T = W.make_template(h, w, 60, (2.0, 6.0), offset=10.0, seed=seed)
    dx, dy = W.make_motion(n, h, 0.05, 0.0, motion, seed=seed + 1)
    fr = W.make_frames(T, dx, dy, h, w, dtype, True, seed=seed + 2)
    return W.group_args(T, fr, ssa.init_settings(h, w, T.shape, nknots=4), flags=flags, max_iter=6)


@pytest.mark.parametrize("lines", [8, 12])
@pytest.mark.parametrize("w", [1023, 1024, 1030])
def test_wide_frames(w, lines):
    """Bounds as in test_gpu_corr_runs.py: 1e-9, more columns adding terms to
    sums that are compared after the same cancellation."""
    a = group(w, lines, np.uint16, "DC")
    out = ssa.align_group_to_template(*[a[k] for k in W.ARG_ORDER], nargout=8)
    ref = O.align_group_to_template(a, threads=4)
    m, it = ref["mask"].astype(bool), ref["iterations"]
    assert not m.all() and np.array_equal(out[4].astype(bool).reshape(m.shape), m)
    assert int(out[3]) == it
    assert np.max(np.abs(out[7].ravel()[:it] - ref["iteration_corr"][:it])) <= 1e-9
    assert np.max(np.abs(out[2].ravel() - ref["frame_corr"])) <= 1e-9


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("w", [200, 300, 600])
def test_pixels_that_are_not_finite(w, bad):
    """One such pixel in the last column of a frame, where the motion leaves
    the template, or in the middle, whence it reaches every knot: the group's
    correlations are NaN where the oracle's are, and so are the other frames'."""
    for row in (-3, w * 4):
        a = group(w, 8, np.float32, "DC")
        bm = np.asfortranarray(a["bmData"])
        bm[row, 4] = bad  # frame 1
        a["bmData"] = bm
        out = ssa.align_group_to_template(*[a[k] for k in W.ARG_ORDER], nargout=8)
        ref = O.align_group_to_template(a, threads=4)
        it = ref["iterations"]
        assert int(out[3]) == it
        got, exp = out[7].ravel()[:it], ref["iteration_corr"][:it]
        assert np.array_equal(np.isnan(got), np.isnan(exp))
        assert np.all(np.isnan(exp) | (np.abs(got - exp) <= 1e-9))
        fc, rfc = out[2].ravel()[[0, 2, 3]], np.ravel(ref["frame_corr"])[[0, 2, 3]]
        assert np.array_equal(np.isnan(fc), np.isnan(rfc))
        assert np.all(np.isnan(rfc) | (np.abs(fc - rfc) <= 1e-9))


@pytest.mark.parametrize("w", [40, 300])
def test_bf16_gradients_in_the_general_loop(w):
    """Frames two bytes past a 16-byte boundary take the general loop, whose
    arithmetic is the fast loop's: bit for bit."""
    a = dict(group(w, 16, np.int16, "S", motion=(2.0, 1.5)), template_bf16=True)
    bm = np.asfortranarray(a["bmData"])
    buf = DeviceBuffer(bm.nbytes + 16)
    results = []
    for off in (0, 2):
        raw = np.zeros(bm.nbytes + 16, np.uint8)
        raw[off:off + bm.nbytes] = bm.ravel(order="F").view(np.uint8)
        buf.upload(raw)
        results.append(ssa.align_groups([dict(a, bmData=(buf.ptr.value + off, np.int16))])[0])
    plain = ssa.align_groups([dict(a, template_bf16=False)])[0]
    buf.free()
    assert not np.array_equal(results[0]["knots_x"], plain["knots_x"])  # the gradients are in use
    for k in ("knots_x", "knots_y", "frame_corr", "residrms", "mask"):
        assert np.array_equal(results[0][k], results[1][k]), k
