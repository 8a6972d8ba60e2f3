"""The pixel kernels' two row loops against the FP64 oracle: whole aligned
chunks of 8 lines of one image column with the affine geometry ("fast"), and
every form that has to take the general loop -- lines per knot that are no
multiple of 8 or more than 64, misaligned frames, gradient pairs of their
own, per-pixel geometry -- at column counts around the 256 threads of a
workgroup.  FP64 knots are held to 1e-9 px, the bound of the other parity
tests; FP32 ones to 0.01 px after two iterations."""
import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import oracle as O
from steadyscan_amd import workloads as W

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu


def group(h, w, lines, dtype, flags, n=4, seed=31, **geo):
    T = W.make_template(h, w, 40, (2.0, 6.0), offset=10.0, seed=seed)
    dx, dy = W.make_motion(n, h, 0.05, 0.0, (2.0, 1.5), seed=seed + 1)
    fr = W.make_frames(T, dx, dy, h, w, dtype, True, seed=seed + 2)
    nknots = geo.pop("nknots", None) or h // lines + 1
    geom = ssa.init_settings(h, w, T.shape, nknots=nknots, **geo)
    return W.group_args(T, fr, geom, flags=flags, max_iter=6 if flags == "D" else 2)


def check(a, r):
    ref = O.align_group_to_template(a, threads=4)
    nk, n = a["basex"].shape[1] + 1, a["nsetframes"]
    d = np.concatenate([(r[k] - ref[k]).reshape(n, nk)[:-1].ravel() for k in ("knots_x", "knots_y")])
    rms = float(np.sqrt(np.mean(d ** 2)))
    print(f"knot RMS vs FP64 oracle = {rms:.2e} px", flush=True)
    assert r["iterations"] == ref["iterations"]
    assert rms <= (1e-9 if a["flags"] == "D" else 0.01)
    assert np.mean(r["mask"] == ref["mask"].astype(bool)) >= (0.99999 if a["flags"] == "D" else 0.999)


@pytest.mark.parametrize("h,w,lines,dtype,flags", [
    (32, 16, 8, np.uint16, "D"),     # one chunk per column
    (48, 65, 16, np.int16, "D"),     # a wave and one column
    (32, 257, 16, np.float32, "D"),  # one column past a workgroup's threads
    (32, 300, 8, np.float64, "D"),
    (64, 256, 64, np.uint16, "D"),   # the longest run
    (64, 40, 16, np.float64, "S"),
    (60, 50, 12, np.uint16, "D"),    # chunks of 8 and 4 lines
    (36, 70, 4, np.float32, "D"),    # half a chunk
    (144, 24, 72, np.int16, "D"),    # more lines than a run holds
    (35, 33, 7, np.uint16, "S"),
])
def test_lines_and_columns(h, w, lines, dtype, flags):
    a = group(h, w, lines, dtype, flags)
    check(a, ssa.align_groups([a])[0])


@pytest.mark.parametrize("form", ["gradients", "bidirectional", "between_lines"])
def test_general_forms(form):
    if form == "gradients":  # not the template's forward differences
        a = group(48, 40, 16, np.uint16, "D")
        a["xgrad"], a["ygrad"] = a["xgrad"] * 1.01, a["ygrad"] * 0.99
    elif form == "bidirectional":
        a = group(48, 40, 16, np.uint16, "D", isbidirectional=True)
    else:
        a = group(50, 37, 0, np.float32, "D", nknots=5)
    check(a, ssa.align_groups([a])[0])


def test_misaligned_frames():
    """Resident frames two bytes past a 16-byte boundary give the aligned
    frames' results bit for bit."""
    a = group(48, 40, 16, np.uint16, "D")
    bm = np.asfortranarray(a["bmData"])
    buf = DeviceBuffer(bm.nbytes + 16)
    results = []
    for off in (0, 2):
        raw = np.zeros(bm.nbytes + 16, np.uint8)
        raw[off:off + bm.nbytes] = bm.ravel(order="F").view(np.uint8)
        buf.upload(raw)
        results.append(ssa.align_groups([dict(a, bmData=(buf.ptr.value + off, np.uint16))])[0])
    for k in ("knots_x", "knots_y", "frame_corr", "residrms", "mask"):
        assert np.array_equal(results[0][k], results[1][k]), k
