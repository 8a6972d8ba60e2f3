"""The driver's frame stack on the device: recordings longer than a piece of
the upload (256 MiB) and than its staging (two halves of 32 MiB), and raw
frames of more pixels than 32 bits count, of which the cropping leaves a few,
and a device that holds the stack or a batch, not both."""
import ctypes

import numpy as np
import pytest

import steadyscan_amd as ssa
from steadyscan_amd import workloads as W

from devbuf import DeviceBuffer

pytestmark = pytest.mark.gpu

KEYS = ("dx_knots", "dy_knots", "corr", "iter_used", "residrms", "failed")


@pytest.mark.parametrize("pregauss", [0.0, 1.0])
def test_pieces_of_a_long_recording(handle, pregauss):
    """Sets are aligned independently, so that a set of a long recording has
    the outputs of a recording that holds its frames alone, bit for bit."""
    h, per_set = 512, 130
    T = W.make_template(h, h, 200, (2.0, 6.0), offset=10.0, seed=15)
    dx, dy = W.make_motion(per_set + 1, h, 0.05, 0.0, (1.5, 1.0), seed=16)
    part = W.make_frames(T, dx, dy, h, h, np.uint16, True, seed=17)
    fr = np.empty((h, h, 1100), np.uint16, order="F")  # 2.1 pieces
    for f in range(fr.shape[2]):
        fr[:, :, f] = part[:, :, f % part.shape[2]]
        fr[f % h, :, f] += 1 + f // h  # no two frames alike
    kw = dict(nknots=33, frames_per_set=per_set, min_frames_per_set=10, pregauss=pregauss, handle=handle, max_iter=3)
    got = ssa.estimate_displacements(fr, T, **kw)
    for first in (0, 3 * per_set, 7 * per_set):  # the first, the one with frame 512, the one with frame 1024
        alone = ssa.estimate_displacements(fr[:, :, first:first + per_set + 1], T, **dict(kw, frames_per_set=per_set + 1))
        for k in KEYS:
            assert np.array_equal(got[k][..., first:first + per_set], alone[k][..., :per_set], equal_nan=True), (first, k)


def test_wide_raw_frames(handle):
    """8 lines of 2**29 pixels, all but 40 columns cropped.  The rest of the
    array is never written, so that it takes no memory."""
    h, w, n = 8, 1 << 29, 2
    crop = (w - 40, 0, 0, 0)
    T = W.make_template(64, 64, 60, (2.0, 6.0), offset=10.0, seed=25)
    fr = np.zeros((h, w, n), np.uint16, order="F")
    for f in range(n):  # template columns 21 .. 60, moved by a third of a pixel
        fr[:, crop[0]:, f] = np.round((2 * T[9:17, 20:60] + T[9:17, 21:61]) / 3)
    kw = dict(nknots=2, cropping=crop, subrec=(60.0 - (w - 1), 60.0, 10.0, 17.0))
    got = ssa.estimate_displacements(fr, T, frames_per_set=2, min_frames_per_set=1, corr_thresh=-2.0, handle=handle,
                                     max_iter=3, **kw)
    geom = ssa.init_settings(h, w, T.shape, **kw)
    a = W.group_args(T, fr, geom, max_iter=3)
    r = ssa.align_groups([dict(a, bmData=np.asfortranarray(a["bmData"]))], handle=handle)[0]
    for out, k in ((got["dx_knots"], "knots_x"), (got["dy_knots"], "knots_y")):
        assert np.isfinite(out[:, 0]).all() and np.array_equal(out[:, 0], r[k].reshape(n, 2)[0])
    assert (got["dx_knots"][:, 0] > 0).all()


def test_stack_and_batch_in_turn():
    """A call of the driver and a batch of about 1.2 GiB each, with 2 GiB of
    the device left: either runs after the other."""
    h, n, per_set = 256, 6200, 310
    T = W.make_template(h, h, 100, (2.0, 6.0), offset=10.0, seed=35)
    dx, dy = W.make_motion(per_set, h, 0.05, 0.0, (1.5, 1.0), seed=36)
    part = W.make_frames(T, dx, dy, h, h, np.uint16, True, seed=37)
    fr = np.asfortranarray(np.broadcast_to(part[:, :, None, :], (h, h, n // per_set, per_set)).reshape((h, h, n)))
    hd = ssa.Handle(0)
    a = W.group_args(T, part, ssa.init_settings(h, h, T.shape, nknots=17), max_iter=2)
    calls = [dict(a, bmData=np.asfortranarray(np.tile(a["bmData"], (1, 31))), nsetframes=31 * per_set,
                  est_dx_knots=np.zeros((17, 31 * per_set)), est_dy_knots=np.zeros((17, 31 * per_set)))]
    kw = dict(nknots=17, min_frames_per_set=2, handle=hd, max_iter=2)
    ssa.estimate_displacements(fr[:, :, :8], T, frames_per_set=8, **kw)  # the kernels' own memory
    hip = DeviceBuffer(1 << 20)._hip
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    ballast = DeviceBuffer(free.value - (2 << 30))
    try:
        for _ in range(2):
            est = ssa.estimate_displacements(fr, T, frames_per_set=per_set, **kw)
            assert np.isfinite(est["dx_knots"][:, :-1]).all()
            assert np.isfinite(ssa.align_groups(calls, handle=hd, with_mask=False)[0]["frame_corr"]).all()
    finally:
        ballast.free()
        hd.close()


def test_doubles_in_single_precision(handle):
    """FP64 frames in precision 'S' are packed as floats, with the results of
    the same sets as host frames, and no more than 6 bytes a pixel held."""
    h, n = 256, 800
    T = W.make_template(h, h, 100, (2.0, 6.0), offset=10.0, seed=45)
    dx, dy = W.make_motion(9, h, 0.05, 0.0, (1.5, 1.0), seed=46)
    part = W.make_frames(T, dx, dy, h, h, np.float64, True, seed=47) / 3
    fr = np.asfortranarray(np.resize(part.transpose(2, 1, 0), (n, h, h)).transpose(2, 1, 0))
    kw = dict(flags="S", nknots=17, frames_per_set=100, min_frames_per_set=10, max_iter=3)
    hd = ssa.Handle(0)
    ssa.estimate_displacements(fr[:, :, :8], T, handle=hd, **kw)
    hip = DeviceBuffer(1 << 20)._hip
    free = [ctypes.c_size_t(), ctypes.c_size_t()]
    total = ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free[0]), ctypes.byref(total)) == 0
    got = ssa.estimate_displacements(fr, T, handle=hd, **kw)
    assert hip.hipMemGetInfo(ctypes.byref(free[1]), ctypes.byref(total)) == 0
    hd.close()
    held = free[0].value - free[1].value
    print(f"{held / fr.size:.2f} bytes a pixel with the raw piece of 256 MiB", flush=True)
    # floats and masks 5 bytes, the state of the batch (16 blocks of 4096 pixels a frame) below 1
    assert held - (256 << 20) <= 6 * fr.size
    geom = ssa.init_settings(h, h, T.shape, nknots=17)
    a = W.group_args(T, fr, geom, flags="S", first=100, count=101, max_iter=3)
    r = ssa.align_groups([dict(a, bmData=np.asfortranarray(a["bmData"]))], handle=handle)[0]
    for out, k in (("dx_knots", "knots_x"), ("dy_knots", "knots_y")):
        assert np.array_equal(got[out][:, 100:200].T, r[k].reshape(101, 17)[:100])
    assert np.array_equal(got["corr"][100:200], r["frame_corr"][:100])
