"""The driver packs its frames on the GPU: for every element type, for blocks
of different lengths, bidirectional and cropped scans, its knots are those of
the same sets packed on the host (image2blockmatrix), bit for bit."""
import numpy as np
import pytest

import steadyscan_amd as ssa
from steadyscan_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,nknots,dtype,geo", [
    (48, 40, 7, np.uint16, {}),
    (50, 37, 6, np.int16, {}),
    (50, 37, 6, np.float32, dict(isbidirectional=True)),
    (48, 44, 4, np.float64, dict(cropping=(3, 2, 0, 0))),
])
def test_packed_on_the_device(handle, h, w, nknots, dtype, geo):
    T = W.make_template(h, w, 40, (2.0, 6.0), offset=10.0, seed=5)
    dx, dy = W.make_motion(9, h, 0.05, 0.0, (1.5, 1.0), seed=6)
    fr = W.make_frames(T, dx, dy, h, w, dtype, True, seed=7)
    got = ssa.estimate_displacements(fr, T, nknots=nknots, frames_per_set=4, min_frames_per_set=2, corr_thresh=0.0,
                                     handle=handle, max_iter=5, **geo)
    geom = ssa.init_settings(h, w, T.shape, nknots=nknots, **geo)
    calls = []
    for first, n in ((0, 5), (4, 5), (8, 1)):  # each set with the next one's first frame
        a = W.group_args(T, fr, geom, first=first, count=n, max_iter=5)
        calls.append(dict(a, bmData=np.asfortranarray(a["bmData"])))
    for (first, n), r in zip(((0, 5), (4, 5)), ssa.align_groups(calls, handle=handle)):
        used = r["mask"].reshape(geom["frame_h"], nknots - 1, n, order="F").any(axis=0)
        for f in range(n - 1):
            if not used[:, f].all():
                continue  # extended from the first and last used block
            for out, k in ((got["dx_knots"], "knots_x"), (got["dy_knots"], "knots_y")):
                assert np.array_equal(out[:, first + f], r[k].reshape(n, nknots)[f])
            assert got["corr"][first + f] == r["frame_corr"][f]
