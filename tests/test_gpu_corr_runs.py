"""The global correlation against the FP64 oracle at column counts around one
and two runs of rows per thread (256 and 512 image columns), where the pass
that looks for the column's first row outside the template ends.  Motion of a
few pixels over a template of the frame's size puts that row before, into and
behind either run.  Correlations are sums of at most 20,000 FP64 terms in
another order, with a cancellation of about 100: held to 1e-9, as are the
knots in pixels."""
import numpy as np
import pytest

import steadyscan_amd as ssa
from oracle import oracle as O
from steadyscan_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lines", [8, 12])
@pytest.mark.parametrize("w", [200, 256, 257, 300, 512, 513, 600])
def test_corr_runs(w, lines):
    h, n = 3 * lines, 4
    T = W.make_template(h, w, 60, (2.0, 6.0), offset=10.0, seed=61)
    dx, dy = W.make_motion(n, h, 0.05, 0.0, (6.0, 0.5), seed=62)
    fr = W.make_frames(T, dx, dy, h, w, np.uint16, True, seed=63)
    a = W.group_args(T, fr, ssa.init_settings(h, w, T.shape, nknots=4), flags="DC", max_iter=6)
    out = ssa.align_group_to_template(*[a[k] for k in W.ARG_ORDER], nargout=8)
    ref = O.align_group_to_template(a, threads=4)
    m, it = ref["mask"].astype(bool), ref["iterations"]
    assert not m.all() and np.array_equal(out[4].astype(bool).reshape(m.shape), m)
    assert int(out[3]) == it
    assert np.max(np.abs(out[7].ravel()[:it] - ref["iteration_corr"][:it])) <= 1e-9
    assert np.max(np.abs(out[2].ravel() - ref["frame_corr"])) <= 1e-9
    for i, k in enumerate(("knots_x", "knots_y")):
        assert np.max(np.abs(out[i].ravel() - ref[k]).ravel()[:-4]) <= 1e-9, k
