"""Windowed-sinc surface from a zoom window of 2 x 2 (raw oversampling 1), the smallest that
setup accepts: the patch covers the whole surface, starts before it, and its taps wrap around
the two samples more than once. Against a periodic numpy interpolation put in the oracle's
place (whose indices, like the reference's, wrap once); FP64, integer peaks equal.
"""
import numpy as np
import pytest

from isce2_amd.engine import MODE_AUTO, MODE_STAGED, Engine
from isce2_amd.synth import speckle_pair_shift
from oracle import ampcor_oracle as O

from .gpu_helpers import compare, run_both

pytestmark = pytest.mark.gpu


def _periodic(surf, out_n, covs, center_shift, factor, window=2):
    table, taps, dec = O.sinc_filter_table()
    table = table.astype(np.float32).astype(np.float64)          # as the engine stores it
    n, h, w = surf.shape
    out = np.zeros((n, out_n, out_n))
    for k in range(n):
        pos = [(np.arange(2 * window * covs + 1) + out_n // 2 - window * covs + int(s) * factor) % out_n
               for s in center_shift[k]]
        (mx, my) = (np.zeros((len(p), m)) for p, m in zip(pos, (h, w)))
        for mat, p in ((mx, pos[0]), (my, pos[1])):
            for t in range(taps):
                coef = table[t * dec + (p % covs) * dec // covs]
                np.add.at(mat, (np.arange(len(p)), (p // covs - t + taps // 2) % mat.shape[1]), coef)
            mat /= mat.sum(1, keepdims=True)
        out[k][np.ix_(*pos)] = mx @ surf[k] @ my.T
    return out


@pytest.mark.parametrize("ovs", [1, 4, 16])
@pytest.mark.parametrize("shift", [(1.4, -2.2), (6.3, -6.4)])      # inside, and at the edge of the search range
def test_two_by_two_zoom(ovs, shift, monkeypatch):
    monkeypatch.setattr(O, "oversample_sinc", _periodic)
    ref, sec = speckle_pair_shift(200, 200, shift=shift, snr_db=15.0, seed=21)
    cfg = O.AmpcorConfig(window_h=32, window_w=24, hs_down=6, hs_across=6, raw_ovs=1, zoom=2, surf_ovs=ovs, surf_method=1)
    starts = O.start_pixels(4, 4, 12, 12, 36, 36, 0, 0, 6, 6)[:4]
    eng = Engine(0)
    eng.set_precision(2)
    for mode in (MODE_AUTO, MODE_STAGED):
        c = compare(*run_both(eng, ref, sec, cfg, starts, mode))
        assert c["maxloc_mismatch"] == c["start_mismatch"] == c["shift_mismatch"] == c["zoom_mismatch"] == 0
        assert c["offset_max_err"] <= 0.01 and c["snr_max_rel"] <= 1e-6
    eng.close()
