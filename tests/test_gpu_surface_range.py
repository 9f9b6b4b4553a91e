"""Surfaces other than factor 16 by the FFT keep the staged pipeline's FP64 normalization in
the fused kernels that automatic mode runs for them: images whose sums of squares, multiplied,
leave FP32's range (amplitudes around 1e10 and 1e15; FP32 correlations themselves reach 1e34) give what
the FP64 oracle gives, without the FP64 re-run. Bar as in test_gpu_parity where the argmax is
clear of FP32 rounding (both leads above 2e-6): integer peaks equal, offsets within 0.01 px,
SNR and covariance within 1e-3.
"""
import numpy as np
import pytest

from isce2_amd.engine import MODE_AUTO, MODE_STAGED, Engine
from isce2_amd.synth import speckle_pair_shift
from oracle import ampcor_oracle as O

from .gpu_helpers import compare, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,hs", [(64, 20), (32, 9)])
@pytest.mark.parametrize("kw", [dict(surf_ovs=32), dict(surf_ovs=5), dict(surf_method=1)])
@pytest.mark.parametrize("real,scale", [(False, 1e10), (True, 1e10), (False, 1e15)])
def test_bright_images(W, hs, kw, real, scale):
    ref, sec = (z * np.float32(scale) for z in speckle_pair_shift(400, 400, shift=(3.7, -2.4), snr_db=15.0, seed=11))
    if real:
        ref, sec = np.abs(ref), np.abs(sec)
    cfg = O.AmpcorConfig(window_h=W, window_w=W, hs_down=hs, hs_across=hs, **kw)
    starts = O.start_pixels(4, 4, 32, 32, 70, 70, 0, 0, hs, hs)[:4]
    eng = Engine(0)
    eng.set_precision(0)
    for mode in (MODE_AUTO, MODE_STAGED):
        g, o = run_both(eng, ref, sec, cfg, starts, mode)
        clear = (g["margin_coarse"] > 2e-6) & (g["margin_fine"] > 2e-6)
        assert clear.sum() >= 8, mode
        c = compare({k: v[clear] for k, v in g.items()}, {k: v[clear] for k, v in o.items()})
        print(f"\n[bright W={W} {kw} real={real} mode={mode}] {c}")
        assert c["maxloc_mismatch"] == c["start_mismatch"] == c["shift_mismatch"] == c["zoom_mismatch"] == 0
        assert c["offset_max_err"] <= 0.01 and c["snr_max_rel"] <= 1e-3 and c["cov_max_rel"] <= 1e-3
    eng.close()
