"""FP64 pipeline on both sides of the line between direct lag sums and transformed lag rows
(1.5e7 products), by window count and by search range, against the FP64 oracle. Bar as in
test_gpu_staged_lags: integer peaks equal, offsets within 0.01 px, SNR and covariance within
1e-6 (the outputs are FP32 numbers)."""
import numpy as np
import pytest
import torch

from isce2_amd.engine import MODE_STAGED, Engine
from isce2_amd.synth import speckle_pair_shift
from oracle import ampcor_oracle as O

from .gpu_helpers import compare, params_from_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wh,ww,hd,ha,n", [(64, 64, 64, 64, 9), (64, 64, 64, 64, 10), (20, 24, 150, 12, 60), (40, 33, 9, 150, 17),
                                           (64, 64, 20, 20, 180), (24, 24, 160, 160, 2)])
def test_fp64_lags(wh, ww, hd, ha, n):
    scene = speckle_pair_shift(420, 400, shift=(2.3, -1.6), snr_db=12.0, seed=31)
    cfg = O.AmpcorConfig(window_h=wh, window_w=ww, hs_down=hd, hs_across=ha)
    rng = np.random.default_rng(5)
    rd, ra = rng.integers(hd, 420 - wh - hd, n), rng.integers(ha, 400 - ww - ha, n)
    st = (rd, ra, rd - hd, ra - ha)
    dev = torch.device("cuda", 0)
    eng = Engine(0)
    eng.setup(params_from_cfg(cfg))
    eng.set_precision(2)
    g = eng.run_windows(*(torch.from_numpy(z).to(dev) for z in scene),
                        *(torch.as_tensor(s.astype(np.int32)).to(dev) for s in st), mode=MODE_STAGED, debug=True)
    g = {k: v.cpu().numpy() for k, v in g.items()}
    eng.close()
    c = compare(g, O.run_windows(*scene, *st, cfg))
    print(f"\n[fp64 lags {wh}x{ww} hs={hd}x{ha} n={n}] {c}")
    assert c["maxloc_mismatch"] == c["start_mismatch"] == c["shift_mismatch"] == c["zoom_mismatch"] == 0
    assert c["offset_max_err"] <= 0.01 and c["snr_max_rel"] <= 1e-6 and c["cov_max_rel"] <= 1e-6
