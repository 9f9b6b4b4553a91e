"""Staged pipeline at odd sizes, few windows and partial chunks, FP32 and FP64, against the
FP64 oracle; and the FP64 re-run's scatter.

Sizes sit at the edges of the lag-row kernels: template heights below, at and off multiples
of 16 rows, odd transform lengths, one to a few lag rows per workgroup, search columns off
multiples of 64. Bar: integer peaks equal, offsets within 0.01 px, SNR and covariance within
1e-3 (FP32) or 1e-6 (FP64 pipeline: the outputs are FP32 numbers).
"""
import numpy as np
import pytest
import torch

from isce2_amd.engine import MODE_FUSED, MODE_STAGED, Engine
from isce2_amd.synth import speckle_pair_shift
from oracle import ampcor_oracle as O

from .gpu_helpers import compare, params_from_cfg

pytestmark = pytest.mark.gpu
KEYS = ("offset", "snr", "cov", "maxloc", "start", "shift", "zoom_idx", "maxval")


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def scene():
    return speckle_pair_shift(420, 400, shift=(2.3, -1.6), snr_db=12.0, seed=31)


def _run(eng, scene, cfg, n, precision, chunk=0, tau=(-1.0, -1.0), mode=MODE_STAGED):
    ref, sec = scene
    rng = np.random.default_rng(5)
    rd = rng.integers(cfg.hs_down, ref.shape[0] - cfg.window_h - cfg.hs_down, n)
    ra = rng.integers(cfg.hs_across, ref.shape[1] - cfg.window_w - cfg.hs_across, n)
    st = (rd, ra, rd - cfg.hs_down, ra - cfg.hs_across)
    dev = torch.device("cuda", 0)
    eng.setup(params_from_cfg(cfg))
    eng.set_precision(precision, *tau)
    try:
        g = eng.run_windows(torch.from_numpy(ref).to(dev), torch.from_numpy(sec).to(dev),
                            *[torch.as_tensor(s.astype(np.int32)).to(dev) for s in st], mode=mode, chunk=chunk,
                            debug=True)
    finally:
        eng.set_precision(1, 2e-6, 2e-6)
    return {k: v.cpu().numpy() for k, v in g.items()}, st


@pytest.mark.parametrize("wh,ww,hd,ha", [(12, 13, 4, 5), (15, 64, 7, 4), (16, 16, 4, 4), (17, 70, 9, 6), (48, 40, 24, 7),
                                         (64, 128, 8, 5), (130, 20, 5, 30), (256, 256, 4, 6)])
@pytest.mark.parametrize("precision", [1, 2])
def test_sizes(eng, scene, wh, ww, hd, ha, precision):
    cfg = O.AmpcorConfig(window_h=wh, window_w=ww, hs_down=hd, hs_across=ha)
    for n, chunk in ((1, 0), (5, 2)):
        g, st = _run(eng, scene, cfg, n, precision, chunk)
        c = compare(g, O.run_windows(*scene, *st, cfg))
        print(f"\n[staged {wh}x{ww} hs={hd}x{ha} p={precision} n={n}] {c}")
        tol = 1e-6 if precision == 2 else 1e-3
        assert c["maxloc_mismatch"] == c["start_mismatch"] == c["shift_mismatch"] == c["zoom_mismatch"] == 0
        assert c["offset_max_err"] <= 0.01 and c["snr_max_rel"] <= tol and c["cov_max_rel"] <= tol


@pytest.mark.parametrize("W,hs", [(64, 12), (32, 9)])
def test_rerun_scatter(eng, scene, W, hs):
    """Thresholds that pick every window, every fine stage, or about half the raw stages for the FP64
    re-run of the fused kernels: a window re-run whole has the FP64 pipeline's results, one re-run from
    the zoom stage on its offset and zoom peak, and the FP32 raw results."""
    cfg = O.AmpcorConfig(window_h=W, window_w=W, hs_down=hs, hs_across=hs)
    n = 11
    f32, _ = _run(eng, scene, cfg, n, 0, mode=MODE_FUSED)
    f64, _ = _run(eng, scene, cfg, n, 2)
    assert np.array_equal(f32["start"], f64["start"])
    mid = float(np.median(f32["margin_coarse"]))
    for tau in ((1e9, 0.0), (0.0, 1e9), (mid, 1e9)):
        g, _ = _run(eng, scene, cfg, n, 1, tau=tau, mode=MODE_FUSED)
        full = ~(f32["margin_coarse"] >= tau[0])
        for k in KEYS:
            whole = full | (k in ("offset", "zoom_idx"))
            want = np.where(whole.reshape(-1, *[1] * (f64[k].ndim - 1)), f64[k], f32[k])
            assert np.array_equal(g[k], want), (tau, k)
