"""Surface oversampling factors and methods through the fused and the staged kernels.

The FFT surface is evaluated from its 16-sparse spectrum for factors 2 to 32, the
windowed-sinc surface from its patch alone; both against the FP64 oracle at the
smallest, the largest and odd factors, with shifts that put some peaks at the edge
of the search range (the zoom chip is clamped there and the sinc patch moves).
Bar as in test_gpu_parity: integer peaks equal, offsets within 0.01 px.
"""
import numpy as np
import pytest

from isce2_amd.engine import MODE_AUTO, MODE_FUSED, MODE_STAGED, Engine
from isce2_amd.synth import speckle_pair_shift
from oracle import ampcor_oracle as O

from .gpu_helpers import compare, params_from_cfg, run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def scene():
    return speckle_pair_shift(400, 400, shift=(6.7, -5.4), snr_db=15.0, seed=11)


def _check(eng, scene, cfg, modes):
    rd, ra, sd, sa = O.start_pixels(4, 4, 32, 32, 70, 70, 0, 0, cfg.hs_down, cfg.hs_across)[:4]
    for mode in modes:
        c = compare(*run_both(eng, *scene, cfg, (rd, ra, sd, sa), mode))
        print(f"\n[surface mode={mode} W={cfg.window_h} ovs={cfg.surf_ovs} method={cfg.surf_method}] {c}")
        assert c["maxloc_mismatch"] == c["start_mismatch"] == c["shift_mismatch"] == c["zoom_mismatch"] == 0
        assert c["offset_max_err"] <= 0.01 and c["snr_max_rel"] <= 1e-3 and c["cov_max_rel"] <= 1e-3


@pytest.mark.parametrize("W,hs", [(64, 20), (64, 7), (32, 12)])
@pytest.mark.parametrize("ovs", [2, 5, 16, 17, 31, 32])
def test_fft_surface_factor(eng, scene, W, hs, ovs):
    _check(eng, scene, O.AmpcorConfig(window_h=W, window_w=W, hs_down=hs, hs_across=hs, surf_ovs=ovs), (MODE_AUTO, MODE_STAGED))


@pytest.mark.parametrize("W,hs", [(64, 20), (64, 7), (32, 12)])
@pytest.mark.parametrize("ovs", [2, 16, 32])
def test_sinc_surface_factor(eng, scene, W, hs, ovs):
    _check(eng, scene, O.AmpcorConfig(window_h=W, window_w=W, hs_down=hs, hs_across=hs, surf_ovs=ovs, surf_method=1),
           (MODE_AUTO, MODE_STAGED))


@pytest.mark.parametrize("kw", [dict(surf_ovs=1), dict(surf_ovs=33), dict(zoom=8, surf_ovs=32), dict(zoom=8, surf_ovs=8, surf_method=1),
                                dict(zoom=4, surf_ovs=16, surf_method=1), dict(zoom=32, surf_ovs=64, surf_method=1)])
def test_staged_surface(eng, scene, kw):
    _check(eng, scene, O.AmpcorConfig(window_h=48, window_w=40, hs_down=12, hs_across=9, **kw), (MODE_STAGED,))


def test_fused_mode_accepts_what_it_did(eng):
    """MODE_FUSED and sizes["fused"] stand for surface factor 16 by the FFT only; AUTO chooses for the rest."""
    for kw, fused in ((dict(), 1), (dict(surf_ovs=32), 0), (dict(surf_method=1), 0)):
        assert eng.setup(params_from_cfg(O.AmpcorConfig(**kw)))["fused"] == fused
    ref, sec = speckle_pair_shift(128, 128, seed=2)
    z = np.zeros(1, np.int64)
    with pytest.raises(NotImplementedError):
        run_both(eng, ref, sec, O.AmpcorConfig(surf_ovs=32), (z + 20, z + 20, z, z), MODE_FUSED)
