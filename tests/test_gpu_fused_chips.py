"""Fused kernels on every chip kind at the image's corners and edges, against the FP64 oracle.

Both window sizes, the three deramp methods and real images, on a scene with a phase
ramp (so that the deramp rotates) whose windows touch all four image borders. Bar as in
test_gpu_parity: integer peaks equal, offsets within 0.01 px, SNR and covariance within 1e-3.
"""
import numpy as np
import pytest

from isce2_amd.engine import MODE_FUSED, Engine
from isce2_amd.synth import speckle_pair_shift
from oracle import ampcor_oracle as O

from .gpu_helpers import compare, run_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = Engine(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def scene():
    ref, sec = speckle_pair_shift(260, 272, shift=(1.4, -2.2), snr_db=15.0, seed=21)
    y, x = np.mgrid[0:260, 0:272]
    ramp = np.exp(1j * (0.11 * y - 0.07 * x)).astype(np.complex64)
    return ref * ramp, sec * ramp


@pytest.mark.parametrize("W,hs", [(32, 9), (64, 14), (64, 32)])
@pytest.mark.parametrize("deramp", [0, 1, 2])
@pytest.mark.parametrize("real", [False, True])
def test_fused_chips(eng, scene, W, hs, deramp, real):
    ref, sec = scene
    if real:
        ref, sec = np.abs(ref).astype(np.float32), np.abs(sec).astype(np.float32)
    d = np.linspace(hs, ref.shape[0] - W - hs, 3).astype(np.int64)
    a = np.linspace(hs, ref.shape[1] - W - hs, 3).astype(np.int64)
    rd, ra = (v.ravel() for v in np.meshgrid(d, a, indexing="ij"))
    cfg = O.AmpcorConfig(window_h=W, window_w=W, hs_down=hs, hs_across=hs, deramp=deramp)
    c = compare(*run_both(eng, ref, sec, cfg, (rd, ra, rd - hs, ra - hs), MODE_FUSED))
    print(f"\n[fused chips W={W} hs={hs} deramp={deramp} real={real}] {c}")
    assert c["maxloc_mismatch"] == c["start_mismatch"] == c["shift_mismatch"] == c["zoom_mismatch"] == 0
    assert c["offset_max_err"] <= 0.01 and c["snr_max_rel"] <= 1e-3 and c["cov_max_rel"] <= 1e-3
