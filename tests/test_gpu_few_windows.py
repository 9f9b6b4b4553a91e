"""Calls of up to 256 windows, whose reference chips are oversampled in the coarse stage's
launch, give each window what a larger call gives it, bit for bit."""
import numpy as np
import pytest
import torch

from isce2_amd.engine import MODE_FUSED, Engine, WindowParams
from isce2_amd.synth import speckle_pair_shift

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,hs", [(32, 8), (32, 24), (64, 20), (64, 32)])
@pytest.mark.parametrize("deramp", [0, 1])
def test_few_windows(W, hs, deramp):
    ref, sec = speckle_pair_shift(400, 400, shift=(1.3, -0.7), snr_db=12.0, seed=8)
    dev = torch.device("cuda", 0)
    ref, sec = torch.from_numpy(ref).to(dev), torch.from_numpy(sec).to(dev)
    rng = np.random.default_rng(2)
    d, a = rng.integers(hs, 400 - W - hs, (2, 257)).astype(np.int32)
    st = [torch.as_tensor(v).to(dev) for v in (d, a, d - hs, a - hs)]
    eng = Engine(0)
    eng.setup(WindowParams(window_h=W, window_w=W, hs_down=hs, hs_across=hs, deramp=deramp))
    many = eng.run_windows(ref, sec, *st, mode=MODE_FUSED, debug=True)
    many = {k: v.cpu().numpy() for k, v in many.items()}
    for n in (1, 2, 9, 256):
        few = eng.run_windows(ref, sec, *(v[257 - n:] for v in st), mode=MODE_FUSED, debug=True)
        for k, v in few.items():
            assert np.array_equal(v.cpu().numpy(), many[k][257 - n:], equal_nan=True), (n, k)
    eng.close()
