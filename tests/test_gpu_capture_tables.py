"""A captured call that lacks a device table fails and asks for a plain call first; that
plain call builds the table, and its results are those of a context that never failed.

The first two calls leave every buffer in place at its size and every transform's twiddles,
so that under capture only the tables of the in-place oversampler can be missing."""
import numpy as np
import pytest
import torch

from isce2_amd.engine import MODE_STAGED, Engine, WindowParams
from isce2_amd.synth import speckle_pair_shift

pytestmark = pytest.mark.gpu


def test_plain_call_after_a_refused_capture():
    ref, sec = speckle_pair_shift(400, 400, shift=(1.3, -0.7), snr_db=12.0, seed=8)
    dev = torch.device("cuda", 0)
    ref, sec = torch.from_numpy(ref).to(dev), torch.from_numpy(sec).to(dev)
    st = [torch.full((2,), v, dtype=torch.int32, device=dev) for v in (20, 24, 12, 16)]
    big, small = (WindowParams(window_h=w, window_w=w, hs_down=8, hs_across=8) for w in (256, 128))

    def run(eng, **kw):
        return eng.run_windows(ref, sec, *st, mode=MODE_STAGED, debug=True, nosync=True, **kw)

    eng = Engine(0)
    eng.set_precision(0)
    eng.setup(big)
    run(eng)
    eng.setup(small)
    eng.set_option("oversampler", 3)        # the general transforms: twiddles, no shift tables
    out = run(eng)
    eng.set_option("oversampler", 2)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(device=dev)
    try:
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=side):
            run(eng, out=out)
    except ValueError as e:
        assert "before capturing it" in str(e)
    got = {k: v.cpu().numpy() for k, v in run(eng).items()}
    eng.close()
    fresh = Engine(0)
    fresh.set_precision(0)
    fresh.setup(small)
    want = {k: v.cpu().numpy() for k, v in run(fresh).items()}
    fresh.close()
    for k in want:
        assert np.array_equal(got[k], want[k], equal_nan=True), k
    assert np.isfinite(got["offset"]).all()
