"""Fine correlation over all 17 x 17 lags: the streamed kernel's matrix-core lag sums against
the staged pipeline's.

Images of independent noise put the oversampled surface's peak anywhere in it, so a wrong
lag, bin or template row shows in the peak or in its lead over the runner-up (margin). Both
pipelines sum 16,384 products of unit-variance order in FP32 (about 1e-7 sqrt(128) a bin):
leads agree within 1e-5, and peaks wherever the lead is larger.
"""
import numpy as np
import pytest
import torch

from isce2_amd.engine import MODE_FUSED, MODE_STAGED, Engine, WindowParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ovs,mode", [(16, MODE_FUSED), (8, 0), (32, 0)])
@pytest.mark.parametrize("real", [False, True])
def test_streamed_fine_kernel(ovs, mode, real):
    rng = np.random.default_rng(5)
    img = [rng.standard_normal((2, 420, 420)).astype(np.float32) for _ in range(2)]
    img = [np.abs(z[0]) if real else (z[0] + 1j * z[1]).astype(np.complex64) for z in img]
    dev = torch.device("cuda", 0)
    ref, sec = (torch.from_numpy(z).to(dev) for z in img)
    d, a = np.meshgrid(np.arange(20, 330, 39), np.arange(20, 330, 39), indexing="ij")
    st = [torch.as_tensor(v.ravel() - o, dtype=torch.int32).to(dev) for v, o in ((d, 0), (a, 0), (d, 16), (a, 16))]
    eng = Engine(0)
    eng.setup(WindowParams(hs_down=16, hs_across=16, surf_ovs=ovs, image_complex=int(not real)))
    eng.set_precision(0)
    out = []
    for m in (mode, MODE_STAGED):
        g = eng.run_windows(ref, sec, *st, mode=m, debug=True)
        out.append({k: g[k].cpu().numpy() for k in ("zoom_idx", "margin_fine", "offset")})
    eng.close()
    new, old = out
    assert np.abs(new["margin_fine"] - old["margin_fine"]).max() < 1e-5
    clear = old["margin_fine"] > 1e-5
    assert clear.sum() >= 8          # (leads shrink with the square of the factor)
    assert np.array_equal(new["zoom_idx"][clear], old["zoom_idx"][clear])
    assert np.array_equal(new["offset"][clear], old["offset"][clear])
    assert np.ptp(new["zoom_idx"], axis=0).min() > 8 * ovs
