"""Bounds check of a synchronous call: the first window whose chips leave their images, across
the check's blocks of 256 windows and the selection's of 1,024, and none."""
import numpy as np
import pytest
import torch

from isce2_amd.engine import Engine, WindowParams
from isce2_amd.synth import speckle_pair_shift

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bad", [(1, []), (1, [0]), (256, [255]), (257, [256, 3]), (1024, []), (1025, [1024]),
                                   (2100, [2099, 1500, 300]), (2100, [])])
def test_first_window_outside(n, bad):
    ref, sec = speckle_pair_shift(128, 128, shift=(0.5, -0.25), snr_db=20.0, seed=3)
    dev = torch.device("cuda", 0)
    ref, sec = torch.from_numpy(ref).to(dev), torch.from_numpy(sec).to(dev)
    st = np.empty((4, n), np.int32)
    st[0] = st[1] = 40
    st[2] = st[3] = 32
    for k, i in enumerate(bad):
        st[k % 4, i] = (-1, 97, 81, -1)[k % 4]      # one past each image's last (or first) start
    eng = Engine(0)
    eng.setup(WindowParams(window_h=32, window_w=32, hs_down=8, hs_across=8))
    t = [torch.as_tensor(v).to(dev) for v in st]
    if bad:
        with pytest.raises(Exception, match=rf"window {min(bad)} reads outside its image"):
            eng.run_windows(ref, sec, *t)
    else:
        g = eng.run_windows(ref, sec, *t)["offset"].cpu().numpy()
        assert np.all(g == g[0]) and np.isfinite(g).all()
    eng.close()
