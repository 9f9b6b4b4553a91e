"""The tuner offers what automatic mode runs: at a surface factor or method that MODE_FUSED does
not take but automatic mode runs through the fused kernels (several times faster than the staged
pipeline), it chooses MODE_AUTO, also over a staged schedule that a file holds from before."""
import json

import numpy as np
import pytest
import torch

from isce2_amd.autotune import Autotuner
from isce2_amd.engine import MODE_AUTO, MODE_FUSED, MODE_STAGED, Engine, WindowParams
from isce2_amd.synth import speckle_pair_shift

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def args():
    ref, sec = speckle_pair_shift(700, 700, shift=(1.3, -0.7), snr_db=12.0, seed=8)
    dev = torch.device("cuda", 0)
    d, a = np.random.default_rng(2).integers(20, 700 - 64 - 20, (2, 512)).astype(np.int32)
    return [torch.from_numpy(z).to(dev) for z in (ref, sec)] + [torch.as_tensor(v).to(dev) for v in (d, a, d - 20, a - 20)]


@pytest.mark.parametrize("kw,mode,auto", [(dict(surf_ovs=32), MODE_AUTO, True), (dict(surf_method=1), MODE_AUTO, True),
                                          (dict(), MODE_FUSED, True), (dict(window_h=48, window_w=48), MODE_STAGED, False)])
def test_tuned_mode(args, tmp_path, kw, mode, auto):
    p = WindowParams(**kw)
    path = tmp_path / "tune.json"
    key = Autotuner.key(p)
    path.write_text(json.dumps({key: dict(mode=MODE_STAGED, chunk=64, radices={}, options={}, ms_per_window=1.0)}))
    eng = Engine(0)
    assert not eng.auto_fused
    eng.setup(p)
    assert eng.auto_fused == auto
    tuner = Autotuner(device=0, reps=1, sample=512, radix_sample=16, cache_file=str(path))
    sched = tuner.tune(eng, p, args, 512)
    if mode == MODE_AUTO:
        assert sched.mode == MODE_AUTO and json.loads(path.read_text())[key]["mode"] == MODE_AUTO
        got = eng.run_windows(*args, mode=sched.mode, chunk=sched.chunk)
        want = eng.run_windows(*args)
        for k in want:
            assert torch.equal(got[k], want[k]), k
    else:
        assert sched.mode == MODE_STAGED                # a valid schedule from the file stands
        sched = Autotuner(device=0, reps=1, sample=512, radix_sample=16).tune(eng, p, args, 512)
        assert sched.mode == mode
    assert tuner.tune(eng, p, args, 512) is tuner.cache[key]
    eng.close()
