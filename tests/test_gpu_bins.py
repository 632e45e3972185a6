"""Binned scatter of groups with 4 to 7 temporal insertions (frames of 32768 blocks and more) against the oracle."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("radius,ps_num,ps_range,extractor_exp", [(1, 2, 4, 0), (1, 3, 5, 2), (2, 1, 7, 0)])
@pytest.mark.parametrize("w,h", [(376, 361), (1101, 131)])  # 33300 and 34125 blocks
def test_output_matches_oracle(w, h, radius, ps_num, ps_range, extractor_exp):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from oracle import pyoracle
    from vsfeel import synth
    from vsfeel.torch_bm3d import Instance

    clip = np.ascontiguousarray(synth.shifted_clip(51, radius + 1, w, h, 3 / 255, (2.0, 1.0)), np.float32)
    kw = dict(sigma=3.0, block_step=2, bm_range=3, radius=radius, ps_num=ps_num, ps_range=ps_range,
              extractor_exp=extractor_exp)
    print(f"{w}x{h} {kw}", flush=True)
    inst = Instance(len(clip), h, w, fp_mode=1, **kw)
    got = inst.process(torch.from_numpy(clip).to("cuda:0")).cpu().numpy()
    assert "bm3d_gather" in _kernels(inst, torch.from_numpy(clip).to("cuda:0"))
    ref = pyoracle.clip(pyoracle.make_params(w, h, fp_mode=1, nthreads=NT, **kw), clip)
    assert float(np.abs(got - ref).max()) <= 1e-5


def _kernels(inst, x):
    inst.set_timing(True)
    inst.process(x)
    names = [k for k, v in inst.kernel_times().items() if v[1]]
    inst.set_timing(False)
    return names
