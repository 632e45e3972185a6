"""Spatial search by columns on contrasts whose squares are below FP32's normal range, against the oracle."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("amplitude", [1e-19, 3e-21, 1e-21, 1e-22, 1e-24])
def test_groups_match_oracle(amplitude):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from oracle import pyoracle
    from vsfeel import synth
    from vsfeel.torch_bm3d import Instance

    w, h = 769, 727  # 34752 blocks
    clip = (synth.gray_clip(21, 1, w, h, 3 / 255) * amplitude).astype(np.float32)
    kw = dict(sigma=3.0, block_step=4, bm_range=16)
    inst = Instance(1, h, w, fp_mode=1, **kw)
    g, _ = inst.groups(torch.from_numpy(clip).to("cuda:0"), 0)
    _, og = pyoracle.estimate(pyoracle.make_params(w, h, fp_mode=1, nthreads=NT, **kw), [clip[0]])
    bad = int((g != og).any(axis=(2, 3)).sum())
    assert bad == 0, f"{bad} of {g.shape[0] * g.shape[1]} groups differ"
