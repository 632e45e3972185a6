"""bm3d_match_cols against the oracle on frames of 32768 blocks and more, which take it.

Its edges at that size: the smallest frames of a run's region in each
direction, partly filled runs and grid-row pairs.
"""

import os

import numpy as np
import pytest

from test_gpu_cols import _clip

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("content", ["noisy", "bars", "clean", "nonfinite"])
@pytest.mark.parametrize("w,h", [(8203, 71), (93, 6301), (64, 9000), (13202, 44)])
def test_groups_match_oracle(w, h, content):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from oracle import pyoracle
    from vsfeel.torch_bm3d import Instance

    clip = _clip(content, w, h)
    kw = dict(sigma=3.0, block_step=4, bm_range=16)
    inst = Instance(1, h, w, fp_mode=1, **kw)
    g, _ = inst.groups(torch.from_numpy(clip).to("cuda:0"), 0)
    p = pyoracle.make_params(w, h, fp_mode=1, nthreads=NT, **kw)
    _, og = pyoracle.estimate(p, [clip[0]])
    bad = int((g != og).any(axis=(2, 3)).sum())
    assert bad == 0, f"{bad} of {g.shape[0] * g.shape[1]} groups differ"
