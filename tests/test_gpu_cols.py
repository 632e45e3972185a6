"""Spatial search at bm_range 16, block_step 4 on small frames against the oracle: groups entry for entry.

bm3d_match_rows searches these; bm3d_match_cols takes frames of 32768 blocks
and more (test_gpu_cols_content.py, test_gpu_cols_large.py).  Frames of a few
runs, partly filled runs, windows clipped on every side; equal and near-equal
pixels, huge and non-finite ones, texture along columns.
"""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)

# 135 to 8160 blocks
SIZES = [(64, 40), (65, 45), (91, 77), (93, 131), (481, 275)]


def _clip(content, w, h):
    from vsfeel import synth
    rng = np.random.default_rng(w * 1000 + h)
    img = synth.gray_clip(21, 1, w, h, 3 / 255)[0]
    if content == "bars":
        img[: h // 4] = 0.0
        img[:, w - w // 5:] = 0.25
    elif content == "clean":
        img = synth.gray_clip(22, 1, w, h, 0.0)[0]
    elif content == "columns":
        img = 0.5 + 0.2 * np.sin(np.arange(w) / 1.1)[None, :] + rng.normal(0, 2 / 255, (h, w))
    elif content == "clipped":
        img = np.clip(img * 4.0 - 1.0, 0.0, 1.0)
    elif content == "nonfinite":
        img[h // 2, w // 3] = np.nan
        img[h // 3, w // 2] = np.inf
        img[5:9, 7:9] = -3e19
        img[h - 9:h - 2, w - 20:w - 4] = 1e30
    return np.stack([img]).astype(np.float32)


@pytest.mark.parametrize("content", ["noisy", "bars", "clean", "columns", "clipped", "nonfinite"])
@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("fp_mode", [1, 2])
def test_groups_match_oracle(w, h, content, fp_mode):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from oracle import pyoracle
    from vsfeel.torch_bm3d import Instance

    if fp_mode == 2 and (w, h) != (91, 77):
        pytest.skip("one size is enough for the other rounding")
    clip = _clip(content, w, h)
    kw = dict(sigma=3.0, block_step=4, bm_range=16)
    inst = Instance(1, h, w, fp_mode=fp_mode, **kw)
    g, _ = inst.groups(torch.from_numpy(clip).to("cuda:0"), 0)
    p = pyoracle.make_params(w, h, fp_mode=fp_mode, nthreads=NT, **kw)
    _, og = pyoracle.estimate(p, [clip[0]])
    bad = int((g != og).any(axis=(2, 3)).sum())
    assert bad == 0, f"{bad} of {g.shape[0] * g.shape[1]} groups differ"
