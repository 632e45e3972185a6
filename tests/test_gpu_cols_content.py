"""bm3d_match_cols on frames that take it (bm_range 16, block_step 4, 32768 blocks and more), in both rounding modes:
content that its shortlist does not hold or its expanded distances do not resolve, groups against the oracle."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)


def _clip(content, w, h):
    from vsfeel import synth
    rng = np.random.default_rng(w * 1000 + h)
    img = synth.gray_clip(21, 1, w, h, 3 / 255)[0].astype(np.float64)
    if content == "columns":  # texture along columns crowds a column's keys
        img = 0.5 + 0.2 * np.sin(np.arange(w) / 1.1)[None, :] + rng.normal(0, 2 / 255, (h, w))
    elif content == "rows":
        img = 0.5 + 0.2 * np.sin(np.arange(h) / 1.1)[:, None] + rng.normal(0, 2 / 255, (h, w))
    elif content == "clipped":  # saturated areas with ragged borders
        img = np.clip(img * 4.0 - 1.0, 0.0, 1.0)
    elif content == "dark":  # noise clipped at 0: blocks with few pixels above it tie with one another
        img = np.clip(0.12 * np.arange(w)[None, :] / w - 0.06 + rng.normal(0, 5 / 255, (h, w)), 0.0, 1.0)
    elif content == "periodic":  # exactly equal matches a period apart
        img = np.tile(rng.random((8, 8)), (h // 8 + 1, w // 8 + 1))[:h, :w]
    elif content == "nonfinite":
        img[h // 2, w // 3] = np.nan
        img[h // 3, w // 2] = np.inf
        img[5:9, 7:9] = -3e19
        img[h - 9:h - 2, w - 20:w - 4] = 1e30
    return np.stack([img]).astype(np.float32)


@pytest.mark.parametrize("content", ["noisy", "columns", "rows", "clipped", "dark", "periodic", "nonfinite"])
@pytest.mark.parametrize("w,h,fp_mode", [(769, 727, 1), (769, 727, 2), (8203, 71, 2), (93, 6301, 1)])
def test_groups_match_oracle(w, h, fp_mode, content):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from oracle import pyoracle
    from vsfeel.torch_bm3d import Instance

    clip = _clip(content, w, h)
    kw = dict(sigma=3.0, block_step=4, bm_range=16)
    print(f"{w}x{h} fp_mode {fp_mode} {content}", flush=True)
    inst = Instance(1, h, w, fp_mode=fp_mode, **kw)
    g, _ = inst.groups(torch.from_numpy(clip).to("cuda:0"), 0)
    p = pyoracle.make_params(w, h, fp_mode=fp_mode, nthreads=NT, **kw)
    _, og = pyoracle.estimate(p, [clip[0]])
    bad = int((g != og).any(axis=(2, 3)).sum())
    assert bad == 0, f"{bad} of {g.shape[0] * g.shape[1]} groups differ"
