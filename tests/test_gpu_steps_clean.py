"""bm3d_match_steps on content whose near matches its distances do not tell apart: gradients, cartoons, huge pixels.

Such blocks take the general search inside the kernel: groups against the oracle, and its time against content with
noise.  Its buffers' sizes differ by window set: distance rows (up to 64, of up to 31 columns) or a list.
"""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def _clip(content, frames, w, h):
    y, x = np.mgrid[0:h, 0:w].astype(np.float64)
    out = []
    for t in range(frames):
        img = 0.3 + 2e-4 * (x - 0.7 * t) + 1e-4 * y
        if content == "cartoon":
            img[h // 5:h // 2, w // 4 + t:w // 2 + t] = 0.8
            img[h // 3:2 * h // 3, w // 2:3 * w // 4] = 0.1
        elif content == "huge":
            img = img * 1e16
            img[h // 2:] *= 1e3
        elif content == "uniform":
            img[:] = 0.25
            img[h // 2:] = 2e19
        out.append(img)
    return np.stack(out).astype(np.float32)


@pytest.mark.parametrize("content", ["gradient", "cartoon", "huge", "uniform"])
@pytest.mark.parametrize("ps_num,ps_range", [(3, 5), (2, 15), (1, 15), (8, 4), (4, 8), (8, 15)])
@pytest.mark.parametrize("radius,fp_mode", [(1, 2), (2, 1)])
def test_groups_match_oracle(radius, fp_mode, ps_num, ps_range, content):
    torch = _torch()
    from oracle import pyoracle
    from vsfeel.torch_bm3d import Instance

    w, h = 101, 97  # 2208 blocks
    clip = _clip(content, 2 * radius + 1, w, h)
    kw = dict(sigma=3.0, block_step=2, bm_range=5, radius=radius, ps_num=ps_num, ps_range=ps_range)
    print(f"{content} {kw}", flush=True)
    inst = Instance(len(clip), h, w, fp_mode=fp_mode, **kw)
    g, _ = inst.groups(torch.from_numpy(clip).to("cuda:0"), radius)
    p = pyoracle.make_params(w, h, fp_mode=fp_mode, nthreads=NT, **kw)
    _, og = pyoracle.estimate(p, list(clip))
    bad = int((g != og).any(axis=(2, 3)).sum())
    assert bad == 0, f"{bad} of {g.shape[0] * g.shape[1]} groups differ"


def test_clean_content_costs_little_more_than_noise():
    # (before the general search took such blocks: 4.6 times as much, 930 us against 200)
    torch = _torch()
    from vsfeel.torch_bm3d import Instance

    w, h, n = 1280, 720, 3
    clean = _clip("cartoon", n, w, h)
    noisy = clean + np.random.default_rng(1).normal(0.0, 3 / 255, clean.shape).astype(np.float32)
    inst = Instance(n, h, w, sigma=3.0, block_step=4, bm_range=9, radius=1, ps_num=3, ps_range=5)
    inst.process(torch.from_numpy(noisy).to("cuda:0"))

    def temporal_ms(clip):
        x = torch.from_numpy(clip).to("cuda:0")
        inst.process(x)
        inst.set_timing(True)
        for _ in range(3):
            inst.process(x)
        (ms,) = [v[0] for k, v in inst.kernel_times().items() if "temporal" in k]
        inst.set_timing(False)
        return ms

    noise_ms, clean_ms = temporal_ms(noisy), temporal_ms(clean)
    assert clean_ms < 3.0 * noise_ms, f"{clean_ms:.3f} ms without noise, {noise_ms:.3f} with"
