"""bm3d_match_steps (temporal search of larger window sets) against the oracle.

The kernel's edges: 16 and 32 lanes a window, one pass and several, windows
clipped on every side; and the content its expanded distances do not resolve,
which has to end in the exact distances: equal, huge and non-finite pixels.
Also the frames whose sums a search reads: of a clip rewritten between calls,
and of requests in any order.
"""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NT = min(16, os.cpu_count() or 1)

# (ps_num, ps_range): rows of all windows past 32, or a window past 25 columns
WINDOWS = [(3, 7), (8, 4), (2, 8), (1, 15), (8, 15)]


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def _clip(content, frames, w, h):
    from vsfeel import synth
    clip = np.array(synth.shifted_clip(31, frames, w, h, 0.0 if content == "clean" else 3 / 255, (1.0, -2.0)),
                    np.float32)
    if content == "bars":
        clip[:, : h // 4] = 0.0
        clip[:, :, w - w // 5:] = 0.25
    elif content == "columns":
        clip[:] = 0.5 + 0.2 * np.sin(np.arange(w) / 1.1)[None, None, :]
        clip[1:, h // 3] += 0.125
    elif content == "nonfinite":
        clip[0, h // 2, w // 3] = np.nan
        clip[-1, h // 3, w // 2] = np.inf
        clip[:, 5:9, 7:9] = -3e19
        clip[1:, h - 9:h - 2, w - 20:w - 4] = 1e30
        clip[:, 40:52, 20:32] = 2e15
    return clip


@pytest.mark.parametrize("content", ["noisy", "bars", "clean", "columns", "nonfinite"])
@pytest.mark.parametrize("ps_num,ps_range", WINDOWS)
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


@pytest.mark.parametrize("radius", [1, 2])
def test_sums_are_of_the_frames_searched(radius):
    torch = _torch()
    from vsfeel import BM3Dv2, Clip, synth
    from vsfeel.torch_bm3d import Instance

    w, h, n = 120, 104, 8
    kw = dict(sigma=3.0, block_step=2, bm_range=5, radius=radius, ps_num=3, ps_range=7, extractor_exp=2)
    clips = [np.ascontiguousarray(synth.shifted_clip(s, n, w, h, 3 / 255, (1.0, 2.0)), np.float32) for s in (41, 42)]

    def fresh(c):
        return Instance(n, h, w, **kw).process(torch.from_numpy(c).to("cuda:0")).cpu().numpy()

    want = [fresh(c) for c in clips]
    # one instance and one buffer, rewritten between calls; parts of the clip
    inst = Instance(n, h, w, **kw)
    x = torch.from_numpy(clips[0]).to("cuda:0")
    assert np.array_equal(inst.process(x).cpu().numpy(), want[0])
    x.copy_(torch.from_numpy(clips[1]))
    assert np.array_equal(inst.process(x, first=3, count=2).cpu().numpy(), want[1][3:5])
    assert np.array_equal(inst.process(x).cpu().numpy(), want[1])
    # requests of single frames in any order
    node = BM3Dv2(Clip.gray(clips[1]), **kw)
    for m in [5, 0, 7, 2, 3, 3, 4, 1, 6, 0]:
        assert np.array_equal(node.get_frame(m)[0], want[1][m]), f"frame {m} differs"
