"""Device calls of several frames that repeat and change their arguments: every call equals direct launches."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_frames_equal_direct_launches():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from vsfeel import synth
    from vsfeel.torch_bm3d import Instance

    frames, w, h = 7, 131, 94
    kw = dict(sigma=3.0, block_step=8, bm_range=9)
    clip = np.ascontiguousarray(synth.shifted_clip(62, frames, w, h, 3 / 255, (1.0, 0.0)), np.float32)
    x = torch.from_numpy(clip).to("cuda:0")
    direct = Instance(frames, h, w, **kw)
    direct.set_graphs(False)
    inst = Instance(frames, h, w, **kw)
    inst.set_graphs(True)
    outs = {c: torch.empty_like(x) for c in "AB"}
    # the whole clip into A or B, or (C) two of its frames
    for i, c in enumerate("AABBAACCBB"):
        x.copy_(torch.from_numpy(clip) * (1.0 - 0.05 * i))
        want = direct.process(x).cpu().numpy()
        if c == "C":
            got = inst.process(x, first=1, count=2, out=outs["A"]).cpu().numpy()[:2]
            assert np.array_equal(got, want[1:3]), f"call {i} ({c}) differs"
        else:
            outs[c].fill_(-1.0)
            inst.process(x, out=outs[c])
            assert np.array_equal(outs[c].cpu().numpy(), want), f"call {i} ({c}) differs"
