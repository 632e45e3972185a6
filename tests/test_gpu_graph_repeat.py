"""Calls that repeat the last one's arguments (captured and replayed) among calls that do not (launched directly)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("frames,order", [
    (1, "AAABBBABAABA"),  # captures, replays, a capture after other arguments, direct launches between
    (5, "ABABAB"),        # several lanes, never the same twice in a row
    (5, "AAABAB"),        # a replay, then direct launches with the graph held
])
def test_frames_equal_direct_launches(frames, order):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from vsfeel import synth
    from vsfeel.torch_bm3d import Instance

    w, h = 131, 94
    clip = np.ascontiguousarray(synth.shifted_clip(61, frames, w, h, 3 / 255, (1.0, 0.0)), np.float32)
    x = torch.from_numpy(clip).to("cuda:0")
    kw = dict(sigma=3.0, block_step=4, bm_range=9)
    direct = Instance(frames, h, w, **kw)
    direct.set_graphs(False)
    inst = Instance(frames, h, w, **kw)
    outs = {c: torch.empty_like(x) for c in "AB"}
    for i, c in enumerate(order):
        x.copy_(torch.from_numpy(clip) * (1.0 - 0.05 * i))
        want = direct.process(x).cpu().numpy()
        outs[c].fill_(-1.0)
        inst.process(x, out=outs[c])
        assert np.array_equal(outs[c].cpu().numpy(), want), f"call {i} ({c}) differs"
