"""Device calls and host requests on one handle: what one leaves on the device must not reach the other's frames."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# window sets whose temporal search reads sums of the frames, kept on the device between requests
KW = dict(sigma=3.0, block_step=2, bm_range=5, ps_num=3, ps_range=7, extractor_exp=2)


# (lanes, graphs): a call on two lanes launches, one on one lane is captured and replayed
@pytest.mark.parametrize("lanes,graphs", [(None, 0), (None, 1), (1, 1)])
@pytest.mark.parametrize("radius", [1, 2])
def test_requests_after_device_calls_of_another_clip(radius, lanes, graphs, monkeypatch):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from vsfeel import BM3Dv2, Clip, _lib, synth

    w, h, n = 120, 104, 9
    host, dev = (np.ascontiguousarray(synth.shifted_clip(s, n, w, h, 3 / 255, (1.0, 2.0)), np.float32)
                 for s in (43, 44))
    fresh = BM3Dv2(Clip.gray(host), radius=radius, **KW)
    want = [fresh.get_frame(i)[0] for i in range(n)]

    if lanes is not None:
        monkeypatch.setenv("VSFEEL_BM3D_LANES", str(lanes))
    node = BM3Dv2(Clip.gray(host), radius=radius, **KW)
    L = _lib.load()
    assert L.vsfeel_bm3d_set_graphs(node._handle, graphs) == _lib.OK
    x = torch.from_numpy(dev).to("cuda:0")
    out = torch.empty_like(x)
    clip = _lib.DeviceClip()
    clip.data, clip.frame_stride, clip.pitch, clip.ref = x.data_ptr(), x.stride(0), x.stride(1), None

    def process():
        err = _lib.err_buf()
        stream = ctypes.c_void_p(torch.cuda.current_stream(x.device).cuda_stream)
        rc = L.vsfeel_bm3d_process_device(node._handle, ctypes.byref(clip), 0, n, out.data_ptr(), out.stride(1),
                                          out.stride(0), stream, err, len(err))
        assert rc == _lib.OK, err.value
        return out.cpu().numpy()

    first = process()
    assert np.array_equal(process(), first)
    for m in (5, 6, 4, 0, 8):
        got = node.get_frame(m)[0]
        assert np.array_equal(got, want[m]), f"frame {m} differs by {float(np.abs(got - want[m]).max())}"
        assert np.array_equal(process(), first), f"device frames differ after request {m}"
