"""Device calls of libvsfeel_bm3d.so on the stand-in HIP runtime: driver.py STUB CALLS, as JSON on stdin and stdout.

A call is a list: ["limit", bytes], ["create", width, height, frames, arguments], ["process", output, first, count],
["get_frame", n], ["set_graphs", bits], ["free"].  Each prints what it logged, its return code and the bytes held.
"""

import ctypes
import json
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, os.path.join(ROOT, "vapoursynth-feel_amd"))

stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_limit.argtypes = [ctypes.c_size_t]
stub.stub_live.restype = ctypes.c_size_t
stub.stub_take_log.restype = ctypes.c_char_p

from vsfeel import BM3Dv2, Clip, Error, _lib  # noqa: E402

node, planes = None, {}


def call(op, *a):
    global node, planes
    L, err = _lib.load(), _lib.err_buf()
    if op == "limit":
        stub.stub_limit(a[0])
        return 0
    if op == "create":
        w, h, n, kw = a
        planes = {"clip": np.zeros((n, h, w), np.float32)}
        try:
            node = BM3Dv2(Clip.gray(planes["clip"]), **kw)
        except Error:
            return _lib.EDEVICE
        return 0
    if op == "process":
        name, first, count = a
        x = planes["clip"]
        out = planes.setdefault(name, np.empty_like(x))
        c = _lib.DeviceClip()
        c.data, c.frame_stride, c.pitch, c.ref = x.ctypes.data, x.shape[1] * x.shape[2], x.shape[2], None
        return L.vsfeel_bm3d_process_device(node._handle, ctypes.byref(c), first, count, out.ctypes.data, x.shape[2],
                                            x.shape[1] * x.shape[2], None, err, len(err))
    if op == "get_frame":
        node.get_frame(a[0])
        return 0
    if op == "set_graphs":
        return L.vsfeel_bm3d_set_graphs(node._handle, a[0])
    assert op == "free"
    node, planes = None, {}
    return 0


result = []
for c in json.load(sys.stdin):
    rc = call(*c)
    result.append(dict(rc=rc, log=stub.stub_take_log().decode().split("\n")[:-1], live=stub.stub_live()))
json.dump(result, sys.stdout)
