"""What the device calls allocate, launch and capture, on a stand-in HIP runtime (no GPU: kernels are only logged)."""

from __future__ import annotations

import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "hip_stub")
LIB = os.path.join(ROOT, "vapoursynth-feel_amd", "vsfeel", "libvsfeel_bm3d.so")


@pytest.fixture(scope="module")
def calls(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    if not os.path.exists(LIB):
        pytest.skip("libvsfeel_bm3d.so is not built")
    so = str(tmp_path_factory.mktemp("hip_stub") / "libstub_hip.so")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    os.path.join(STUB, "stub_hip.cpp"), "-o", so], check=True, capture_output=True, text=True)

    def run(sequence, lanes=None):
        env = dict(os.environ)
        env.pop("VSFEEL_BM3D_LANES", None)
        if lanes is not None:
            env["VSFEEL_BM3D_LANES"] = str(lanes)
        r = subprocess.run([sys.executable, os.path.join(STUB, "driver.py"), so], input=json.dumps(sequence),
                           capture_output=True, text=True, timeout=120, env=env)
        assert r.returncode == 0, r.stderr
        return json.loads(r.stdout)

    return run


def _kinds(results):
    """Per call: "direct", "capture" (and replay) or "replay"."""
    kinds = []
    for r in results:
        assert r["rc"] == 0, r
        assert any(line.startswith("kernel ") for line in r["log"]), r
        kinds.append("capture" if "capture" in r["log"] else "replay" if "replay" in r["log"] else "direct")
    return kinds


SPATIAL = dict(sigma=3.0, block_step=4, bm_range=9)
TEMPORAL = dict(SPATIAL, radius=1)


@pytest.mark.parametrize("frames,first,count,kw", [
    (5, 0, 5, SPATIAL), (5, 1, 2, SPATIAL), (5, 0, 5, TEMPORAL), (5, 2, 1, TEMPORAL), (1, 0, 1, TEMPORAL),
])
def test_calls_on_several_lanes_are_captured_once(calls, frames, first, count, kw):
    # (capturing such a sequence again after other arguments has ended in a segmentation fault)
    sequence = [["create", 96, 80, frames, kw], ["set_graphs", 1]]
    sequence += [["process", out, first, count] for out in "AABBBAA"]
    sequence += [["set_graphs", 0], ["set_graphs", 1]] + [["process", out, first, count] for out in "AAABB"]
    got = calls(sequence)
    assert _kinds(got[2:9]) == ["direct", "capture"] + ["direct"] * 3 + ["replay"] * 2
    assert _kinds(got[11:]) == ["direct"] * 5


@pytest.mark.parametrize("frames,count,kw,lanes", [(1, 1, SPATIAL, None), (5, 1, SPATIAL, None), (5, 5, SPATIAL, 1),
                                                   (5, 5, TEMPORAL, 1)])
def test_calls_on_one_lane_replay_when_repeated(calls, frames, count, kw, lanes):
    sequence = [["create", 96, 80, frames, kw], ["set_graphs", 1]]
    sequence += [["process", out, 0, count] for out in "AAABABB"]
    got = _kinds(calls(sequence, lanes)[2:])
    assert got == ["direct", "capture", "replay", "direct", "replay", "direct", "capture"]


@pytest.mark.parametrize("counts", [(1, 1, 5, 5, 5, 1), (5, 5, 1, 1, 1, 5)])
def test_other_calls_leave_a_held_graph(calls, counts):
    # one frame or several (captured), then several or one (launched), then the first again
    sequence = [["create", 96, 80, 5, SPATIAL]] + [["process", "A", 0, n] for n in counts]
    assert _kinds(calls(sequence)[1:]) == ["direct", "capture", "direct", "direct", "direct", "replay"]
