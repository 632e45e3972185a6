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
def test_calls_on_several_lanes_are_never_captured(calls, frames, first, count, kw):
    # (a capture after such a graph was destroyed has ended in a segmentation fault)
    sequence = [["create", 96, 80, frames, kw], ["set_graphs", 1]]
    sequence += [["process", out, first, count] for out in "AABBBAA"]
    assert _kinds(calls(sequence)[2:]) == ["direct"] * 7


@pytest.mark.parametrize("frames,count,kw,lanes", [(1, 1, SPATIAL, None), (5, 1, SPATIAL, None), (5, 5, SPATIAL, 1),
                                                   (5, 5, TEMPORAL, 1)])
def test_calls_on_one_lane_replay_when_repeated(calls, frames, count, kw, lanes):
    sequence = [["create", 96, 80, frames, kw], ["set_graphs", 1]]
    sequence += [["process", out, 0, count] for out in "AAABABB"]
    got = _kinds(calls(sequence, lanes)[2:])
    assert got == ["direct", "capture", "replay", "direct", "replay", "direct", "capture"]


def test_other_calls_leave_a_held_graph(calls):
    # one frame (captured), then several (launched), then the frame again
    sequence = [["create", 96, 80, 5, SPATIAL]] + [["process", "A", 0, n] for n in (1, 1, 5, 5, 5, 1)]
    assert _kinds(calls(sequence)[1:]) == ["direct", "capture", "direct", "direct", "direct", "replay"]


# 2 radius ps_num insertions: as many as always bin, and few on a frame of 32768 blocks and more
@pytest.mark.parametrize("w,h,kw", [
    (120, 104, dict(sigma=3.0, block_step=4, bm_range=5, radius=2, ps_num=2, ps_range=4)),
    (376, 361, dict(sigma=3.0, block_step=2, bm_range=3, radius=1, ps_num=2, ps_range=4)),
])
def test_no_room_for_the_bins_leaves_the_atomic_scatter(calls, w, h, kw):
    def run(limit):
        return calls([["limit", limit], ["create", w, h, 3, kw], ["process", "A", 0, 3], ["free"]])[1:]

    def bins(result):
        return any("bm3d_gather" in line for line in result[1]["log"])

    roomy = run(1 << 50)
    assert roomy[0]["rc"] == roomy[1]["rc"] == 0 and bins(roomy)
    everything = roomy[0]["live"]
    # the records of a lane: 64 floats for each of 7 blocks of every group
    ny, nx = ((q - 8 + kw["block_step"] - 1) // kw["block_step"] + 1 for q in (h, w))
    records = nx * ny * 7 * 64 * 4
    assert everything > 2 * records
    for limit in (everything - 1, everything - records, everything - records - 1, everything - 2 * records):
        tight = run(limit)
        assert tight[0]["rc"] == tight[1]["rc"] == 0, (limit, everything)
        assert not bins(tight) and any("bm3d_estimate" in line for line in tight[1]["log"])
        # what was made before one of them failed is given back
        assert tight[0]["live"] <= everything - 2 * records
        assert tight[2]["live"] == 0


def test_no_room_for_the_sums_leaves_the_search_without_them(calls):
    # 3 windows of 15 rows on 2448 blocks and more, searched with planes of sums
    w, h = 120, 104
    kw = dict(sigma=3.0, block_step=2, bm_range=5, radius=1, ps_num=3, ps_range=7)

    def run(limit):
        return calls([["limit", limit], ["create", w, h, 3, kw], ["process", "A", 0, 3], ["free"]])[1:]

    def sums(result):
        return any("bm3d_sum_planes" in line for line in result[1]["log"])

    roomy = run(1 << 50)
    assert roomy[0]["rc"] == roomy[1]["rc"] == 0 and sums(roomy)
    everything = roomy[0]["live"]
    # a lane's: 3 planes for each of 3 frames, rows of a multiple of 16 floats, 40 rows past the frame
    planes = 3 * 3 * ((w + 15) // 16 * 16) * (h + 40) * 4
    needed = everything - 2 * planes
    for limit in (everything - 1, everything - planes, everything - planes - 1, needed + planes // 2, needed):
        tight = run(limit)
        assert tight[0]["rc"] == tight[1]["rc"] == 0, (limit, everything)
        assert sums(tight) == (limit >= needed + planes)
        assert any("bm3d_match" in line for line in tight[1]["log"])
        assert tight[2]["live"] == 0


def _bins(result):
    assert result["rc"] == 0, result
    return any("bm3d_gather" in line for line in result["log"])


# 8 insertions and more, or 4 to 7 where blocks lie close together on frames of many blocks
@pytest.mark.parametrize("w,h,kw,binned", [
    (640, 360, dict(block_step=8, radius=2, ps_num=2), True),
    (640, 360, dict(block_step=4, radius=1, ps_num=3), False),
    (768, 720, dict(block_step=3, radius=1, ps_num=2), True),
    (768, 720, dict(block_step=4, radius=1, ps_num=2), False),
    (1280, 720, dict(block_step=4, radius=1, ps_num=2, bm_range=12), True),
    (1280, 720, dict(block_step=4, radius=1, ps_num=2, bm_range=16), False),
    (1920, 1080, dict(block_step=4, radius=1, ps_num=2, bm_range=16), True),
    (1920, 1080, dict(block_step=4, radius=1, ps_num=2, bm_range=20), False),
    (1920, 1080, dict(block_step=4, radius=2, ps_num=1), False),
    (1920, 1080, dict(block_step=5, radius=1, ps_num=3), False),
    (2560, 1440, dict(block_step=5, radius=1, ps_num=2), True),
    (2560, 1440, dict(block_step=5, radius=2, ps_num=1), False),
    (3840, 2160, dict(block_step=8, radius=1, ps_num=2), False),
])
def test_which_calls_bin(calls, w, h, kw, binned):
    kw = dict(dict(sigma=3.0, bm_range=9, ps_range=4), **kw)
    assert _bins(calls([["create", w, h, 2, kw], ["process", "A", 0, 1]], lanes=1)[1]) == binned


def test_bins_hold_what_dense_blocks_send(calls):
    # (lists of 512 blocks overflowed at block_step 2 and 3, which was slower than no binning at all)
    w, h, step = 512, 512, 2
    live = {}
    for ps_num in (2, 3, 4):
        kw = dict(sigma=3.0, block_step=step, bm_range=7, radius=1, ps_num=ps_num, ps_range=3)
        result = calls([["create", w, h, 2, kw], ["process", "A", 0, 2]])
        assert _bins(result[1])
        live[ps_num] = result[0]["live"]
    # 2 lanes, 2 other frames, 16 x 16 cells, 8 bytes a block: 1024 blocks a cell, then 2048 and 2048
    assert live[3] - live[2] == 2 * 2 * 16 * 16 * 8 * 1024
    assert live[4] == live[3]


# the frames of the GPU tests of either kernel, and the line between them (32768 blocks, 64 x 44 pixels)
@pytest.mark.parametrize("w,h,bm_range,block_step,kernel", [
    (769, 727, 16, 4, "bm3d_match_cols"), (8203, 71, 16, 4, "bm3d_match_cols"), (93, 6301, 16, 4, "bm3d_match_cols"),
    (64, 9000, 16, 4, "bm3d_match_cols"), (13202, 44, 16, 4, "bm3d_match_cols"),
    (481, 275, 16, 4, "bm3d_match_rows"), (64, 40, 16, 4, "bm3d_match_rows"), (13202, 43, 16, 4, "bm3d_match_rows"),
    (769, 727, 15, 4, "bm3d_match_rows"), (1920, 1080, 16, 5, "bm3d_match_rows"),
])
@pytest.mark.parametrize("radius", [0, 1])
def test_which_kernel_searches(calls, w, h, bm_range, block_step, kernel, radius):
    kw = dict(sigma=3.0, block_step=block_step, bm_range=bm_range, radius=radius)
    result = calls([["create", w, h, 2, kw], ["process", "A", 0, 1]], lanes=1)[1]
    assert result["rc"] == 0
    spatial = {name for name in ("bm3d_match_cols", "bm3d_match_rows") if any(name in x for x in result["log"])}
    assert spatial == {kernel}


# window sets of more than 32 rows (or wider than 25 columns), from 2048 blocks on, but not where 5 windows and more
# overlap widely, or on small frames
@pytest.mark.parametrize("w,h,block_step,ps_num,ps_range,kernel", [
    (101, 97, 2, 3, 7, "bm3d_match_steps"), (101, 97, 2, 8, 4, "bm3d_match_steps"),
    (101, 97, 2, 2, 8, "bm3d_match_steps"), (101, 97, 2, 1, 15, "bm3d_match_steps"),
    (101, 97, 2, 8, 7, "bm3d_match_steps"), (101, 97, 2, 8, 15, "bm3d_match_steps"),
    (101, 97, 2, 8, 8, "bm3d_matchI"), (101, 97, 2, 5, 12, "bm3d_matchI"), (101, 97, 2, 7, 4, "bm3d_matchI"),
    (1280, 720, 8, 7, 4, "bm3d_match_steps"), (101, 97, 2, 3, 16, "bm3d_matchI"), (91, 89, 2, 3, 7, "bm3d_matchI"),
    (101, 97, 2, 2, 7, "bm3d_match_predictive"), (101, 97, 2, 3, 4, "bm3d_match_predictive"),
])
def test_which_kernel_searches_the_other_frames(calls, w, h, block_step, ps_num, ps_range, kernel):
    kw = dict(sigma=3.0, block_step=block_step, bm_range=5, radius=1, ps_num=ps_num, ps_range=ps_range)
    result = calls([["create", w, h, 3, kw], ["process", "A", 0, 1]], lanes=1)[1]
    assert result["rc"] == 0
    names = ("bm3d_match_steps", "bm3d_match_predictive", "bm3d_matchI")  # (the last: bm3d_match<..>, mangled)
    assert {name for name in names if any(name in line for line in result["log"])} == {kernel}
