"""bench.py's roofline entry from kernel times: what is timed and what is counted
belong together."""
import types

import numpy as np
import pytest

import bench
from dgr import workloads as W


def blocks(sizes):
    t = np.zeros(len(sizes), dtype=W.BLOCK_DTYPE)
    t["sz"] = sizes
    return t


def line(t, kt, stages, precision="fp64"):
    wl = types.SimpleNamespace(blocks=t, npts=W.interior_points(t), key="a workload")
    return bench.roofline(wl, kt, stages, precision)


def test_fp64_interior_launches_are_one_entry():
    """dgr_plan_kernel_times divides the time of a launch on 7-deep tiles between
    the regular and the thin kind by points; the device ran one launch (two
    with regular tiles besides), so the entry is that whole time over all points."""
    t = blocks([(13, 13, 13)] * 4)
    r = line(t, {"fused_wide": (8 * 0.7 * 5 / 7, 8), "fused_thin": (8 * 0.7 * 2 / 7, 8), "fused_face": (0.0, 0)}, 8)
    assert r["launch_ms"] == pytest.approx(0.7) and r["stage_ms"] == pytest.approx(0.7)
    assert r["algorithmic_bytes_per_launch"] == pytest.approx(W.stage_bytes(t))
    assert r["achieved"] == pytest.approx(W.stage_bytes(t) / 0.7e-3 / 1e9, abs=0.06)  # printed to 0.1
    # 18 deep: 5 + 7, one launch of each
    t = blocks([(13, 13, 18)] * 4)
    r = line(t, {"fused_wide": (2 * (0.3 + 0.5 * 5 / 7), 2), "fused_thin": (2 * 0.5 * 2 / 7, 2)}, 2)
    assert r["launch_ms"] == pytest.approx(0.8)
    assert r["algorithmic_bytes_per_launch"] == pytest.approx(W.stage_bytes(t))
    # flagged blocks are an entry of their own
    t = blocks([(13, 13, 13)] * 4)
    t["bflag"][0] = 1
    r = line(t, {"fused_wide": (5.0, 1), "fused_thin": (2.0, 1), "fused_face": (1.0, 1)}, 1)
    assert r["launch_ms"] == pytest.approx(7.0) and r["stage_ms"] == pytest.approx(8.0)
    assert r["algorithmic_bytes_per_launch"] == pytest.approx(W.stage_bytes(t[1:]))
    assert r["per_kernel"]["fused_face"]["points"] == 343


def test_mixed_launches_are_entries_as_they_ran():
    t = blocks([(13, 13, 13)] * 4)
    r = line(t, {"fused_full": (8 * 0.9, 8), "fused_face": (0.0, 0)}, 8, "mixed")
    assert r["launch_ms"] == pytest.approx(0.9)
    assert r["algorithmic_bytes_per_launch"] == pytest.approx(W.stage_bytes(t))


def test_stage_bytes_are_what_four_stages_move():
    """Per interior point: stage 0 writes the step's start, the accumulator and the
    next stage (3 x 192), stages 1 and 2 read the first two and write the last two
    (4 x 192), stage 3 reads the accumulator and writes the result (2 x 192); each
    reads its padded state once. No stage writes a right-hand side."""
    t = blocks([(13, 13, 13), (19, 14, 31)])
    padded = 13 ** 3 + 19 * 14 * 31
    inner = 7 ** 3 + 13 * 8 * 25
    assert 4 * W.stage_bytes(t) == 192 * (4 * padded + (3 + 4 + 4 + 2) * inner)
