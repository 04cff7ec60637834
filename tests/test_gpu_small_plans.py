"""Small plans run all their FP64 tiles in one launch (k_stream_small), larger
ones and those of one kind a launch a kind: the same tile bodies, so the two
routes agree bit for bit. With kernel timing on a plan takes the second route."""
import numpy as np
import pytest

import oracle as O
import dgr
from dgr import workloads as W
from gpu_util import host_state, interior_values, log, normwise, oracle_params, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    dgr.load()
    yield


def table(sizes, flags):
    t = np.zeros(len(sizes), dtype=W.BLOCK_DTYPE)
    t["sz"] = sizes
    n3 = np.prod(t["sz"].astype(np.int64), axis=1)
    t["offset"] = np.concatenate([[0], np.cumsum(n3)[:-1]])
    t["bflag"] = flags
    t["pmin"] = np.array([0.3, 0.1, -0.2]) + 3.0 * np.arange(len(t))[:, None]
    t["pmax"] = t["pmin"] + (t["sz"] - 1) * 0.1
    return t


S13, S16, S18 = (13, 13, 13), (14, 15, 16), (16, 17, 18)
# a flagged 13^3 block is two tiles, an unflagged one a 7-deep tile
CASES = {
    "face+full": ([S13] * 3, [5, 0, 0]),
    "face+wide": ([S16] * 2, [63, 0]),
    "wide+full": ([S18] * 2, [0, 0]),
    "all": ([S13, S16, S18, S13], [10, 0, 0, 0]),
    "256 tiles": ([S13] * 160, [1] * 96 + [0] * 64),
    "257 tiles": ([S13] * 161, [1] * 96 + [0] * 65),
}


def both(t, run):
    """run(plan, ...) without and with kernel timing."""
    import torch
    out = []
    for timing in (False, True):
        plan = dgr.Plan(t, W.total_padded(t))
        plan.set_timing(timing)
        out.append(run(plan))
        torch.cuda.synchronize()
        plan.close()
    return out


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("rochester", [0, 1])
def test_one_launch_equals_a_launch_a_kind(case, rochester):
    import torch
    t = table(*CASES[case])
    st = host_state(t, seed=41)
    p = dgr.default_params(ko_sigma=0.4, rochester=rochester)
    log(f"small plan {case} rochester {rochester}")

    def rhs(plan):
        d = to_dev(st)
        out = torch.zeros_like(d)
        plan.rhs(out, d, p)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    def step(plan):
        d = to_dev(st)
        plan.rk4_step(d, 1e-3, p)
        torch.cuda.synchronize()
        return d.cpu().numpy()

    a, b = both(t, rhs)
    assert np.array_equal(a, b, equal_nan=True)
    if not rochester and len(t) < 100:
        ref = interior_values(O.bssnrhs_batch(st, t, oracle_params(p), nthreads=8), t)
        assert normwise(interior_values(a, t), ref).max() <= 1e-12
    a, b = both(t, step)
    assert np.array_equal(a, b, equal_nan=True)


def test_one_launch_with_the_padding_refresh():
    import torch
    t = W.lattice(shape=(3, 2, 2), n=13, h=0.05)
    t["bflag"][:4] = 21
    st = host_state(t, seed=42)
    p = dgr.default_params(ko_sigma=0.4)
    log("small plan, padding refresh")

    def steps(plan):
        plan.link_neighbors()
        plan.set_halo_refresh(True)
        d = to_dev(st)
        for _ in range(2):
            plan.rk4_step(d, 1e-3, p)
        torch.cuda.synchronize()
        return d.cpu().numpy()

    a, b = both(t, steps)
    assert np.array_equal(a, b, equal_nan=True)


def test_each_kind_counts_one_launch_a_stage():
    """Kernel times of a plan with regular and 7-deep tiles: the 7-deep launch's
    regular part adds its time to the regular launch's, not a launch."""
    import torch
    t = table(*CASES["wide+full"])
    plan = dgr.Plan(t, W.total_padded(t))
    plan.set_timing(True)
    d = to_dev(host_state(t, seed=43))
    out = torch.zeros_like(d)
    log("launch counts by kind")
    for _ in range(3):
        plan.rhs(out, d, dgr.default_params())
    torch.cuda.synchronize()
    kt = plan.kernel_times()
    plan.close()
    assert kt["fused_wide"][1] == 3 and kt["fused_thin"][1] == 3, kt
    assert kt["fused_wide"][0] > 0 and kt["fused_thin"][0] > 0
