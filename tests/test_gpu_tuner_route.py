"""dgr_plan_autotune times each block size on the route the plan's stages take:
one launch for all tiles where the whole plan has at most 256 of more than one
kind, a launch a kind of tile otherwise, whatever the sampled size alone has."""
import numpy as np
import pytest

import dgr
from dgr import workloads as W
from gpu_util import host_state, log, to_dev

pytestmark = pytest.mark.gpu

# (sizes, flagged blocks): 300 tiles, and 8 of another size whose own are of two
# kinds; a few tiles of one kind, beside those of a flagged block
CASES = {"launch a kind": ([(13, 13, 13)] * 300 + [(16, 13, 18)] * 2, 0),
         "one launch": ([(13, 13, 13)] * 4, 1)}


def table(sizes, flagged):
    t = np.zeros(len(sizes), dtype=W.BLOCK_DTYPE)
    t["sz"] = sizes
    n3 = np.prod(t["sz"].astype(np.int64), axis=1)
    t["offset"] = np.concatenate([[0], np.cumsum(n3)[:-1]])
    t["bflag"][:flagged] = 63
    t["pmin"] = np.array([0.3, 0.1, -0.2]) + 3.0 * np.arange(len(t))[:, None]
    t["pmax"] = t["pmin"] + (t["sz"] - 1) * 0.1
    return t


@pytest.mark.parametrize("case", CASES)
def test_tuner_times_the_route_the_plan_takes(case):
    import torch
    t = table(*CASES[case])
    log(f"tuner route: {case}")
    plan = dgr.Plan(t, W.total_padded(t))
    u = to_dev(host_state(t, seed=61))
    out = torch.zeros_like(u)
    p = dgr.default_params()

    def stage_kernels(call):
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            call()
            torch.cuda.synchronize()
        return {"one launch" if "k_stream_small" in e.name else "launch a kind"
                for e in prof.events() if "k_stream" in e.name}

    assert stage_kernels(lambda: plan.rhs(out, u, p)) == {case}
    assert stage_kernels(lambda: plan.autotune(out, u, p)) == {case}
    assert stage_kernels(lambda: plan.rhs(out, u, p)) == {case}
    plan.close()
