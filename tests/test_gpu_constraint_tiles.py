"""dgr_constraints walks the FP64 stage kernels' tile list, its own kernel taking
a 6-7 deep tile in two launches (5 planes and the rest). Interiors that end in
such a tile, alone and after regular ones, with short tiles along x and y, with
some blocks flagged: against the oracle (1e-12 of each output's size, as on the
other blocks), every interior point written and no other, and bit for bit as
with the tiling that has no such tiles. And what a plan holds on the device:
one tile list a precision, none of the constraints' own."""
import numpy as np
import pytest

import oracle as O
import dgr
from dgr import workloads as W
from gpu_util import host_state, interior_values, log, to_dev

pytestmark = pytest.mark.gpu

# z interiors 7, 11 = 5+6, 12 = 5+7, 16 = 5+5+6, 17 = 5+5+7, 8 = 5+3, 10 = 5+5; x, y parts of 4 to 7
SHAPES = [(13, 13, 13), (14, 15, 17), (16, 17, 18), (18, 13, 22), (13, 21, 23), (15, 18, 14), (17, 14, 16)]


@pytest.fixture(scope="module", autouse=True)
def _torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    dgr.load()
    yield


def table(flagged):
    t = np.zeros(len(SHAPES), dtype=W.BLOCK_DTYPE)
    t["sz"] = SHAPES
    n3 = np.prod(t["sz"].astype(np.int64), axis=1)
    t["offset"] = np.concatenate([[0], np.cumsum(n3)[:-1]])
    t["bflag"][flagged] = 63
    t["pmin"] = np.array([0.3, 0.1, -0.2]) + 3.0 * np.arange(len(t))[:, None]
    t["pmax"] = t["pmin"] + (t["sz"] - 1) * 0.1
    return t


@pytest.mark.parametrize("flagged", [[], [1, 3]])
def test_constraints_match_oracle_on_either_tiling(flagged):
    import torch
    t = table(flagged)
    st = host_state(t, seed=51, amp=1e-2)
    ham, mom, psi4 = O.constraints_batch(st, t, nthreads=8, psi4=True)
    ref = interior_values(np.concatenate([ham[None], mom, psi4, np.zeros((18, ham.size))]), t)[:6]
    u = to_dev(st)
    plan = dgr.Plan(t, st.shape[1])
    res = []
    for tiling in ("wt", "w"):
        for size in SHAPES:
            plan.set_tiling("fp64", size, tiling)
        log(f"constraints, tiling {tiling}, flagged {flagged}")
        out = torch.full((24, st.shape[1]), np.nan, dtype=torch.float64, device="cuda")
        plan.constraints(out[0], out[1:4], u, psi4=out[4:6])
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        inner = interior_values(got, t)[:6]
        assert np.isfinite(inner).all() and np.isfinite(got).sum() == inner.size
        e = np.abs(inner - ref).max(axis=1) / np.abs(ref).max(axis=1)
        log(f"  {e.max():.2e}")
        assert e.max() <= 1e-12
        res.append(inner)
    plan.close()
    assert np.array_equal(res[0], res[1])


def test_a_plan_holds_one_tile_list_a_precision():
    """100000 blocks of 13^3 (all on the same points: nothing is run): the block
    table (80 bytes a block), the stencil constants (3 x 88), the split path's tiles
    (44) and workgroups (8), and a list of one tile a block for each precision (44
    each), in whole pages of 2 MiB, with two pages for the small tables. A list
    of the constraints' own, two tiles a block, would be five pages more."""
    import torch
    n, page = 100000, 1 << 21
    t = np.zeros(n, dtype=W.BLOCK_DTYPE)
    t["sz"] = 13
    t["pmax"] = 1.2
    torch.cuda.synchronize()
    log("plan of 100000 blocks")
    first = dgr.Plan(t[:1], 13 ** 3)  # whatever a first plan sets up for good
    free = torch.cuda.mem_get_info()[0]
    plan = dgr.Plan(t, 13 ** 3)
    held = free - torch.cuda.mem_get_info()[0]
    plan.close()
    first.close()
    pages = sum(-(-n * size // page) for size in (80, 3 * 88, 44, 8, 44, 44))
    log(f"  {held / page:.1f} pages held, {pages} reckoned")
    assert held <= (pages + 2) * page
