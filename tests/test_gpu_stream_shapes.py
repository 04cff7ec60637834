"""The FP64 stage kernels (csrc/stream_fp64.h) on the tile shapes where they can
go wrong: interior extents that leave parts of 4, 5 and 6 points along x and y
(short rows in the staging tables), 6- and 7-deep tiles and 5-deep ones with a
remainder along z, 3-point parts on flagged blocks, and every combination of
flagged low and high faces on them; alone, and with the padding read from
neighbours. Bounds as for the other sizes: 1e-12 of each variable's largest
right-hand side (stencils round as the oracle's do, the equations differ by a
few units of rounding), 1e-11 of the increments of an RK4 step."""
import numpy as np
import pytest

import oracle as O
import dgr
from dgr import workloads as W
from gpu_util import gpu_rhs, host_state, interior_values, log, normwise, oracle_params, to_dev

pytestmark = pytest.mark.gpu

# padded sizes: interior x, y parts 4+4, 5+4, 5+5, 6+5, 6+6, 5+5+5; z 7, 5+2, 5+3, 5+5+1, 5+5+2, 5+5+3
SHAPES = [(14, 15, 13), (16, 17, 14), (18, 21, 16), (13, 19, 17), (21, 14, 18), (17, 13, 19), (15, 18, 12 + 13)]


@pytest.fixture(scope="module", autouse=True)
def _torch_cuda():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    dgr.load()
    yield


def table(flags):
    t = np.zeros(len(SHAPES), dtype=W.BLOCK_DTYPE)
    t["sz"] = SHAPES
    n3 = np.prod(t["sz"].astype(np.int64), axis=1)
    t["offset"] = np.concatenate([[0], np.cumsum(n3)[:-1]])
    t["bflag"] = flags
    t["pmin"] = np.array([0.3, 0.1, -0.2]) + 3.0 * np.arange(len(t))[:, None]
    t["pmax"] = t["pmin"] + (t["sz"] - 1) * 0.1
    return t


@pytest.mark.parametrize("flags", [0, 1, 2, 4, 8, 16, 32, 63, 0b100101, 0b011010])
@pytest.mark.parametrize("cako", [0, 1])
def test_rhs_matches_oracle(flags, cako):
    t = table(flags)
    st = host_state(t, seed=31)
    p = dgr.default_params(ko_sigma=0.4, eta_central=2.0, eta_outer=2.0, cako_enabled=cako)
    log(f"shapes: rhs flags {flags} cako {cako}")
    got = interior_values(gpu_rhs(t, st, p), t)
    ref = interior_values(O.bssnrhs_batch(st, t, oracle_params(p), nthreads=8), t)
    assert normwise(got, ref).max() <= 1e-12


@pytest.mark.parametrize("flags", [0, 63])
def test_rk4_step_matches_oracle(flags):
    import torch
    t = table(flags)
    st = host_state(t, seed=32)
    p = dgr.default_params(ko_sigma=0.4, eta_central=2.0, eta_outer=2.0)
    log(f"shapes: rk4 flags {flags}")
    plan = dgr.Plan(t, st.shape[1])
    u = to_dev(st)
    plan.rk4_steps(u, 0.02, p, nsteps=2)
    torch.cuda.synchronize()
    assert plan.status() == 0
    ref = st.copy()
    for _ in range(2):
        O.rk4_step(ref, t, 0.02, oracle_params(p), enforce_per_stage=True, nthreads=8)
    assert normwise(interior_values(u.cpu().numpy() - st, t), interior_values(ref - st, t)).max() <= 1e-11
    plan.close()


@pytest.mark.parametrize("size", [(14, 16, 17), (18, 13, 18), (15, 17, 14)])
def test_rk4_with_linked_padding_matches_oracle(size):
    import torch
    h = 0.05
    cells = np.array([(a, b, c) for c in range(2) for b in range(3) for a in range(2)])
    t = np.zeros(len(cells), dtype=W.BLOCK_DTYPE)
    t["sz"] = size
    t["offset"] = np.arange(len(t)) * int(np.prod(size))
    t["pmin"] = np.array([-0.4, -0.3, -0.2]) + cells * (np.array(size) - 7) * h
    t["pmax"] = t["pmin"] + (np.array(size) - 1) * h
    st = np.zeros((24, W.total_padded(t)))
    rng = np.random.default_rng(5)
    k, a = rng.uniform(1, 4, (24, 3)), rng.uniform(-1e-2, 1e-2, 24)
    for b in range(len(t)):
        z, y, x = np.meshgrid(*[t["pmin"][b][d] + h * np.arange(size[d]) for d in (2, 1, 0)], indexing="ij")
        for v in range(24):
            st[v, t["offset"][b]:t["offset"][b] + x.size] = (
                (v in (0, 1, 12, 15, 17)) + a[v] * np.sin(k[v, 0] * x + k[v, 1] * y + k[v, 2] * z)).ravel()
    p = dgr.default_params(ko_sigma=0.4)
    log(f"shapes: linked rk4 {size}")
    plan = dgr.Plan(t, st.shape[1])
    plan.set_halo_refresh(True)
    u = to_dev(st)
    plan.rk4_steps(u, 0.02, p, nsteps=2)
    torch.cuda.synchronize()
    assert plan.status() == 0
    ref = st.copy()
    for _ in range(2):
        O.rk4_step_halo(ref, t, W.neighbors(t), 0.02, oracle_params(p), enforce_per_stage=True, nthreads=8)
    got = u.cpu().numpy()
    assert normwise(interior_values(got - st, t), interior_values(ref - st, t)).max() <= 1e-11
    assert np.abs(got - ref).max() <= 1e-11 * np.abs(ref - st).max()
    plan.close()
