"""The FP64 stage kernels that read padding from neighbours, in every form: blocks
with flagged faces among others, the standard gauge and the reference's other
builds (Rochester gauge; slow-start lapse with the eta function), in plans of at
most 256 tiles (one launch a stage) and of more (a launch a kind of tile), on
block sizes with short tiles. Two RK4 steps against the oracle's, which fill the
padding from the neighbours before every stage: per variable within 1e-11 of the
largest increment, the bound of the other refreshed steps, or within 4 times the
oracle's own response to a 2e-16 perturbation of its input where that is larger
(B under the Rochester gauge moves by its dissipation alone, 1e-8 of its size, so
the sum's rounding shows in the increment)."""
import numpy as np
import pytest

import oracle as O
import dgr
from dgr import workloads as W
from gpu_util import interior_values, log, normwise, oracle_params, to_dev

H, DT = 0.05, 0.02
GAUGES = {"standard": dict(), "rochester": dict(rochester=1, xi=(2.0, 3.0, 5.0)),
          "ssl_etafunc": dict(ssl=1, time=7.5, eta_func=1, eta_r0=0.9, eta_power=(2.0, 1.0))}
# (lattice, padded size): tiles 4+4 x 5+5 x 5+6 and 6+6 x 7 x 5+7 points
SMALL, LARGE = ((2, 2, 2), (18, 13, 18)), ((4, 3, 3), (14, 16, 17))


def lattice(shape, size, flagged):
    cells = np.array([(a, b, c) for c in range(shape[2]) for b in range(shape[1]) for a in range(shape[0])])
    t = np.zeros(len(cells), dtype=W.BLOCK_DTYPE)
    t["sz"] = size
    t["offset"] = np.arange(len(t)) * int(np.prod(size))
    t["pmin"] = np.array([0.3, 0.1, -0.2]) + cells * (np.array(size) - 7) * H
    t["pmax"] = t["pmin"] + (np.array(size) - 1) * H
    if flagged:  # low x and high z faces of the lattice, and one block all around
        t["bflag"] = (cells[:, 0] == 0) * 1 + (cells[:, 2] == shape[2] - 1) * 32
        t["bflag"][np.nonzero(t["bflag"] == 0)[0][0]] = 63
    return t


def state(t):
    """Waves on a flat metric with lapse 0.8 and chi 0.6."""
    st = np.zeros((24, W.total_padded(t)))
    rng = np.random.default_rng(5)
    k, a = rng.uniform(1, 4, (24, 3)), rng.uniform(-1e-2, 1e-2, 24)
    flat = {0: 0.8, 1: 0.6, 12: 1.0, 15: 1.0, 17: 1.0}
    for b in range(len(t)):
        z, y, x = np.meshgrid(*[t["pmin"][b][d] + H * np.arange(t["sz"][b][d]) for d in (2, 1, 0)], indexing="ij")
        for v in range(24):
            st[v, t["offset"][b]:t["offset"][b] + x.size] = (
                flat.get(v, 0.0) + a[v] * np.sin(k[v, 0] * x + k[v, 1] * y + k[v, 2] * z)).ravel()
    return st


def oracle_steps(t, st, gauge):
    ref = st.copy()
    for i in range(2):
        p = params(gauge)
        p.time += i * DT
        O.rk4_step_halo(ref, t, W.neighbors(t), DT, oracle_params(p), enforce_per_stage=True, nthreads=8)
    return ref


def params(gauge):
    return dgr.default_params(ko_sigma=0.4, **GAUGES[gauge])


def increment(u, st, t):
    return interior_values(u - st, t)


@pytest.mark.gpu
@pytest.mark.parametrize("flagged", [0, 1])
@pytest.mark.parametrize("gauge", GAUGES)
@pytest.mark.parametrize("plan_size", ["small", "large"])
def test_rk4_with_linked_padding_matches_oracle(plan_size, gauge, flagged):
    import torch
    t = lattice(*(SMALL if plan_size == "small" else LARGE), flagged)
    st = state(t)
    ref = oracle_steps(t, st, gauge)
    near = st * (1 + 2e-16 * np.random.default_rng(1).standard_normal(st.shape))
    sens = normwise(increment(oracle_steps(t, near, gauge), near, t), increment(ref, st, t))
    log(f"refreshed stages: {plan_size} plan, {gauge}, flagged {flagged}, sensitivity {sens.max():.1e}")
    plan = dgr.Plan(t, st.shape[1])
    plan.set_halo_refresh(True)
    u = to_dev(st)
    plan.rk4_steps(u, DT, params(gauge), nsteps=2)
    torch.cuda.synchronize()
    assert plan.status() == 0
    got = u.cpu().numpy()
    plan.close()
    e = normwise(increment(got, st, t), increment(ref, st, t))
    log(f"  normwise {e.max():.2e}")
    assert (e <= np.maximum(1e-11, 4 * sens)).all(), e
    # with the refresh, neighbours hold the padding the oracle filled
    assert np.abs(got - ref).max() <= 1e-11 * np.abs(ref - st).max()
