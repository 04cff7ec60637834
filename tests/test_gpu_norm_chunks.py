"""The constraint norm's one launch over all chunks of a plan (every workgroup
finds its chunk by bisection): plans of 1, 2, 3 and many chunks, with chunk
sizes that are no multiple of a workgroup's 256 points, against the oracle."""
import numpy as np
import pytest

import oracle as O
import dgr
from dgr import workloads as W
from gpu_util import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nblocks", [1, 11, 12, 23, 24, 150])
def test_norm_over_many_chunks(monkeypatch, nblocks):
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    dgr.load()
    monkeypatch.setenv("DGR_CHUNK_POINTS", "4096")  # 11 blocks of 13^3 (343 points each) a chunk
    log(f"norm over chunks: {nblocks} blocks")
    t = W.uniform_13(nblocks)
    n = W.total_padded(t)
    c = np.random.default_rng(nblocks).standard_normal(n)
    plan = dgr.Plan(t, n)
    got = plan.constraint_norm(torch.from_numpy(c).cuda(), r1=0.0, r2=0.0)
    # sums of up to 51450 non-negative terms, in different orders: the mean of
    # squares is off by at most about 2 * (256 + 255) eps = 1.2e-13, its root by half
    assert got == pytest.approx(O.constraint_l2_norm(c, t, r1=0.0, r2=0.0), rel=1e-12, abs=0)
    plan.close()
