"""Batched eEM of sparse angle sets: buckets that take the tile projector hold no
transposed image, beside one that takes the staged form; each scan as alone."""
import numpy as np
import pytest

import oracle
from sscRaft import phantom as ph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("queue", ["1", "0"])
def test_batch_of_sparse_and_dense_scans(gpu, monkeypatch, queue):
    import torch
    from sscRaft import device as dv

    monkeypatch.setenv("RAFT_BATCH_QUEUE", queue)
    k = 4
    sizes = [(64, 12), (96, 20), (64, 12), (90, 90), (96, 20), (64, 12), (24, 5), (64, 12), (64, 12)]
    ys, angs = [], []
    for i, (n, a) in enumerate(sizes):
        ang = ph.uniform_angles(a)
        p = ph.poisson_log(oracle.radon(ph.phantoms(n, 1, config=6, first=70 + i), ang), 1e4, seed=70 + i)[0]
        ys.append(torch.from_numpy(np.maximum(p, 0).astype(np.float32)).cuda())
        angs.append(ang)
    plans = [dv.proj_plan_info(ang, n, n, n, 1, em=True)[0] for (n, a), ang in zip(sizes, angs)]
    assert plans[0] == 0 and plans[3] > 0
    ems = [torch.ones((n, n), device="cuda") for n, _ in sizes]
    paramf = np.array([[0, 0, 1, 0, 2.0 / n, 2.0 / n, 0] for n, _ in sizes], np.float32)
    dv.batch_device(None, angs, paramf, ys=ys, em=ems, iterations=k)
    for (n, a), y, ang, x in zip(sizes, ys, angs, ems):
        one = dv.eem_device(y[None].contiguous(), ang, k, with_kl=False)[0][0]
        assert torch.equal(x, one), (n, a)
