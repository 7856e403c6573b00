"""The longest padded rows of the FP64 transform form of the row filter: its LDS
(the padded rows too, for the direct sum of rows that are not finite) is the CU's
160 KB to within 128 bytes."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad", [(6425, 2), (6420, 2), (3855, 4)])  # 19275 and 19260 bins
def test_longest_rows(gpu, n, pad):
    import torch
    from sscRaft import device as dv

    a, s = 2, 3
    rng = np.random.default_rng(n)
    y = (1.0 + rng.random((s, a, n))).astype(np.float32)
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, 0.0], np.float32)
    parami = np.array([n, a, s, n, pad, 0, 0, 7, 0, 0], np.int32)
    print(f"lowpass n={n} pad={pad}", flush=True)
    t = torch.from_numpy(y).cuda()
    r = dv.lowpass_device(t, paramf, parami)
    x = (t if r is None else r).cpu().numpy()
    want = oracle.lowpass(y, paramf, parami)
    # FP64 rows rounded once
    assert np.linalg.norm(x - want) <= 1e-6 * np.linalg.norm(want)
    y[1, 0, 5] = np.nan  # the direct sum
    t = torch.from_numpy(y).cuda()
    r = dv.lowpass_device(t, paramf, parami)
    z = (t if r is None else r).cpu().numpy()
    assert np.isnan(z[1, 0]).any() and np.isfinite(z[[0, 2]]).all() and np.isfinite(z[1, 1]).all()
    assert np.linalg.norm(z[0] - want[0]) <= 1e-6 * np.linalg.norm(want[0])
