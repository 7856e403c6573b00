"""The FP64 row filter around its shortest rows: padded sizes on both sides of the
lines between the direct sum and the transforms, FBP and low-pass, and sizes where
one longer transform replaces two of half its length."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad", [(43, 2), (13, 9), (47, 2), (59, 1), (61, 1), (67, 1), (131, 0), (51, 2), (57, 2),
                                   (69, 1), (77, 1), (151, 0), (203, 0)])
def test_short_rows(gpu, n, pad):
    import torch
    from sscRaft import device as dv

    a, s = 7, 19
    rng = np.random.default_rng(n)
    t = np.linspace(-1.0, 1.0, n)
    y = (np.maximum(0.2, 1.0 - t * t) * (1.0 + np.arange(s) / s)[:, None, None]
         + 0.05 * rng.standard_normal((s, a, n))).astype(np.float32)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, 0.0], np.float32)
    parami = np.array([n, a, s, n, pad, 0, 0, 7, 0, 0], np.int32)
    dy = torch.from_numpy(y).cuda()
    print(f"n={n} pad={pad}", flush=True)
    x = dv.fbp_device(dy, ang, paramf, parami)
    want = oracle.fbp(y, ang, paramf, parami)
    # FP64 rows rounded once, FP32 sums of a terms
    assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-6 * np.linalg.norm(want)
    out = torch.empty_like(x)
    dv.fbp_device(dy, ang, paramf, parami, out=out, noalloc=True)
    assert torch.equal(out, x)
    r = dv.lowpass_device(dy, paramf, parami)
    rows = (dy if r is None else r).cpu().numpy()
    want = oracle.lowpass(y, paramf, parami)
    assert np.linalg.norm(rows - want) <= 1e-6 * np.linalg.norm(want)
