"""The FP64 transform form of the row filter (k_filter_conv), which serves padded
sizes with a prime factor above 5: every first radix, several transforms a row,
windows narrower than the row, FP16 rows, the matrix backprojector's rows."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _tomo(s, a, n, seed):
    rng = np.random.default_rng(seed)
    t = np.linspace(-1.0, 1.0, n)
    y = np.maximum(0.2, 1.0 - t * t) * (1.0 + np.arange(s) / s)[:, None, None]
    return (y + 0.05 * rng.standard_normal((s, a, n))).astype(np.float32)


def _params(n, a, s, pad, filt=7, offset=0.0):
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, offset], np.float32)
    return paramf, np.array([n, a, s, n, pad, 0, 0, filt, 0, 0], np.int32)


@pytest.mark.parametrize("n,a,s,pad,filt,offset,store", [
    (43, 5, 3, 2, 7, 0.0, "f32"),      # 129 bins, the shortest; 192 = 3 8 8
    (67, 6, 5, 1, 5, 1.5, "f32"),      # 256 = 4 8 8
    (101, 7, 1, 1, 7, -4.0, "f32"),    # 320 = 5 8 8; half a pair
    (127, 4, 4, 1, 7, 0.0, "f32"),     # 384 = 3 4 4 8
    (167, 4, 3, 1, 7, 0.0, "f16"),     # 512 = 8 8 8
    (337, 3, 18, 1, 7, 2.5, "f16"),    # 1024 = 4 4 8 8; the matrix backprojector
    (517, 4, 64, 1, 7, 0.0, "f32"),    # rows in pieces
    (1301, 3, 2, 1, 5, 7.5, "f32"),    # 4096
    (3407, 2, 2, 1, 7, 0.0, "f32"),    # two transforms a row
    (211, 5, 2, 0, 7, 0.0, "f32"),     # no padding; bins outside the row are zero
])
def test_fbp_rows_by_transforms(gpu, n, a, s, pad, filt, offset, store):
    import torch
    from sscRaft import device as dv

    y = _tomo(s, a, n, 5)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    paramf, parami = _params(n, a, s, pad, filt, offset)
    print(f"fbp n={n} a={a} s={s} pad={pad} filter={filt} offset={offset} {store}", flush=True)
    dy = torch.from_numpy(y).cuda()
    x = dv.fbp_device(dy, ang, paramf, parami, store=store)
    for k in sorted({0, s // 2, s - 1}):
        want = oracle.fbp(np.ascontiguousarray(y[k:k + 1]), ang, *_params(n, a, 1, pad, filt, offset))[0]
        e = float(np.linalg.norm(x[k].cpu().numpy().astype(np.float64) - want) / np.linalg.norm(want))
        print(f"slice {k}: rel-L2 {e:.2e}", flush=True)
        # FP64 rows rounded once (FP32 2^-24, FP16 2^-11), FP32 sums of a terms
        assert e < (1e-6 if store == "f32" else 5e-4)
    out = torch.empty_like(x)
    dv.fbp_device(dy, ang, paramf, parami, out=out, store=store, noalloc=True)
    assert torch.equal(out, x)


def test_non_finite_row_stays_in_its_slice(gpu):
    """A row pair shares one complex transform; a slice with a NaN or an infinity
    leaves the other slice of the pair as it is."""
    import torch
    from sscRaft import device as dv

    n, a, s = 101, 6, 4
    y = _tomo(s, a, n, 9)
    ang = np.linspace(0.0, np.pi, a, endpoint=False).astype(np.float32)
    paramf, parami = _params(n, a, s, 1)
    x = dv.fbp_device(torch.from_numpy(y).cuda(), ang, paramf, parami).cpu().numpy()
    y[0, 2, 50], y[3, 1, 0] = np.nan, np.inf
    z = dv.fbp_device(torch.from_numpy(y).cuda(), ang, paramf, parami).cpu().numpy()
    assert not np.isfinite(z[0]).all() and not np.isfinite(z[3]).all()
    for k in (1, 2):
        assert np.isfinite(z[k]).all()
        assert np.linalg.norm(z[k].astype(np.float64) - x[k]) <= 1e-6 * np.linalg.norm(x[k])
