"""The FP32 row filter of n = 64 M and 512 M bins (k_filter_dif): every size it
has, FP32 and FP16 rows, the rows in pieces, rows written in place, slice counts
that leave pairs and halves of an entry empty, bins outside the padded row."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SIZES = [(256, 1), (320, 1), (256, 2), (512, 1), (512, 2), (1024, 1), (1280, 1), (1024, 2), (2048, 1), (2560, 1),
         (2048, 2), (4096, 1)]  # (rays, pad): n = rays (1 + pad) = 512 .. 8192


def _tomo(s, a, n, seed):
    rng = np.random.default_rng(seed)
    t = np.linspace(-1.0, 1.0, n)
    y = np.maximum(0.1, 1.0 - t * t) * (1.0 + np.arange(s) / s)[:, None, None]
    return (y + 0.05 * rng.standard_normal((s, a, n))).astype(np.float32)


def _params(n, a, s, pad, offset):
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, offset], np.float32)
    return paramf, np.array([n, a, s, n, pad, 0, 0, 5, 0, 0], np.int32)


@pytest.mark.parametrize("store", ["f32", "f16"])
@pytest.mark.parametrize("n,pad", SIZES)
def test_fbp_rows(gpu, n, pad, store):
    import torch
    from sscRaft import device as dv

    i = SIZES.index((n, pad))
    s, a, offset = (1, 2, 3, 5, 6, 9)[i % 6], 3 + i % 3, 1.5 * (i % 4) - 2.0
    y = _tomo(s, a, n, i)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    paramf, parami = _params(n, a, s, pad, offset)
    print(f"fbp n={n} pad={pad} s={s} a={a} offset={offset} {store}", flush=True)
    dy = torch.from_numpy(y).cuda()
    x = dv.fbp_device(dy, ang, paramf, parami, store=store)
    for k in sorted({0, s - 1}):
        want = oracle.fbp(np.ascontiguousarray(y[k:k + 1]), ang, *_params(n, a, 1, pad, offset))[0]
        e = float(np.linalg.norm(x[k].cpu().numpy() - want) / np.linalg.norm(want))
        print(f"slice {k}: rel-L2 {e:.2e}", flush=True)
        assert e < (1e-5 if store == "f32" else 5e-4)  # as for the transforms in natural order
    out = torch.empty_like(x)
    dv.fbp_device(dy, ang, paramf, parami, out=out, store=store, noalloc=True)
    assert torch.equal(out, x)


def test_fbp_rows_in_pieces(gpu):
    import torch
    from sscRaft import device as dv

    n, a, s = 512, 4, 64
    y = _tomo(s, a, n, 20)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    x = dv.fbp_device(torch.from_numpy(y).cuda(), ang, *_params(n, a, s, 2, 0.0)).cpu().numpy()
    for k in (0, 31, 63):
        want = oracle.fbp(np.ascontiguousarray(y[k:k + 1]), ang, *_params(n, a, 1, 2, 0.0))[0]
        assert np.linalg.norm(x[k] - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("n,pad,s", [(256, 1, 1), (320, 1, 3), (1024, 2, 6), (2048, 2, 5), (4096, 1, 2)])
def test_lowpass_in_place(gpu, n, pad, s):
    import torch
    from sscRaft import device as dv

    a = 3
    y = _tomo(s, a, n, 30)
    paramf, parami = _params(n, a, s, pad, 0.0)
    t = torch.from_numpy(y).cuda()
    print(f"lowpass n={n} pad={pad} s={s}", flush=True)
    r = dv.lowpass_device(t, paramf, parami)
    x = (t if r is None else r).cpu().numpy()
    want = oracle.lowpass(y, paramf, parami)
    e = float(np.linalg.norm(x - want) / np.linalg.norm(want))
    print(f"rel-L2 {e:.2e}", flush=True)
    assert e < 1e-5
