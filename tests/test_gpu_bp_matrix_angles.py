"""The matrix-core backprojector over as many angles as its calls have: several
turns of its ring of LDS buffers (3 or 4 rounds of 4 angles), last rounds of 1 to
4 angles, every pack width, rows in pieces from both FP32 filter forms, each call
asserted to take it.  References: the FP64 oracle, the same sums staged through
registers (raft_fbp_device_noalloc), the gather kernels."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

MATRIX = 2


def _tomo(s, a, n, seed):
    rng = np.random.default_rng(seed)
    t = np.linspace(-1.0, 1.0, n)
    y = np.maximum(0.0, 1.0 - t * t) * (1.0 + np.arange(s) / s)[:, None, None]
    return (y + 0.05 * rng.standard_normal((s, a, n))).astype(np.float32)


def _angles(a):
    return (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)


def _params(n, a, s, filt=7, pad=2, offset=0.0):
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, offset], np.float32)
    return paramf, np.array([n, a, s, n, pad, 0, 0, filt, 0, 0], np.int32)


@pytest.mark.parametrize("n,a,s,pad,store,offset", [
    (200, 37, 150, 2, "f32", 0.0),     # wide packs, the last partly filled; a last round of one angle
    (200, 1002, 150, 2, "f32", 2.5),   # many angles; two left over
    (512, 257, 64, 2, "f32", 0.0),     # rows in pieces from the permuted transforms
    (517, 259, 64, 1, "f32", -3.0),    # and from the FP64 ones; three left over
    (512, 150, 203, 1, "f32", 0.0),    # the narrow pack (three buffers), 11 of 16 slices
    (2048, 400, 16, 0, "f32", 0.0),    # narrow packs alone; no padding: windows start before the row
    (24, 37, 16, 1, "f16", 0.0),       # one tile row, half a narrow pack
    (130, 1001, 20, 1, "f16", 1.5),
    (97, 70, 45, 2, "f16", 0.0),       # a wide pack partly filled
    (512, 81, 85, 2, "f16", 0.0),      # wide and narrow
    (337, 60, 18, 1, "f16", 0.0),      # rows from the FP64 transforms
])
def test_fbp_many_angles(gpu, n, a, s, pad, store, offset):
    import torch
    from sscRaft import device as dv

    y, ang = _tomo(s, a, n, 7), _angles(a)
    paramf, parami = _params(n, a, s, pad=pad, offset=offset)
    assert dv.fbp_form_info(ang, paramf, parami, store=store)[0] == MATRIX
    dy = torch.from_numpy(y).cuda()
    print(f"fbp n={n} a={a} s={s} pad={pad} {store} offset={offset}", flush=True)
    out = torch.full((s, n, n), float("nan"), device="cuda")
    dv.fbp_device(dy, ang, paramf, parami, out=out, store=store)
    sel = [0, s - 1] if n > 1000 else [0, s // 2, s - 1]
    want = oracle.fbp(np.ascontiguousarray(y[sel]), ang, *_params(n, a, len(sel), pad=pad, offset=offset))
    for i, k in enumerate(sel):
        x = out[k].cpu().numpy().astype(np.float64)
        e = float(np.linalg.norm(x - want[i]) / np.linalg.norm(want[i]))
        print(f"slice {k}: rel-L2 {e:.2e}", flush=True)
        # row values rounded once (FP32 2^-24, FP16 2^-11), FP32 filter arithmetic: as for the gather kernels
        assert e < (1e-5 if store == "f32" else 5e-4)
    again = torch.full((s, n, n), float("nan"), device="cuda")
    dv.fbp_device(dy, ang, paramf, parami, out=again, store=store, noalloc=True)
    assert torch.equal(out, again)


@pytest.mark.parametrize("store", ["f32", "f16"])
def test_non_finite_samples_stay_where_they_are_read(gpu, store):
    """Unfiltered rows with NaN and infinities: the same pixels as the gather
    kernels (a call of one slice) are non-finite, the others untouched by them."""
    import torch
    from sscRaft import device as dv

    n, a, s = 200, 50, 150
    y, ang = _tomo(s, a, n, 11), _angles(a)
    y[3, 2, 50], y[40, 0, 101], y[149, 45, 7], y[149, 49, 150] = np.nan, np.inf, -np.inf, np.inf
    paramf, parami = _params(n, a, s, filt=0)
    assert dv.fbp_form_info(ang, paramf, parami, store=store)[0] == MATRIX
    dy = torch.from_numpy(y).cuda()
    x = dv.fbp_device(dy, ang, paramf, parami, store=store)
    for k in (3, 40, 149, 4):
        few = dv.fbp_device(dy[k:k + 1].contiguous(), ang, *_params(n, a, 1, filt=0), store=store)[0]
        bad = ~torch.isfinite(few)
        assert bool(bad.any()) == (k != 4)
        assert torch.equal(x[k][bad].isnan(), few[bad].isnan())
        assert torch.equal(x[k][bad].nan_to_num(), few[bad].nan_to_num())
        assert torch.isfinite(x[k][~bad]).all()
        # sums of a terms in another order
        assert float((x[k] - few)[~bad].abs().max()) <= 2 * a * 2.0**-24 * a * float(few[~bad].abs().max() + 2)


@pytest.mark.parametrize("store,exp", [("f32", -118), ("f16", -19)])
def test_small_values_keep_their_bits(gpu, store, exp):
    """Rows scaled by a power of two down to where the pieces of an FP32 value, or
    FP16 values, are subnormal: nothing is flushed on the way."""
    import torch
    from sscRaft import device as dv

    n, a, s = 200, 64, 150
    rng = np.random.default_rng(5)
    # whole numbers below 2^10, weights of 2^-5: every sum is exact, and the smallest FP16
    # value is 2^-24
    ang = (np.arange(a) * 2.0**-5).astype(np.float32)
    y = rng.integers(0, 1024, (s, a, n)).astype(np.float32)
    paramf, parami = _params(n, a, s, filt=0)
    assert dv.fbp_form_info(ang, paramf, parami, store=store)[0] == MATRIX
    want = dv.fbp_device(torch.from_numpy(y).cuda(), ang, paramf, parami, store="f32")
    x = dv.fbp_device(torch.from_numpy(y * np.float32(2.0**exp)).cuda(), ang, paramf, parami, store=store)
    # scaled back in two steps: 2^-exp alone may overflow
    assert torch.equal(x * 2.0**(-exp // 2) * 2.0**(-exp - -exp // 2), want)
