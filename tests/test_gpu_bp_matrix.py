"""The matrix-core backprojector (csrc/backproject_mx.hip): calls of many slices.

Every case runs it at an edge of its range: full and partly filled packs, the
narrow pack, tiles cut by the image, angle counts around its rounds of 4,
non-finite samples.  References: the FP64 oracle,
and calls of few slices, which run the gather kernels.
"""
import re
from pathlib import Path

import numpy as np
import pytest

import oracle

SRC = Path(__file__).resolve().parent.parent / "ssc-raft_amd" / "csrc" / "backproject_mx.hip"


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


def _rel(x, want):
    return float(np.linalg.norm(x.astype(np.float64) - want) / np.linalg.norm(want))


def test_windows_hold_every_bin():
    """The bins a patch's pixels read lie in its 8-bin window, and the windows of
    a tile in its staged bins, for any angle and centre (the kernel's integer
    arithmetic on the CPU, constants from its source)."""
    src = SRC.read_text()
    def c(name):
        return float(re.search(rf"constexpr (?:int|double) {name} = ([0-9.]+);", src).group(1))
    reach, spread, slot = c("BM_REACH"), c("BM_SPREAD"), int(c("BM_SLOT"))
    rng = np.random.default_rng(0)
    px, py = np.meshgrid(np.arange(24), np.arange(40), indexing="ij")
    trunc = lambda v: np.trunc(v).astype(np.int64)
    for case in range(400):
        th = rng.uniform(-7.0, 7.0) if case > 16 else case * np.pi / 8
        n = int(rng.integers(1, 3000))
        xc, c0 = 0.5 * (n - 1), rng.uniform(-50.0, n + 50.0)
        i0, j0 = 24 * int(rng.integers(0, n // 24 + 1)), 40 * int(rng.integers(0, n // 40 + 1))
        ca, cb = np.cos(th), np.sin(th)
        T = trunc((i0 + px - xc) * ca + ((j0 + py - xc) * cb + c0))
        base = trunc((i0 + px // 6 * 6 + 2.5 - xc) * ca + ((j0 + py // 5 * 5 + 2 - xc) * cb + (c0 - reach)))
        assert ((T - base >= 0) & (T - base <= 7)).all()
        w = trunc((i0 + 11.5 - xc) * ca + ((j0 + 19.5 - xc) * cb + (c0 - (spread + reach + 0.01))))
        assert (base - (w - 1) >= 0).all() and (base - (w - 1) + 8 <= slot).all() and (base - w >= 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n,a,s,store,offset", [
    (512, 7, 64, "f32", 0.0),     # two full packs
    (513, 5, 90, "f32", 3.5),     # a partly filled third; tiles cut on both sides
    (512, 9, 203, "f32", 0.0),    # the narrow pack, 11 of 16 slices
    (200, 4, 150, "f32", -7.0),   # the rest on idle CUs; one round per tile pass
    (1031, 2, 31, "f32", 0.0),    # half a round
    (24, 3, 16, "f16", 0.0),      # one tile row, half a narrow pack
    (97, 6, 45, "f16", 1.5),      # a wide pack partly filled
    (512, 8, 85, "f16", 0.0),     # wide and narrow
])
def test_fbp_many_slices(gpu, n, a, s, store, offset):
    import torch
    from sscRaft import device as dv

    y, ang = _tomo(s, a, n, 7), _angles(a)
    paramf, parami = _params(n, a, s, offset=offset)
    dy = torch.from_numpy(y).cuda()
    print(f"fbp n={n} a={a} s={s} {store} offset={offset}", flush=True)
    out = torch.full((s, n, n), float("nan"), device="cuda")
    dv.fbp_device(dy, ang, paramf, parami, out=out, store=store)
    x = out.cpu().numpy()
    assert np.isfinite(x).all()
    sel = [0, s // 2, s - 1]
    want = oracle.fbp(np.ascontiguousarray(y[sel]), ang, *_params(n, a, 3, offset=offset))
    for i, k in enumerate(sel):
        e = _rel(x[k], want[i])
        print(f"slice {k}: rel-L2 {e:.2e}", flush=True)
        # row values rounded once (FP32 2^-24, FP16 2^-11), FP32 filter arithmetic: as for the gather kernels
        assert e < (1e-5 if store == "f32" else 5e-4)
    # the same bits without device allocation (checked staging)
    again = torch.full((s, n, n), float("nan"), device="cuda")
    dv.fbp_device(dy, ang, paramf, parami, out=again, store=store, noalloc=True)
    assert torch.equal(out, again)


@pytest.mark.gpu
@pytest.mark.parametrize("store", ["f32", "f16"])
def test_fbp_non_finite_samples_stay_where_they_are_read(gpu, store):
    """Unfiltered rows with NaN and infinities: the same pixels as the gather
    kernels are non-finite, the others untouched by them."""
    import torch
    from sscRaft import device as dv

    n, a, s = 200, 6, 150
    y, ang = _tomo(s, a, n, 11), _angles(a)
    y[3, 2, 50], y[40, 0, 101], y[149, 5, 7], y[149, 1, 150] = np.nan, np.inf, -np.inf, np.inf
    paramf, parami = _params(n, a, s, filt=0)
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
