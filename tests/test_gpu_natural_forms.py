"""Kernel forms that serve the sizes beside those of the newer ones, against each
other: the FP32 filter's transforms in natural order (padded sizes k_filter_dif does
not have), the variants of the gather backprojector (calls that neither split the
angles nor run on the matrix cores), the direct projector (images below 32 x 32)."""
import json

import numpy as np
import pytest

import oracle
from sscRaft import phantom as ph

pytestmark = pytest.mark.gpu

GATHER = 0
PAIR, SPF = 1024, 2048  # BP_PAIR, BP_SPF


def _sino(s, a, n, seed):
    rng = np.random.default_rng(seed)
    t = np.linspace(-1.0, 1.0, n)
    y = np.maximum(0.1, 1.0 - t * t) * (1.0 + np.arange(s) / s)[:, None, None]
    return (y + 0.05 * rng.standard_normal((s, a, n))).astype(np.float32)


def _params(n, a, s, filt=7, pad=2):
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, 0.0], np.float32)
    return paramf, np.array([n, a, s, n, pad, 0, 0, filt, 0, 0], np.int32)


@pytest.mark.parametrize("switch", [("RAFT_FFT_FORM", "regs"), ("RAFT_FILTER_PAIRS", "1")])
@pytest.mark.parametrize("n,a,s,filt", [(768, 20, 5, 7), (900, 12, 4, 5), (1600, 10, 3, 7), (1800, 8, 6, 5)])
def test_filter_forms_are_bit_identical(gpu, monkeypatch, switch, n, a, s, filt):
    """Padded lengths 2304, 2700 (384 threads), 4800 and 5400 (768): the form with
    the first pair's window in LDS against the window in registers and against
    one pair a workgroup; FBP, and the low-pass written in place."""
    import torch
    from sscRaft import device as dv

    y = _sino(s, a, n, n)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    paramf, parami = _params(n, a, s, filt)
    dy = torch.from_numpy(y).cuda()
    print(f"n={n} a={a} s={s} filter={filt} {switch}", flush=True)

    def both():
        t = dy.clone()
        r = dv.lowpass_device(t, paramf, parami)
        return dv.fbp_device(dy, ang, paramf, parami), (t if r is None else r)

    img, rows = both()
    monkeypatch.setenv(*switch)
    img1, rows1 = both()
    assert torch.equal(img, img1) and torch.equal(rows, rows1)
    want = oracle.lowpass(y, paramf, parami)
    assert np.linalg.norm(rows.cpu().numpy() - want) <= 1e-5 * np.linalg.norm(want)


def _forced(tmp_path, monkeypatch, key, choice):
    from sscRaft import device as dv

    f = tmp_path / "tune.json"
    f.write_text(json.dumps({key: {"choice": choice, "ms": []}}))
    monkeypatch.setenv("RAFT_AUTOTUNE_CACHE", str(f))
    dv.autotune_clear()


@pytest.mark.parametrize("n,a,s", [(600, 180, 10), (300, 63, 7)])
def test_backprojector_variants_are_bit_identical(gpu, tmp_path, monkeypatch, n, a, s):
    """Every FP32 variant forced through the cache file, in calls that run it
    (more workgroups than are split, or too few angles for that), the last pair
    of slice groups without its second group or with a partial one; also
    without device allocation."""
    import torch
    from sscRaft import device as dv

    y = _sino(s, a, n, 5)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    paramf, parami = _params(n, a, s)
    assert dv.fbp_form_info(ang, paramf, parami)[0] == GATHER
    dy = torch.from_numpy(y).cuda()
    monkeypatch.setenv("RAFT_AUTOTUNE_CACHE", str(tmp_path / "fresh.json"))
    dv.autotune_clear()
    ref = dv.fbp_device(dy, ang, paramf, parami)
    keys = [k for k in dv.autotune_choices() if k.startswith(f"bp/n={n}/A={a}/")]
    assert len(keys) == 1
    for variant in (16, 32, 48, PAIR | 16, PAIR | 32, SPF | 16, SPF | 32):
        _forced(tmp_path, monkeypatch, keys[0], variant)
        assert torch.equal(dv.fbp_device(dy, ang, paramf, parami), ref), variant
        out = torch.full_like(ref, float("nan"))
        dv.fbp_device(dy, ang, paramf, parami, out=out, noalloc=True)
        assert torch.equal(out, ref), variant
    want = oracle.fbp(y, ang, paramf, parami)
    assert np.linalg.norm(ref.cpu().numpy() - want) <= 1e-5 * np.linalg.norm(want)


def test_eem_schedule_in_the_direct_projector(gpu):
    """As per-slice runs, bit for bit, in an image too small for the tile form."""
    import torch
    from sscRaft import device as dv

    counts, n, a = [6, 6, 5, 3, 3, 1, 0], 28, 9
    ang = ph.uniform_angles(a)
    y = torch.from_numpy(np.maximum(ph.poisson_log(oracle.radon(ph.phantoms(n, len(counts), config=8, first=3), ang),
                                                   1e4, seed=3), 0).astype(np.float32)).cuda()
    x0 = torch.from_numpy(np.random.default_rng(3).uniform(0.5, 1.5, (len(counts), n, n)).astype(np.float32)).cuda()
    xs = dv.eem_device_sched(y, ang, counts, obj=x0.clone())
    for s, k in enumerate(counts):
        one = x0[s] if k == 0 else dv.eem_device(y[s:s + 1].contiguous(), ang, k, obj=x0[s:s + 1].clone(), with_kl=False)[0][0]
        assert torch.equal(xs[s], one), (s, k)
