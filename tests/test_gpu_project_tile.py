"""The tile form of the projector (k_project_tile, k_project_sum), which serves
sparse angle sets: tiles cut by the image, rays other than pixels, stretched
pixels, angles along the axes and the diagonals, slopes near zero, odd slice
groups, sums taken in turns.  Reference: the direct form (RAFT_PROJ_LDS=0), whose
samples are the same, so that only the order of n positive FP32 terms differs:
|difference| <= 2 n 2^-24 of the sum."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _angles(a, first=0.0):
    ang = np.linspace(first, first + np.pi, a, endpoint=False)
    ang[: min(a, 6)] = [0.0, np.pi / 2, np.pi / 4, 3 * np.pi / 4, -1.0e-8, 4.0][: min(a, 6)]
    return ang.astype(np.float32)


@pytest.mark.parametrize("nx,ny,r,a,s,ax,ay", [
    (64, 64, 64, 9, 1, 1.0, 1.0),
    (65, 63, 65, 20, 5, 1.0, 1.0),
    (33, 200, 50, 12, 9, 1.0, 1.0),
    (129, 128, 300, 17, 4, 1.0, 1.0),
    (190, 130, 150, 30, 7, 1.0, 0.7),
    (100, 140, 100, 11, 3, 0.5, 1.0),
    (700, 500, 700, 90, 6, 1.0, 1.0),    # two slice groups a workgroup
    (2048, 2048, 2048, 200, 8, 1.0, 1.0),  # angles in turns
])
def test_radon_tiles_match_direct(gpu, monkeypatch, nx, ny, r, a, s, ax, ay):
    import torch
    from sscRaft import device as dv

    torch.manual_seed(nx)
    x = torch.rand((s, ny, nx), device="cuda") + 0.1
    ang = _angles(a)
    print(f"radon {nx}x{ny} r={r} a={a} s={s} ax={ax} ay={ay}", flush=True)
    got = dv.radon_device(x, ang, nrays=r, ax=ax, ay=ay).double()
    monkeypatch.setenv("RAFT_PROJ_LDS", "0")
    want = dv.radon_device(x, ang, nrays=r, ax=ax, ay=ay).double()
    assert float((got - want).abs().max()) > 0.0 or want.numel() < 20000  # another form than the direct one
    assert bool(((got - want).abs() <= 2 * ny * 2.0**-24 * want).all())


def test_radon_tiles_keep_non_finite_pixels_to_their_rays(gpu, monkeypatch):
    import torch
    from sscRaft import device as dv

    x = torch.rand((5, 150, 150), device="cuda") + 0.1
    x[1, 70, 63], x[4, 64, 64], x[2, 0, 149] = float("nan"), float("inf"), float("-inf")
    ang = _angles(15)
    got = dv.radon_device(x, ang)
    monkeypatch.setenv("RAFT_PROJ_LDS", "0")
    want = dv.radon_device(x, ang)
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), ok) and not bool(ok.all())
    assert torch.equal(got[~ok].nan_to_num(), want[~ok].nan_to_num())


@pytest.mark.parametrize("r,n,a,s,k", [(90, 90, 12, 5, 3), (134, 128, 25, 2, 3)])
def test_eem_tiles(gpu, r, n, a, s, k):
    """The ratio rows and the recorded KL; an image is the same with and without KL."""
    import torch
    from sscRaft import device as dv
    from sscRaft import phantom as ph

    ang = ph.uniform_angles(a)
    rng = np.random.default_rng(3)
    img = rng.random((s, n, n)) + 0.2
    y = np.stack([oracle.em_forward(img[q], ang, r) for q in range(s)]).astype(np.float32)
    print(f"eem r={r} n={n} a={a} s={s}", flush=True)
    dy = torch.from_numpy(y).cuda()
    x, kl, ex = dv.eem_device(dy, ang, k, obj=torch.ones((s, n, n), device="cuda"))
    plain = dv.eem_device(dy, ang, k, obj=torch.ones((s, n, n), device="cuda"), with_kl=False)[0]
    assert torch.equal(x, plain)
    xr, klr, exr = oracle.eem(y, ang, k, objsize=n)
    # FP32 sums and rows against FP64: as for the other projector forms
    x = x.cpu().numpy().astype(np.float64)
    ok = np.isfinite(xr)
    assert np.array_equal(np.isfinite(x), ok)
    assert np.linalg.norm((x - xr)[ok]) <= 1e-5 * np.linalg.norm(xr[ok])
    assert np.array_equal(ex, exr)
    assert np.abs(kl - klr).max() <= 1e-4 * np.abs(klr).max()


def test_tem_tiles(gpu):
    import torch
    from sscRaft import device as dv
    from sscRaft import phantom as ph

    n, a, s, k = 96, 14, 6, 2
    ang = ph.uniform_angles(a)
    rng = np.random.default_rng(4)
    flat = (rng.random((s, n)) + 100.0).astype(np.float32)
    count = (rng.random((s, a, n)) * 20.0 + 60.0).astype(np.float32)
    x = dv.tem_device(torch.from_numpy(count).cuda(), torch.from_numpy(flat).cuda(), ang, k).cpu().numpy()
    want = np.asarray(oracle.tem(count, flat, ang, k))
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(x), ok)
    assert np.linalg.norm((x - want)[ok]) <= 1e-5 * np.linalg.norm(want[ok])
