"""The workloads this framework is timed on, called as a user's program calls them.

A case is a dict of plain values; `kind` names the entry point.  Sinograms are
the closed-form line integrals of seeded ellipses with counting noise,
images are the ellipses themselves.  `exact` evaluates the same
discretisation (integer bin and pixel indices from FP64 coordinates) with
plain torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "ssc-raft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

FILTERS = {"none": 0, "gaussian": 1, "lorentz": 2, "cosine": 3, "rectangle": 4, "hann": 5, "hamming": 6, "ramp": 7}


def listed():
    return [
        # one slice while a scan is being aligned: latency counts
        dict(name="fbp_preview", kind="fbp", S=1, A=512, N=512, pad=2, filter="ramp", offset=0.0, store="f32"),
        # a full detector's volume resident in device memory, FP32 rows
        dict(name="fbp_volume", kind="fbp", S=64, A=2048, N=2048, pad=2, filter="ramp", offset=0.0, store="f32"),
        # a binned detector's volume with the rows stored in FP16
        dict(name="fbp_half_rows", kind="fbp", S=32, A=1024, N=1024, pad=2, filter="hann", offset=0.0, store="f16"),
        # a cropped region of interest: odd row length, rotation axis off the centre, an uneven number of slices
        dict(name="fbp_ragged", kind="fbp", S=21, A=901, N=1301, pad=1, filter="hamming", offset=7.5, store="f32"),
        # host arrays through the reference's Python call, both copies included
        dict(name="fbp_host", kind="fbp_host", S=24, A=1024, N=1024, pad=2, filter="ramp", offset=0.0),
        # the row filter alone, in place, as a pre-processing step
        dict(name="lowpass", kind="lowpass", S=32, A=1024, N=2048, pad=2, filter="hann"),
        # FBP by the slice theorem
        dict(name="bst", kind="bst", S=16, A=1024, N=1024, pad=2, filter="ramp"),
        # projections of a full-size volume
        dict(name="radon_volume", kind="radon", S=32, A=2048, Nx=2048, Ny=2048, R=2048),
        # a few projections of a small rectangular volume
        dict(name="radon_sparse", kind="radon", S=6, A=90, Nx=700, Ny=500, R=700),
        # emission EM on a densely sampled scan
        dict(name="eem_dense", kind="eem", S=16, A=1024, N=1024, K=4),
        # emission EM on many slices of a sparsely sampled scan
        dict(name="eem_sparse", kind="eem", S=64, A=128, N=512, K=10),
        # the warm start network on a batch of reconstructions
        dict(name="unet", kind="unet", S=32, N=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fbp", "fbp", "fbp", "fbp_host", "lowpass", "bst", "radon", "radon", "eem", "eem", "unet"])
    S = _log(rng, 1, 64)
    if kind == "unet":
        return dict(kind=kind, S=max(1, S // 2), N=8 * rng.randint(16, 64))
    if kind == "bst":
        N = rng.choice([256, 320, 400, 512, 648, 720, 1000, 1024])
        return dict(kind=kind, S=max(1, S // 4), A=rng.randint(N // 2, N), N=N, pad=rng.choice([1, 2]),
                    filter=rng.choice(["ramp", "hann"]))
    N = _log(rng, 200, 2048)
    if rng.random() < 0.4:
        N = max(256, N // 128 * 128)
    A = rng.randint(N // 2, N)
    if kind == "eem":
        N = min(N, 1024)
        A = rng.randint(N // 8, N)
        return dict(kind=kind, S=min(S, 16 if N > 512 else 64), A=max(A, 32), N=N, K=rng.randint(1, 8))
    if kind == "radon":
        if rng.random() < 0.3:
            A = max(16, A // 8)
        square = rng.random() < 0.6
        Ny = N if square else max(128, N * rng.randint(60, 99) // 100)
        return dict(kind=kind, S=max(1, S // 2), A=A, Nx=N, Ny=Ny, R=N)
    pad = rng.choice([0, 1, 2, 2])
    filt = rng.choice(["ramp", "hann", "hamming", "cosine"])
    if kind == "lowpass":
        return dict(kind=kind, S=max(1, S // 2), A=min(A, 1024), N=N, pad=pad, filter=filt)
    offset = rng.choice([0.0, 0.0, round(rng.uniform(-9.0, 9.0), 2)])
    if kind == "fbp_host":
        N = min(N, 1024)
        return dict(kind=kind, S=min(S, 24), A=min(A, N), N=N, pad=pad, filter=filt, offset=offset)
    return dict(kind=kind, S=S, A=A, N=N, pad=pad, filter=filt, offset=offset, store=rng.choice(["f32", "f32", "f16"]))


# ---- inputs ---------------------------------------------------------------


def _angles(A):
    return np.linspace(0.0, np.pi, A, endpoint=False).astype(np.float32)


def _ellipses(S, seed, count=8):
    """[S, count, 6] centre, semi-axes, rotation and value of each slice's ellipses on [-1, 1]^2."""
    rng = np.random.Generator(np.random.PCG64(seed))
    r, t = 0.6 * np.sqrt(rng.random((S, count))), 2.0 * np.pi * rng.random((S, count))
    return np.stack([r * np.cos(t), r * np.sin(t), rng.uniform(0.05, 0.35, (S, count)),
                     rng.uniform(0.05, 0.35, (S, count)), rng.uniform(0.0, np.pi, (S, count)),
                     rng.uniform(0.1, 1.0, (S, count))], axis=-1)


def _sinogram(S, A, N, seed, i0=1.0e4):
    """Line integrals [S, A, N] (float32, on the GPU) with the noise of i0 counts per bin."""
    e = torch.tensor(_ellipses(S, seed), dtype=torch.float32, device="cuda")
    th = torch.tensor(_angles(A), device="cuda")[:, None]
    t = torch.linspace(-1.0, 1.0, N, device="cuda")[None, :]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    out = torch.empty((S, A, N), dtype=torch.float32, device="cuda")
    for s in range(S):
        p = torch.zeros((A, N), dtype=torch.float32, device="cuda")
        for cx, cy, a, b, phi, v in e[s].tolist():
            r2 = (a * torch.cos(th - phi)) ** 2 + (b * torch.sin(th - phi)) ** 2
            d = t - (cx * torch.cos(th) + cy * torch.sin(th))
            p += 2.0 * v * a * b * torch.sqrt(torch.clamp(r2 - d * d, min=0.0)) / r2
        counts = torch.poisson(i0 * torch.exp(-p), generator=gen)
        out[s] = -torch.log(torch.clamp(counts, min=1.0) / i0)
    return out


def _images(S, Ny, Nx, seed):
    e = torch.tensor(_ellipses(S, seed), dtype=torch.float32, device="cuda")
    x = torch.linspace(-1.0, 1.0, Nx, device="cuda")[None, :]
    y = torch.linspace(-1.0, 1.0, Ny, device="cuda")[:, None]
    out = torch.zeros((S, Ny, Nx), dtype=torch.float32, device="cuda")
    for s in range(S):
        for cx, cy, a, b, phi, v in e[s].tolist():
            c, sn = math.cos(phi), math.sin(phi)
            u, w = ((x - cx) * c + (y - cy) * sn) / a, ((y - cy) * c - (x - cx) * sn) / b
            out[s] += v * (u * u + w * w <= 1.0)
    return out


def _fbp_params(case):
    N = case["N"]
    paramf = np.array([0.0, 0.0, 1.0, 0.0, 2.0 / N, 2.0 / N, case.get("offset", 0.0)], np.float32)
    parami = np.array([N, case["A"], case["S"], N, case["pad"], 0, 0, FILTERS[case["filter"]], 0, 0], np.int32)
    return paramf, parami


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "radon":
        st["img"] = _images(case["S"], case["Ny"], case["Nx"], seed)
        st["angles"] = _angles(case["A"])
        st["out"] = torch.empty((case["S"], case["A"], case["R"]), dtype=torch.float32, device="cuda")
        return st
    if kind == "unet":
        from sscRaft.learned import default_weights_path
        from sscRaft.nn import UNet

        st["net"] = UNet.load(default_weights_path())
        st["img"] = _images(case["S"], case["N"], case["N"], seed)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        st["img"] += 0.05 * torch.randn(st["img"].shape, generator=gen, device="cuda")
        st["out"] = torch.empty_like(st["img"])
        return st
    st["tomo"] = _sinogram(case["S"], case["A"], case["N"], seed)
    st["angles"] = _angles(case["A"])
    if kind == "eem":
        st["tomo"].clamp_(min=0.0)
        return st
    st["paramf"], st["parami"] = _fbp_params(case)
    if kind == "fbp_host":
        st["tomo"] = st["tomo"].cpu().numpy()
        st["dic"] = {"gpu": [0], "angles[rad]": st["angles"], "filter": case["filter"], "padding": case["pad"],
                     "rotation axis offset": case["offset"], "detectorPixel[m]": 2.0 / case["N"]}
    elif kind != "lowpass":
        st["out"] = torch.empty((case["S"], case["N"], case["N"]), dtype=torch.float32, device="cuda")
    return st


def run(st):
    import sscRaft
    from sscRaft import device as dev

    case = st["case"]
    kind = case["kind"]
    if kind == "fbp":
        return dev.fbp_device(st["tomo"], st["angles"], st["paramf"], st["parami"], out=st["out"], store=case["store"])
    if kind == "fbp_host":
        return sscRaft.fbp(st["tomo"], dic=dict(st["dic"]))
    if kind == "lowpass":  # in place, so on a copy: the raw rows are kept
        return dev.lowpass_device(st["tomo"].clone(), st["paramf"], st["parami"])
    if kind == "bst":
        return dev.bst_device(st["tomo"], st["paramf"], st["parami"], out=st["out"])
    if kind == "radon":
        return dev.radon_device(st["img"], st["angles"], nrays=case["R"], out=st["out"])
    if kind == "eem":
        return dev.eem_device(st["tomo"], st["angles"], case["K"], with_kl=False)[0]
    return st["net"].forward(st["img"], out=st["out"], floor=1.0e-3)


def work(case):
    """Inputs read once and outputs written once; the additions of the sums
    (one per sample or pixel and slice), the butterflies of the row transforms."""
    kind, S, N = case["kind"], case["S"], case.get("N", 0)
    if kind == "radon":
        Nx, Ny, A, R = case["Nx"], case["Ny"], case["A"], case["R"]
        return dict(bytes=4.0 * S * (Nx * Ny + A * R), flops=1.0 * S * A * R * Ny)
    if kind == "unet":
        # multiply-adds of the 3x3 convolutions per full-resolution pixel: two
        # per level, decoder inputs concatenated
        macs = 9 * (32 * 1 + 32 * 32 + (32 * 64 + 64 * 64) / 4 + (64 * 128 + 128 * 128) / 16
                    + (128 * 256 + 256 * 256) / 64 + (384 * 128 + 128 * 128) / 16 + (192 * 64 + 64 * 64) / 4
                    + 96 * 32 + 32 * 32) + 32
        return dict(bytes=8.0 * S * N * N, flops=2.0 * macs * S * N * N)
    A = case["A"]
    if kind == "eem":
        return dict(bytes=4.0 * S * (A * N + N * N), flops=2.0 * case["K"] * S * A * N * N)
    n = N * (1 + case["pad"])
    fft = 5.0 * S * A * n * math.log2(n)  # forward and inverse transform of real rows
    if kind == "lowpass":
        return dict(bytes=8.0 * S * A * N, flops=fft)
    if kind == "bst":
        return dict(bytes=4.0 * S * (A * N + N * N), flops=2.0 * fft + 5.0 * S * n * n * math.log2(n))
    return dict(bytes=4.0 * S * (A * N + N * N), flops=fft + 1.0 * S * A * N * N)


# ---- the same values in 64 bits -------------------------------------------


def _fma(a, b, c):
    """a * b + c rounded once (a: integers and halves of at most 26 bits), from error-free float64 steps."""
    t = b * 134217729.0
    hi = t - (t - b)
    lo = b - hi
    p = a * b
    e = (a * hi - p) + a * lo
    s = p + c
    bb = s - p
    return s + (((p - (s - bb)) + (c - bb)) + e)


def _f64(x):
    return torch.as_tensor(x, dtype=torch.float64, device="cuda")


def _filter_amp(name, w):
    """The row filters at tent weight w (no regularisation, no phase retrieval)."""
    if name == "cosine":
        return w * torch.cos(math.pi * 0.5 * w)
    if name == "hann":
        return w * (0.5 + 0.5 * torch.cos(2.0 * math.pi * w))
    if name == "hamming":
        return w * (float(np.float32(0.54)) + float(np.float32(0.46)) * torch.cos(2.0 * math.pi * w))
    return w


def _pad_rows(rows, pad):
    N = rows.shape[-1]
    i = torch.clamp(torch.arange(N * (1 + pad), device="cuda") - (pad * N) // 2, 0, N - 1)
    return rows.to(torch.float64)[..., i]


def _filtered(rows, case, offset):
    """Padded rows of one slice [A, npad], filtered: edge replicate, tent weights, 1 / (npad pixel)."""
    n = case["N"] * (1 + case["pad"])
    M = n // 2 + 1
    k = torch.arange(M, dtype=torch.float64, device="cuda")
    amp = _filter_amp(case["filter"], 0.5 * torch.minimum(k, M - k) / M)
    ph = -2.0 * math.pi * offset * k / (2 * M - 2)
    U = torch.fft.rfft(_pad_rows(rows, case["pad"]), dim=-1)
    return torch.fft.irfft(U * torch.polar(amp, ph), n=n, dim=-1) / float(np.float32(2.0 / case["N"]))


def _steps(ang):
    a = ang.astype(np.float64)
    d = np.empty_like(a)
    d[:-1] = a[1:] - a[:-1]
    d[-1] = a[-1] - a[-2]
    return d


def _backproject(q, ang, n, xc, c0, cA, cB):
    """sum over angles of q[s, a, (int)u] * step, u = fma(X, cA, fma(Y, cB, c0)), zero outside the rows."""
    S, A, nb = q.shape
    d = _steps(ang)
    X = (_f64(np.arange(n)) - xc)
    out = torch.zeros((S, n * n), dtype=torch.float64, device="cuda")
    for a in range(A):
        u = _fma(X[None, :], _f64(cA[a]), _fma(X, _f64(cB[a]), _f64(c0))[:, None])
        T = torch.trunc(u).to(torch.int64).reshape(-1)
        w = q[:, a, :] * d[a]
        ok = (T >= 0) & (T < nb)
        v = w[:, torch.clamp(T, 0, nb - 1)]
        out += v if bool(ok.all()) else v * ok
    return out.reshape(S, n, n)


def _project(img, ang, R, ci, nk, ck, ucx, ucy, ry, rx):
    """Sums over samples k of img[s, Y, X] along each ray, [S, A, R]."""
    S, Ny, Nx = img.shape
    flat = img.reshape(S, -1)
    ir, kr = _f64(np.arange(R)) - ci, _f64(np.arange(nk)) - ck
    out = torch.empty((S, len(ang), R), dtype=torch.float64, device="cuda")
    for a, th in enumerate(ang.astype(np.float64)):
        c, s = math.cos(th), math.sin(th)
        X = torch.trunc(_fma(kr[None, :], _f64(-s * ry), _fma(ir, _f64(c), _f64(ucx))[:, None])).to(torch.int64)
        Y = torch.trunc(_fma(kr[None, :], _f64(c), _fma(ir, _f64(s * rx), _f64(ucy))[:, None])).to(torch.int64)
        ok = (X >= 0) & (X < Nx) & (Y >= 0) & (Y < Ny)
        idx = torch.where(ok, Y * Nx + X, 0)
        out[:, a] = torch.einsum("srk,rk->sr", flat[:, idx], ok.to(torch.float64)) if S * R * nk < 5e7 else torch.stack(
            [(flat[t][idx] * ok).sum(-1) for t in range(S)])
    return out


def _em_project(x, ang, R):
    c = (R - 1) / 2.0
    return _project(x, ang, R, c, R, c, c, c, 1.0, 1.0) * float(np.float32(2.0 / (R - 1)))


def _em_backproject(q, ang, n, R):
    rr = (R - 1) / (n - 1)
    th = ang.astype(np.float64)
    return _backproject(q, ang, n, (n - 1) / 2.0, (R - 1) / 2.0, np.cos(th) * rr, np.sin(th) * rr)


def _exact_fbp(case, tomo, ang, offset):
    N, n = case["N"], case["N"] * (1 + case["pad"])
    q = torch.stack([_filtered(tomo[s], case, offset) for s in range(case["S"])])
    th = ang.astype(np.float64)
    c0 = n / 2.0
    scale = math.pi / th[-1] if ang[-1] > np.float32(math.pi) else 1.0
    return _backproject(q, ang, N, c0 - (case["pad"] * N) // 2, c0, np.cos(th), -np.sin(th)) * scale


def _exact_bst(case, tomo):
    N, n = case["N"], case["N"] * (1 + case["pad"])
    A, A2, L, h = case["A"], 2 * case["A"], (case["pad"] * N) // 2, n // 2
    k = torch.arange(n, dtype=torch.float64, device="cuda")
    amp = _filter_amp(case["filter"], torch.minimum(k, n - k) / n)
    wts = torch.full((h,), 4.0, dtype=torch.float64, device="cuda")
    wts[0] = 2.0
    sigma = 2.0 / (n * torch.clamp(torch.minimum(k, n - k), min=0.5))
    pos = k - n // 2
    rho = torch.hypot(pos[None, :], pos[:, None])
    angle = A2 * (0.5 * torch.atan2(pos[:, None], pos[None, :]) / math.pi + 0.5)
    ir, ia = torch.floor(rho).to(torch.int64), torch.floor(angle).to(torch.int64)
    pf, tf = rho - ir, ia - angle
    ok = ir < h - 1
    ir = torch.where(ok, ir, 0)
    ia = ia % A2
    ua = (ia + 1) % A2
    par = torch.arange(n, device="cuda") % 2
    sign = torch.where(par[None, :] == par[:, None], 1.0, -1.0) * ok
    out = []
    for s in range(case["S"]):
        u = torch.fft.ifft(torch.fft.fft(_pad_rows(tomo[s], case["pad"]), dim=-1) * amp, dim=-1).real * n
        P = torch.zeros((A2, n), dtype=torch.float64, device="cuda")
        P[:A, :h] = torch.flip(u[:, :h], [1]) * wts
        P[A:, :h] = u[:, h:h + h] * wts
        Q = torch.fft.fft(P, dim=-1) * sigma
        val = ((Q[ia, ir] * (1 - pf) + Q[ia, ir + 1] * pf) * tf + (Q[ua, ir] * (1 - pf) + Q[ua, ir + 1] * pf) * (1 - tf)) * sign
        C = torch.roll(val, (n // 2, n // 2), (0, 1))
        im = torch.fft.ifft2(C).real * (float(n) * n) / (4.0 * n * float(np.float32(2.0 / N)))
        out.append(im[L:L + N, L:L + N].clone())
    return torch.stack(out)


def _exact_unet(img, floor):
    """The network in float64 (weights as stored, input rounded to bf16), one image at a time."""
    from sscRaft.learned import default_weights_path

    with np.load(default_weights_path(), allow_pickle=False) as z:
        conv = torch.from_numpy((z["conv_bf16"].astype(np.uint32) << 16).view(np.float32).astype(np.float64)).cuda()
        rest = torch.from_numpy(z["other_f32"].astype(np.float64)).cuda()
    layers = [(32, 32), (32, 32), (64, 32), (64, 64), (128, 64), (128, 128), (256, 128), (256, 256), (128, 384),
              (128, 128), (64, 192), (64, 64), (32, 96), (32, 32)]
    par, w0, b0 = [], 0, 0
    for co, ci in layers:
        par.append((conv[w0:w0 + co * 9 * ci].reshape(co, 9, ci), rest[b0:b0 + co]))
        w0, b0 = w0 + co * 9 * ci, b0 + co
    head_w, head_b = rest[b0:b0 + 32], rest[b0 + 32]

    def layer(x, i):
        w, b = par[i]
        H, W = x.shape[1:]
        xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
        y = b[:, None].expand(-1, H * W)
        for t in range(9):
            dy, dx = t // 3, t % 3
            y = y + w[:, t, :].contiguous() @ xp[:, dy:dy + H, dx:dx + W].reshape(x.shape[0], -1)
        return torch.clamp(y, min=0.0).reshape(-1, H, W)

    def pool(x):
        return (x[:, 0::2, 0::2] + x[:, 0::2, 1::2] + x[:, 1::2, 0::2] + x[:, 1::2, 1::2]) / 4.0

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    out = torch.empty(img.shape, dtype=torch.float64, device="cuda")
    for s in range(img.shape[0]):
        x0 = torch.zeros((32,) + tuple(img.shape[1:]), dtype=torch.float64, device="cuda")
        x0[0] = img[s].to(torch.bfloat16).to(torch.float64)
        e1 = layer(layer(x0, 0), 1)
        e2 = layer(layer(pool(e1), 2), 3)
        e3 = layer(layer(pool(e2), 4), 5)
        e4 = layer(layer(pool(e3), 6), 7)
        d3 = layer(layer(torch.cat([e3, up(e4)]), 8), 9)
        d2 = layer(layer(torch.cat([e2, up(d3)]), 10), 11)
        d1 = layer(layer(torch.cat([e1, up(d2)]), 12), 13)
        out[s] = img[s].to(torch.float64) + (head_w[:, None, None] * d1).sum(0) + head_b
    return torch.clamp(out, min=floor)


def exact(case, seed):
    kind = case["kind"]
    ang = _angles(case["A"]) if "A" in case else None
    if kind == "unet":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        img = _images(case["S"], case["N"], case["N"], seed)
        img += 0.05 * torch.randn(img.shape, generator=gen, device="cuda")
        return _exact_unet(img, float(np.float32(1.0e-3)))
    if kind == "radon":
        Nx, Ny = case["Nx"], case["Ny"]
        img = _images(case["S"], Ny, Nx, seed).to(torch.float64)
        out = _project(img, ang, case["R"], (Nx - 1) / 2.0, Ny, (Ny - 1) / 2.0, (Nx - 1) / 2.0, (Ny - 1) / 2.0,
                       (Nx - 1) / (Ny - 1), (Ny - 1) / (Nx - 1))
        return out * (2.0 / (Ny - 1))
    tomo = _sinogram(case["S"], case["A"], case["N"], seed)
    if kind == "eem":
        N = case["N"]
        y = tomo.clamp_(min=0.0).to(torch.float64)
        e = float(np.float32(1.0e-4))
        back = _em_backproject(torch.ones((1, case["A"], N), dtype=torch.float64, device="cuda"), ang, N, N)
        x = torch.ones((case["S"], N, N), dtype=torch.float64, device="cuda")
        for _ in range(case["K"]):
            v = _em_project(x, ang, N)
            r = torch.clamp(y * torch.sign(v) / torch.sqrt(e * e + v * v), min=0.0)
            x = x * _em_backproject(r, ang, N, N) / back
        return x
    if kind == "bst":
        return _exact_bst(case, tomo)
    if kind == "lowpass":
        L = (case["pad"] * case["N"]) // 2
        return torch.stack([_filtered(tomo[s], case, 0.0)[:, L:L + case["N"]] for s in range(case["S"])])
    out = _exact_fbp(case, tomo, ang, case["offset"])
    return out.cpu().numpy() if kind == "fbp_host" else out
