"""raft_fbp_device_noalloc gives raft_fbp_device's output bit for bit also where
few slice groups fit its scratch: calls that run on the matrix cores, and
geometries so large that one group of rows nearly fills its limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMIT = 256 << 20  # RAFT_NOALLOC_SCRATCH_BYTES


def _params(n, a, s, pad):
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, 0.0], np.float32)
    return paramf, np.array([n, a, s, n, pad, 0, 0, 7, 0, 0], np.int32)


def _largest_angles(n, pad):
    """Angles at which a slice group's rows leave room for the general tables in the
    limit (filter, and the direct sum's kernel where there is no FFT), but not for
    those of the faster filter forms."""
    from sscRaft import device as dv

    a = 8192
    for _ in range(2): # the width hardly depends on so many angles
        ang = np.linspace(0.0, np.pi, a, endpoint=False).astype(np.float32)
        _, width, fft = dv.fbp_plan_info(ang, *_params(n, a, 1, pad))
        a = (LIMIT - (8 if fft else 16) * n * (1 + pad) - 4096) // (16 * width + 20)
    return a


@pytest.mark.parametrize("n,a,s,pad,store,form", [
    (2048, 2048, 64, 2, "f32", 2),  # 91 MiB a group
    (2300, 4500, 16, 1, "f32", 2),  # 224 MiB
    (2048, 5500, 35, 1, "f16", 2),
    (1301, 0, 3, 1, "f32", 0),      # FP64 transforms
    (1024, 0, 2, 2, "f32", 0),      # permuted FP32 transforms
])
def test_same_bits(gpu, n, a, s, pad, store, form):
    import torch
    from sscRaft import device as dv

    a = a or _largest_angles(n, pad)
    ang = np.linspace(0.0, np.pi, a, endpoint=False).astype(np.float32)
    paramf, parami = _params(n, a, s, pad)
    assert dv.fbp_form_info(ang, paramf, parami, store=store)[0] == form
    print(f"noalloc n={n} a={a} s={s} pad={pad} {store}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    y = torch.rand((s, a, n), device="cuda", generator=gen)
    out = torch.full((s, n, n), float("nan"), device="cuda")
    dv.fbp_device(y, ang, paramf, parami, out=out, store=store, noalloc=True)
    assert torch.equal(out, dv.fbp_device(y, ang, paramf, parami, store=store))
