"""The FP64 transform form of the row filter takes two slices in one complex
transform; slices of very different magnitude stay apart, and a slice of zeros
stays zero, as in the direct sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad,store", [(67, 1, "f32"), (101, 1, "f32"), (1301, 1, "f32"), (3407, 1, "f32"), (167, 1, "f16")])
def test_slices_of_a_pair_stay_apart(gpu, n, pad, store):
    import torch
    from sscRaft import device as dv

    a, s = 5, 8
    rng = np.random.default_rng(n)
    y = (1.0 + 0.5 * rng.random((s, a, n))).astype(np.float32)
    big, small = (1.0e13, 1.0e-13) if store == "f32" else (1.0e-1, 1.0e-3)
    # pairs (0, 1), (2, 3), ...: each order of large and small, zeros beside either, the smallest numbers
    for k, f in enumerate([big, small, small, big, 0.0, big, 1.0e-30, 0.0]):
        y[k] *= np.float32(f)
    ang = (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, 0.0], np.float32)
    dy = torch.from_numpy(y).cuda()
    print(f"fbp n={n} pad={pad} {store}", flush=True)
    x = dv.fbp_device(dy, ang, paramf, np.array([n, a, s, n, pad, 0, 0, 7, 0, 0], np.int32), store=store)
    assert not bool(x[4].any()) and not bool(x[7].any())
    for k in (0, 1, 2, 3, 5, 6):
        one = dv.fbp_device(dy[k:k + 1].contiguous(), ang, paramf,
                            np.array([n, a, 1, n, pad, 0, 0, 7, 0, 0], np.int32), store=store)[0]
        if store == "f16" and k == 6:
            continue  # below the smallest FP16 value
        # FP64 rows rounded once: one FP32 (FP16) rounding may fall to the other side
        tol = 2.0**-22 if store == "f32" else 2.0**-9
        assert float((x[k] - one).double().norm()) <= tol * float(one.double().norm()), k
