"""FBP calls of few tiles split the angles over workgroups (k_backproject MODE 2,
k_bp_groups); raft_fbp_device_noalloc runs the whole form, and both add the same
groups of angles in the same order."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,a,s,offset", [
    (2, 64, 1, 0.0),      # fewer pixels than a float4
    (65, 64, 1, 0.0),     # the fewest angles; count no multiple of 4
    (97, 71, 3, 2.0),     # a last group of 7 angles
    (200, 257, 5, 0.0),   # two slice groups
    (512, 300, 2, -3.0),  # several groups a workgroup
    (64, 4099, 9, 0.0),   # many groups
])
def test_split_equals_whole(gpu, n, a, s, offset):
    import torch
    from sscRaft import device as dv

    rng = np.random.default_rng(n)
    y = rng.standard_normal((s, a, n)).astype(np.float32) + np.float32(1.0)
    ang = np.linspace(0.0, np.pi, a, endpoint=False).astype(np.float32)
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, offset], np.float32)
    parami = np.array([n, a, s, n, 2, 0, 0, 7, 0, 0], np.int32)
    print(f"fbp n={n} a={a} s={s} offset={offset}", flush=True)
    dy = torch.from_numpy(y).cuda()
    x = torch.full((s, n, n), float("nan"), device="cuda")
    w = torch.full((s, n, n), float("nan"), device="cuda")
    dv.fbp_device(dy, ang, paramf, parami, out=x)
    dv.fbp_device(dy, ang, paramf, parami, out=w, noalloc=True)
    assert torch.equal(x, w)
    want = oracle.fbp(y, ang, paramf, parami)
    assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-5 * np.linalg.norm(want)
