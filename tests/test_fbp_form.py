"""Which backprojector an FBP call takes (raft_fbp_form_info): the matrix form
only where its staged windows and offsets hold."""
import numpy as np
import pytest

GATHER, SPLIT, MATRIX = 0, 1, 2


def _angles(a):
    return (np.linspace(0.0, np.pi, a, endpoint=False) + 0.01).astype(np.float32)


def _params(n, a, s, filt=7, pad=2, blocksize=0):
    paramf = np.array([0.0, 0.0, 0.0, 0.0, 2.0 / n, 2.0 / n, 0.0], np.float32)
    return paramf, np.array([n, a, s, n, pad, 0, 0, filt, 0, blocksize], np.int32)


def _form(ang, n, s, store, **kw):
    from sscRaft import device as dv

    return dv.fbp_form_info(ang, *_params(n, len(ang), s, **kw), store=store)


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("n,a,s,store", [(128, 200, 16, "f16"), (512, 260, 64, "f32")])
def test_non_finite_angle_keeps_the_gather_form(n, a, s, store, bad):
    ang = _angles(a)
    form, tlo, width = _form(ang, n, s, store)
    assert form == MATRIX and width > n
    ang[a // 3] = bad
    assert _form(ang, n, s, store)[0] != MATRIX


@pytest.mark.parametrize("n,s,store", [
    (64, 6_400_000, "f32"),   # 4.5 GB of rows an angle: 32-bit offsets would wrap
    (8, 36_000_000, "f16"),
    (8, 524_281, "f16"),      # one slice past 65535 groups, which the gather form refuses
    (64, 262_141, "f32"),
])
def test_blocks_past_one_launch_keep_the_gather_form(n, s, store):
    ang = _angles(400)
    assert _form(ang, n, s, store)[0] != MATRIX
    # in blocks each launch is small
    form, _, width = _form(ang, n, s, store, blocksize=4096)
    assert form == MATRIX and width <= 1.5 * n + 128


@pytest.mark.parametrize("n,s,store,few,many", [
    # angles at which the matrix form took longer, and at which it gains
    (2048, 64, "f32", 32, 128),
    (2048, 32, "f32", 24, 128),
    (2048, 16, "f32", 96, 2048),
    (1024, 64, "f32", 16, 96),
    (512, 200, "f32", 48, 512),
    (512, 64, "f32", 32, 256),
    (200, 150, "f32", 8, 48),
    (2048, 32, "f16", 16, 64),
    (1024, 16, "f16", 64, 512),
    (512, 64, "f16", 24, 96),
    (200, 70, "f16", 32, 200),
    (64, 70, "f16", 32, 96),
    (16, 16, "f16", 24, 48),
])
def test_few_angles_keep_the_gather_form(n, s, store, few, many):
    assert _form(_angles(few), n, s, store)[0] != MATRIX
    assert _form(_angles(2), n, s, store)[0] != MATRIX
    assert _form(_angles(many), n, s, store)[0] == MATRIX


@pytest.mark.parametrize("n,s,whole,split", [
    (512, 1, 63, 64),     # 128 workgroups
    (400, 8, 64, 128),    # 182
    (512, 8, 128, 160),   # 256
    (600, 4, 64, 128),    # 190
    (64, 9, 63, 64),
])
def test_few_angles_are_not_split(n, s, whole, split):
    assert _form(_angles(whole), n, s, "f32")[0] == GATHER
    assert _form(_angles(split), n, s, "f32")[0] == SPLIT
