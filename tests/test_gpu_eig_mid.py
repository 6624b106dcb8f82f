"""The batched solver's FP32 Householder stage with its FP64 refinement, at the widths where its kernels
change course: whole and partial strips (16 rows), tiles (64) and register blocks (more than 384 rows are
reduced in memory first), one-column panels, the widest block it takes (768).

H = Q diag(lam) Q^T with Haar Q.  Bounds, in units of the largest |lam|: forming H rounds it by about n eps
(1.7e-13 at 768 rows), the refinement leaves an orthogonality defect of at most 1e-12; everything is held
to 4e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 4e-12
SIZES = [65, 79, 80, 81, 96, 97, 127, 128, 129, 191, 192, 193, 256, 257, 319, 320, 321, 383, 384, 385, 400, 641, 767, 768]


def _block(rng, lam):
    n = len(lam)
    Q, R = np.linalg.qr(rng.standard_normal((n, n)))
    Q = Q * np.sign(np.diag(R))
    H = (Q * lam) @ Q.T
    return 0.5 * (H + H.T)


def _check(H, w, U, lam=None, scale=1.0):
    n = len(w)
    assert np.all(np.diff(w) >= 0), n
    if lam is not None:
        assert np.abs(w - lam).max() <= TOL * scale, n
    assert np.abs(U.T @ U - np.eye(n)).max() <= TOL, n
    assert np.abs(H @ U - U * w).max() <= TOL * scale, n


@pytest.mark.parametrize("kind", ["uniform", "degenerate", "graded"])
def test_edges(nk, kind):
    rng = np.random.default_rng(29)
    blocks, lams = [], []
    for n in SIZES:
        if kind == "degenerate":
            lam = rng.choice([-1.0, -0.5, 0.0, 0.25, 0.75], n)
        elif kind == "graded":
            lam = rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(-8, 0, n)
        else:
            lam = rng.uniform(-1, 1, n)
        lams.append(np.sort(lam))
        blocks.append(_block(rng, lams[-1]))
    for H, lam, (w, U) in zip(blocks, lams, nk.eigh_batched(blocks)):
        _check(H, w, U, lam)


@pytest.mark.parametrize("scale", [1e-60, 1e60])
def test_far_from_unit_scale(nk, scale):
    """entries whose FP32 values or squares would under- or overflow"""
    rng = np.random.default_rng(5)
    lams = [np.sort(rng.uniform(-1, 1, n)) for n in (100, 330)]
    blocks = [_block(rng, lam) * scale for lam in lams]
    for H, lam, (w, U) in zip(blocks, lams, nk.eigh_batched(blocks)):
        _check(H, w, U, lam * scale, scale)


def test_blocks_that_fall_apart(nk):
    """columns that are zero below the diagonal when the reduction reaches them (diagonal, block diagonal
    and tridiagonal blocks, a zero block, weak couplings), after a call that left NaN in device memory"""
    rng = np.random.default_rng(8)
    bad = _block(rng, rng.uniform(-1, 1, 400))
    bad[7, 9] = bad[9, 7] = np.nan
    (w, _), = nk.eigh_batched([bad])
    assert np.isnan(w).all()
    d = np.sort(rng.uniform(-1, 1, 200))
    two = np.zeros((350, 350))
    two[:150, :150] = _block(rng, rng.uniform(-1, 1, 150))
    two[150:, 150:] = _block(rng, rng.uniform(-1, 1, 200))
    weak = two.copy()
    weak[:150, 150:] = 1e-14 * rng.standard_normal((150, 200))
    weak[150:, :150] = weak[:150, 150:].T
    tri = np.diag(rng.uniform(-1, 1, 90)) + np.diag(np.full(89, 0.3), 1) + np.diag(np.full(89, 0.3), -1)
    blocks = [np.diag(d), two, weak, tri, np.zeros((70, 70)), np.eye(66)]
    out = nk.eigh_batched(blocks)
    for H, (w, U) in zip(blocks, out):
        _check(H, w, U, np.linalg.eigvalsh(H))
    np.testing.assert_array_equal(out[4][0], np.zeros(70))


def test_multiplets(nk):
    """clusters of one to 70 members, many of each size in a block: those of up to 8, up to 64 and more take
    different paths, and a block's are shared out over its workgroups"""
    rng = np.random.default_rng(13)
    blocks, lams = [], []
    for n in (66, 95, 96, 127, 128, 500, 768):
        sizes = []
        while sum(sizes) < n:
            sizes.append(int(rng.choice([1, 2, 3, 8, 9, 20, 64, 65, 70])))
        lam = np.repeat(rng.permutation(np.linspace(-1, 1, len(sizes))), sizes)[:n]
        lams.append(np.sort(lam))
        blocks.append(_block(rng, lam))
    for H, lam, (w, U) in zip(blocks, lams, nk.eigh_batched(blocks)):
        _check(H, w, U, lam)
