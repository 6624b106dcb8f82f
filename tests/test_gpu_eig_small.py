"""The one-launch solver of the small blocks (up to 64 rows), at the edges of its lanes and tiles: a
16-lane row of matrix rows (15, 16, 17, ... 64), odd counts (a column without a partner), one row, and
the first width it leaves to the batched solver (65).

H = Q diag(lam) Q^T with Haar Q.  Bounds, in units of the largest |lam|: forming H rounds it by about
n eps (1.4e-14 at 64 rows), a rotation stops at cosines of 1e-13 between columns, so orthogonality,
residual and eigenvalues are held to 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _block(rng, lam):
    n = len(lam)
    Q, R = np.linalg.qr(rng.standard_normal((n, n)))
    Q = Q * np.sign(np.diag(R))
    H = (Q * lam) @ Q.T
    return 0.5 * (H + H.T)


def _check(H, lam, w, U, scale):
    n = len(lam)
    assert np.all(np.diff(w) >= 0)
    assert np.abs(w - lam).max() <= TOL * scale
    assert np.abs(U.T @ U - np.eye(n)).max() <= TOL
    assert np.abs(H @ U - U * w).max() <= TOL * scale


@pytest.mark.parametrize("kind", ["uniform", "degenerate", "clustered", "graded"])
@pytest.mark.parametrize("scale", [1.0, 1e-160, 1e120])
def test_edges(nk, kind, scale):
    """also far from unit scale: squares of the entries would under- or overflow"""
    rng = np.random.default_rng(17)
    blocks, lams = [], []
    for n in (1, 2, 3, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64):
        if kind == "degenerate":
            lam = rng.choice([-1.0, 0.0, 0.25], n)
        elif kind == "clustered":
            lam = np.repeat(rng.uniform(-1, 1, n), 3)[:n] + 1e-12 * np.arange(n)
        elif kind == "graded":
            lam = rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(-10, 0, n)
        else:
            lam = rng.uniform(-1, 1, n)
        lam = np.sort(lam) * scale
        lams.append(lam)
        blocks.append(_block(rng, lam / scale) * scale)
    for H, lam, (w, U) in zip(blocks, lams, nk.eigh_batched(blocks)):
        _check(H, lam, w, U, scale)


def test_beside_wider_blocks(nk):
    """small blocks in a batch with the first wider ones, in mixed order"""
    rng = np.random.default_rng(3)
    lams = [np.sort(rng.uniform(-1, 1, n)) for n in (65, 64, 1, 130, 40, 66)]
    blocks = [_block(rng, lam) for lam in lams]
    for H, lam, (w, U) in zip(blocks, lams, nk.eigh_batched(blocks)):
        _check(H, lam, w, U, 1.0)


def test_non_finite_block_gives_nan(nk):
    """in that block alone"""
    H = np.eye(20)
    H[3, 4] = H[4, 3] = np.nan
    (w0, U0), (w, _) = nk.eigh_batched([np.eye(5), H])
    assert np.isnan(w).all()
    np.testing.assert_allclose(w0, np.ones(5), atol=1e-15)
    np.testing.assert_allclose(U0 @ U0.T, np.eye(5), atol=1e-15)


def test_nan_block(nk):
    """a NaN entry: every eigenvalue of that block is NaN, as the wider blocks' are, and the others' stand"""
    rng = np.random.default_rng(4)
    lams = [np.sort(rng.uniform(-1, 1, n)) for n in (64, 20, 33)]
    blocks = [_block(rng, lam) for lam in lams]
    nk.eigh_batched(blocks)
    blocks[1][3, 5] = blocks[1][5, 3] = np.nan
    out = nk.eigh_batched(blocks)
    assert np.isnan(out[1][0]).all()
    for i in (0, 2):
        _check(blocks[i], lams[i], *out[i], 1.0)
