"""Weakly coupled levels: tridiagonal and block-tridiagonal matrices whose eigenvalues come in many copies,
equal to entries of the diagonal to the last bit, with couplings of 1e-20 to 1e-3 between them.  Orthogonality,
residual and eigenvalues to 1e-10 (the bar of the wide blocks' path; the inverse iteration leaves 1e-13 to 1e-12),
above the crossover, on narrow blocks sent there and through the batched solver."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _block(rng, kind, n):
    off = np.zeros(n - 1)
    if kind == "two_levels":
        d, off = rng.choice([0.0, 1.0], n), 10.0 ** rng.uniform(-14, -4, n - 1)
    elif kind == "very_weak":
        d, off = rng.choice([0.0, 1.0], n), 10.0 ** rng.uniform(-20, -6, n - 1)
    elif kind == "five_levels":
        d, off = rng.choice([-1.0, -0.5, 0.25, 0.3, 2.0], n), 10.0 ** rng.uniform(-16, -3, n - 1)
    elif kind == "one_level":
        d, off = np.full(n, 0.7), 10.0 ** rng.uniform(-16, -5, n - 1)
    else:  # copies of one 8 x 8 tridiagonal block
        d = np.resize(rng.uniform(-1, 1, 8), n)
        off = np.resize(rng.uniform(0.1, 1, 8), n - 1)
        off[7::8] = 10.0 ** rng.uniform(-18, -8, len(off[7::8]))
    return np.diag(d) + np.diag(off, 1) + np.diag(off, -1)


@pytest.mark.parametrize("kind", ["two_levels", "very_weak", "five_levels", "one_level", "copies"])
@pytest.mark.parametrize("sizes,mixed_max", [((769, 900), None), ((66, 150, 260, 333), "0"), ((66, 150, 260, 333, 640), None)])
def test_weak_couplings(nk, monkeypatch, kind, sizes, mixed_max):
    if mixed_max is not None:
        monkeypatch.setenv("NRGK_MIXED_MAX", mixed_max)
    rng = np.random.default_rng(77)
    blocks = [_block(rng, kind, n) for n in sizes for _ in range(4)]
    for H, (w, U) in zip(blocks, nk.eigh_batched(blocks)):
        n = len(w)
        assert np.abs(w - np.linalg.eigvalsh(H)).max() <= 1e-10, n
        assert np.abs(U.T @ U - np.eye(n)).max() <= 1e-10, n
        assert np.abs(H @ U - U * w).max() <= 1e-10, n
