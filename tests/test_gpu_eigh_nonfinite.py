"""Blocks above the crossover whose tridiagonal form is not finite: a NaN, an infinity, or finite entries
whose squares overflow.  Every eigenvalue of such a block is NaN (never a plausible number), the other
blocks' results stand, and a chain whose hopping makes its blocks overflow fails its step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sym(rng, n):
    A = rng.standard_normal((n, n))
    return 0.5 * (A + A.T)


def _spoil(H, how):
    n = len(H)
    H = H.copy()
    if how == "nan":
        H[n // 2, n // 3] = H[n // 3, n // 2] = np.nan
    elif how == "nan_diagonal":
        H[n - 1, n - 1] = np.nan
    elif how == "inf_column0":
        H[0, n - 1] = H[n - 1, 0] = np.inf
    else:
        H *= 1e160
    return H


@pytest.mark.parametrize("how", ["nan", "nan_diagonal", "inf_column0", "overflow"])
@pytest.mark.parametrize("sizes,mixed_max", [((800, 820, 90), None), ((70, 65, 129, 300), "0")])
def test_wide_block_gives_nan(nk, monkeypatch, how, sizes, mixed_max):
    if mixed_max is not None:
        monkeypatch.setenv("NRGK_MIXED_MAX", mixed_max)
    rng = np.random.default_rng(11)
    blocks = [_sym(rng, n) for n in sizes]
    good = [H.copy() for H in blocks]
    blocks[0] = _spoil(blocks[0], how)
    out = nk.eigh_batched(blocks)
    assert np.isnan(out[0][0]).all()
    for H, (w, U) in list(zip(good, out))[1:]:
        assert np.abs(w - np.linalg.eigvalsh(H)).max() <= 1e-12 * np.abs(w).max()
        assert np.abs(H @ U - U * w).max() <= 1e-12 * np.abs(w).max()


def test_chain_step_reports_it(nk, monkeypatch):
    """an overflowing hopping: the step fails, it does not go on with zeros"""
    monkeypatch.setenv("NRGK_MIXED_MAX", "0")
    g = nk.NrgCore(nk.Site.spinhalf(-0.25, 0.5), nk.Site.spinhalf(0, 0), 64)
    with pytest.raises(nk.NrgkError, match="non-finite"):
        g.add_bath_site([1e160, 1e160], 1.0)
        g.update_internal_state()
