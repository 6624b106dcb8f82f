"""A crossover above the widest block that the batched solver takes (768 rows) stands for that width: wider
blocks take the wide blocks' path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed_max", ["769", "1000", "1000000"])
def test_crossover_above_the_batched_solver(nk, monkeypatch, mixed_max):
    rng = np.random.default_rng(6)
    blocks = []
    for n in (769, 800, 768, 90):
        A = rng.standard_normal((n, n))
        blocks.append(0.5 * (A + A.T))
    ref = nk.eigh_batched(blocks)
    monkeypatch.setenv("NRGK_MIXED_MAX", mixed_max)
    for (w0, U0), (w, U) in zip(ref, nk.eigh_batched(blocks)):
        np.testing.assert_array_equal(w, w0)
        np.testing.assert_array_equal(U, U0)
