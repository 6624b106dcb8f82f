"""The sweep count of a step's statistics is that step's: of the small blocks' Jacobi where it ran, zero in
the steps whose blocks went to another solver."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_sweeps_of_the_step(nk):
    L = 3.0
    g = nk.NrgCore(nk.Site.spinhalf(-0.25, 0.5), nk.Site.spinhalf(0, 0), 400)
    small, other = 0, 0
    for n in range(7):
        g.add_bath_site([0.4 * L ** (-0.1 * n)] * 2, 1.0 if n == 0 else np.sqrt(L))
        dims = [int(d) for d in g.sectors()[1]]
        sweeps = g.step_stats()["jacobi_sweeps"]
        if max(dims) <= 64:
            assert sweeps > 0, n
            small += 1
        else:
            assert sweeps == 0, n
            other += 1
        g.update_internal_state()
    assert small and other
