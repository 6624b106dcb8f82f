"""The element of rank K that cuts the spectrum: among few keys (compared with each other) and among many equal
ones (all digits by histogram).  Kept counts against sorted[K] + 1e-8 of the same eigenvalues
(nrgcore/include/nrgcore/nrgcore.hpp:269-327), exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [3, 20, 63, 64, 65, 100, 400])
@pytest.mark.parametrize("t,eps,U", [(0.0, 0.0, 0.0), (0.0, -0.3, 0.5), (0.7, 0.0, 0.0), (0.4, -0.23, 0.5)])
def test_kept_counts(nk, K, t, eps, U):
    g = nk.NrgCore(nk.Site.spinhalf(eps, U), nk.Site.spinhalf(0, 0), K)
    cut = 0
    for n in range(6):
        g.add_bath_site([t * 0.9 ** n] * 2, 1.0 if n == 0 else np.sqrt(2.5))
        g.update_internal_state()
        e = np.sort(g.all_eigenvalue)
        want = len(e) if len(e) <= K else int((e < e[K] + 1e-8).sum())
        assert int(np.sum(g.kept_counts())) == want, (n, len(e))
        cut += len(e) > K
        if cut == 2:
            break
    assert cut
