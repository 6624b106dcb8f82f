"""Device memory that a context keeps from one chain for the next: chains built, grown and dropped in
several threads at once end bit-identical to the first chains of a fresh context, memory in use is accounted
as if every buffer were allocated anew, and what lies idle makes room before an allocation is refused."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = 3.0
KS = (40, 150, 300, 90)


def _flow(nk, ctx, K, drop_early=False):
    g = nk.NrgCore(nk.Site.spinhalf(-0.25, 0.5), nk.Site.spinhalf(0, 0), K, ctx=ctx)
    op = nk.SystemOperator(g, nk.Site.fdag_chi_spinhalf())
    rec = nk.FdmRecorder(g, op)
    for n in range(7):
        g.add_bath_site([0.4 * L ** (-0.1 * n)] * 2, 1.0 if n == 0 else np.sqrt(L))
        if op is not None:
            op.update()
        if g.checkHigherEnergyDiscarded():
            rec.record()
        g.update_internal_state()
        if drop_early and n == 4:
            del rec, op  # an observable and a recorder may go before their chain
            op, rec = None, nk.FdmRecorder(g, None)
    return g.all_eigenvalue.copy(), ctx.used_bytes()[0]


def test_chains_in_threads_reuse_memory(nk):
    ctx = nk.Context()
    first = [_flow(nk, ctx, K)[0] for K in KS]
    assert ctx.used_bytes()[0] == 0
    bad = []

    def work(i):
        for r in range(4):
            e, _ = _flow(nk, ctx, KS[(i + r) % 4], drop_early=r % 2 == 1)
            if not np.array_equal(e, first[(i + r) % 4]):
                bad.append((i, r))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    assert ctx.used_bytes()[0] == 0


def test_idle_memory_makes_room(nk):
    ctx = nk.Context()
    e0, need = _flow(nk, ctx, 300)
    ctx.set_capacity(int(need * 1.05))
    for K in (40, 300, 90, 300):  # fits as in a fresh context, whatever the chains before it left
        e, used = _flow(nk, ctx, K)
        if K == 300:
            assert used == need
            np.testing.assert_array_equal(e, e0)
    ctx.set_capacity(need // 2)
    with pytest.raises(nk.NrgkError):
        _flow(nk, ctx, 300)
    ctx.set_capacity(0)
    np.testing.assert_array_equal(_flow(nk, ctx, 300)[0], e0)
