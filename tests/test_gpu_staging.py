"""Several solves of one context at once whose descriptor tables and readbacks take more than one staging
chunk (over 1 MiB between two synchronisations): each is bit-identical to the same solve alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _blocks(seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in [70] + [int(n) for n in rng.integers(2, 16, 2500)]:
        H = rng.standard_normal((n, n))
        out.append(0.5 * (H + H.T))
    return out


def test_concurrent_solves_above_one_chunk(nk):
    ctx = nk.Context()
    batches = [_blocks(s) for s in range(4)]
    alone = [nk.eigh_batched(b, ctx=ctx) for b in batches]
    for H, (w, U) in zip(batches[0], alone[0]):
        assert np.abs(H @ U - U * w).max() <= 1e-12 * np.abs(w).max()
    bad = []

    def work(i):
        for r in range(3):
            k = (i + r) % 4
            out = nk.eigh_batched(batches[k], ctx=ctx)
            if not all(np.array_equal(a, b) for x, y in zip(out, alone[k]) for a, b in zip(x, y)):
                bad.append((i, r))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    assert ctx.used_bytes()[0] == 0
