"""The narrowphase entry point where most pairs miss: its waves claim pairs more often than
they work on them, and take more with a claim the longer a run of misses gets."""
import time

import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu


def _sparse(n, hits, seed):
    """config2's pairs with all but the chosen ones moved apart."""
    pairs = S.config2_pairs(n, seed=seed)
    apart = np.ones(n, bool)
    apart[hits] = False
    pairs["pos_b"] = np.where(apart[:, None], pairs["pos_b"] + np.float32(30), pairs["pos_b"]).astype(np.float32)
    return pairs


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("n", [127, 128, 129, 12289, 98303, 98305, 200_003])
def test_mostly_misses(n, noalloc, oracle_mod):
    """Fewer workgroups than counters and more, shares of 1 to 16 pairs, claims that have
    doubled and fallen back: pairs that touch at the front, in a clump, strewn about and at
    the end.  Every output bit for bit, and every pair written."""
    r = np.random.default_rng(n)
    hits = np.unique(np.concatenate([np.arange(2), n // 2 + np.arange(40), [n - 1], r.integers(0, n, n // 200)]))
    pairs = _sparse(n, hits, S.SEED + n)
    params = S.StepParams()
    ctx = runtime.Context(params)
    out = ctx.alloc_narrow_out(n)
    for k in ("gjk", "contact", "status"):
        out[k].fill_(-7)
    got = ctx.narrow_to_numpy(ctx.narrowphase(ctx.upload_pairs(pairs), out, noalloc=noalloc))
    ref = oracle_mod.narrowphase(pairs, params, "f32")
    assert 0 < int(ref["contact"].sum()) < len(hits) + 1
    for k in ("gjk", "contact", "normal", "depth", "point_a", "point_b"):
        a, b = got[k], ref[k]
        assert ((a == b) | (np.isnan(a) & np.isnan(b))).all(), k
    assert (got["status"] >= 0).all() and got["n_overflow"] == 0
    ctx.close()


def test_misses_cost_less_than_hits():
    """A call whose pairs all miss does nothing but claim pairs and reject them: it takes
    a small part of the time of the same number of random pairs, half of which touch
    (30011 pairs: 0.04 of it with 118 workgroups in lockstep, 0.2 here; 0.68 where one
    counter serialised the claims)."""
    n = 30011
    ctx = runtime.Context(S.StepParams())
    best = []
    for pairs in (_sparse(n, np.zeros(0, int), 3), S.config2_pairs(n, seed=3)):
        dp, out = ctx.upload_pairs(pairs), ctx.alloc_narrow_out(n)
        t = []
        for _ in range(30):
            t0 = time.perf_counter()
            ctx.narrowphase(dp, out)
            t.append(time.perf_counter() - t0)
        best.append(min(t))
        assert (int(out["contact"].sum()) == 0) == (len(best) == 1)
    ctx.close()
    assert best[0] < 0.4 * best[1], best
