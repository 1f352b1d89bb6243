"""The narrowphase entry point at the sizes where its work split changes: one
pair per wave (one, two and three hits take different EPA tiers), the last
partial workgroup, one pair more than a whole number of shares, and the first
sizes with larger shares.  Bit for bit against the oracle in both arithmetic modes."""
import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("islands", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 3, 65, 777, 3073, 24575, 24577, 36865])
def test_sizes_around_the_shares(n, islands, oracle_mod):
    pairs = S.config2_pairs(n, seed=S.SEED + 31 + n)
    params = S.StepParams()
    params.fp64_islands = islands
    ctx = runtime.Context(params)
    got = ctx.narrow_to_numpy(ctx.narrowphase(ctx.upload_pairs(pairs)))
    ref = oracle_mod.narrowphase(pairs, params, "f32")
    assert got["n_overflow"] == 0
    for k in ("gjk", "contact", "normal", "depth", "point_a", "point_b"):
        a, b = got[k], ref[k]
        assert ((a == b) | (np.isnan(a) & np.isnan(b))).all(), k
    ctx.close()
