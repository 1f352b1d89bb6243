"""The adjoint kernel's variants give one world's gradients alike: 64 and 256 threads
a world, the iteration history in LDS and in scratch, contacts beyond the first one
of each thread.  The variant follows from the largest world of the batch."""
import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu


def _stack(side, layers, seed):
    r = np.random.default_rng(seed)
    g = np.array([(0.98 * i, 0.49 + 0.98 * k, 0.98 * j) for k in range(layers) for i in range(side) for j in range(side)])
    pos = (g + r.uniform(-0.01, 0.01, g.shape)).astype(np.float32)
    n = len(pos)
    return S._world(pos, np.ones((n, 3), np.float32), np.ones(n, np.float32), np.zeros((0, 3)), np.zeros((0, 3)), [], [])


@pytest.mark.parametrize("steps,every,iters", [(5, 2, 10), (3, 3, 70)])
def test_variants_agree(steps, every, iters):
    """A 48-body stack (more than 64 contacts) alone, beside 65 and beside 500 bodies,
    at 10 iterations (history in LDS in the first two) and 70 (in scratch).  State and
    mass gradients are the same arithmetic in the same order, so equal bit for bit;
    friction and restitution sum over the contacts in an order set by the thread
    count, so they agree to the rounding of that sum."""
    a = _stack(4, 3, 1)
    dl = np.random.default_rng(3).normal(size=(a.nbodies, 3)).astype(np.float32)
    got = []
    for other in (None, _stack(5, 3, 2), _stack(8, 8, 4)):
        sc = a if other is None else S.concat([a, other])
        sc.params = S.config4().params
        ctx = runtime.Context(sc.params, solver_iterations=iters)
        ctx.upload(sc)
        ctx.record_contacts()
        ctx.rollout(steps, every)
        assert len(ctx.contacts(0)) > 64
        d = np.zeros((sc.nbodies, 3), np.float32)
        d[: a.nbodies] = dl
        got.append(ctx.adjoint(dl_pos=d))
        ctx.close()
    n = a.nbodies
    for g in got[1:]:
        for k in ("pos0", "vel0", "angvel0", "angles0", "mass", "moi"):
            np.testing.assert_array_equal(g[k][:n], got[0][k][:n], err_msg=k)
        for k in ("friction", "restitution"):
            assert np.isfinite(got[0][k][0])
            np.testing.assert_allclose(g[k][0], got[0][k][0], rtol=1e-4, atol=1e-4, err_msg=k)
