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


@pytest.mark.parametrize("steps,every,iters,tape", [(5, 2, 10, True), (3, 3, 70, True), (5, 2, 10, False)])
def test_variants_agree(steps, every, iters, tape):
    """A 48-body stack (more than 64 contacts) alone, beside 65 and beside 500 bodies,
    at 10 iterations (history in LDS in the first two) and 70 (in scratch), from the
    rollout's tape and (a batch that records contacts) from its checkpoints.  State and
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
        ctx.step_batched(1)
        assert len(ctx.contacts(0)) > 64
        ctx.set_state(sc)
        ctx.record_contacts(not tape)
        ctx.rollout(steps, every)
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


def test_tape_and_checkpoints_agree():
    """Gradients through the kept contacts of every step equal those through the
    recomputed segments, also where the tape's room (four contacts per body) runs out
    (every box of a heap of coincident cubes touches all others)."""
    r = np.random.default_rng(5)
    heap = S._world(np.float32([1.0, 3.0, 1.0]) + r.uniform(-0.2, 0.2, (20, 3)).astype(np.float32),
                    np.ones((20, 3), np.float32), np.ones(20, np.float32), np.zeros((0, 3)), np.zeros((0, 3)), [], [])
    for sc in (_stack(3, 2, 7), heap):
        sc.params = S.config4().params
        d = r.normal(size=(sc.nbodies, 3)).astype(np.float32)
        got = []
        for record in (False, True):
            ctx = runtime.Context(sc.params)
            ctx.upload(sc)
            ctx.record_contacts(record)
            for _ in range(2):  # the second rollout's tape has the room the first one lacked
                ctx.set_state(sc)
                ctx.rollout(7, 3)
                got.append((ctx.adjoint(dl_pos=d), ctx.download()))
            ctx.close()
        for g in got[1:]:
            for a, b in zip(got[0], g):
                for k in a:
                    np.testing.assert_array_equal(a[k], b[k], err_msg=k)
