"""What a rollout keeps on the device: the caller's bound of the tape of every step, and
the tape of a longer rollout serving a shorter one."""
import numpy as np
import pytest
import torch

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _batch(worlds=256):
    sc = S.config4(nworlds=worlds, nsteps=1)
    ctx = runtime.Context(sc.params)
    ctx.upload(sc)
    return sc, ctx


def _gradient(sc, ctx, nsteps, every=16):
    ctx.set_state(sc)
    ctx.rollout(nsteps, every)
    return ctx.adjoint(dl_pos=np.ones((sc.nbodies, 3), np.float32))


def test_caller_bounds_the_tape():
    """256 worlds of 16 bodies, 160 steps: every step's state (45 MiB) and contacts (200 MiB)
    are kept by default, not with less allowed, given back once less is allowed, and kept
    again with enough; without them the adjoint holds the contacts of a 16-step segment
    (100 MiB) and ten states (3 MiB) instead.  The gradients are the same bit for bit."""
    sc, ctx = _batch()
    with pytest.raises(runtime.NansError):
        runtime.check(ctx.lib.nans_set_rollout_memory(None, 0))
    ctx.set_rollout_memory(0)
    got = [_gradient(sc, ctx, 160)]
    before = _free()
    for limit, kept in ((-1, True), (100 * MIB, False), (300 * MIB, True), (0, False)):
        ctx.set_rollout_memory(limit)
        got.append(_gradient(sc, ctx, 160))
        more = (before - _free()) / MIB
        assert (110 < more < 170) if kept else (-10 < more < 10), (limit, more)
    for g in got[1:]:
        for k, v in got[0].items():
            np.testing.assert_array_equal(g[k], v, err_msg=k)
    ctx.close()


def test_a_shorter_rollout_fits_the_tape():
    """After 160 steps' tape (245 MiB), rollouts of 100 and 41 steps allocate and free
    nothing; one of 16 takes a tape of its own (25 MiB).  Each gives the gradient that it
    gives on a context of its own, and so does 160 again."""
    sc, ctx = _batch()
    want = {}
    for n in (16, 41, 100, 160):
        _, own = _batch()
        want[n] = _gradient(sc, own, n, 7)
        own.close()
    _gradient(sc, ctx, 160, 7)
    before = _free()
    for n, lo, hi in ((160, -1, 1), (100, -1, 1), (41, -1, 1), (160, -1, 1), (16, 200, 240), (160, -1, 1)):
        got = _gradient(sc, ctx, n, 7)
        assert lo < (_free() - before) / MIB < hi, (n, _free() - before)
        for k, v in want[n].items():
            np.testing.assert_array_equal(got[k], v, err_msg="%d %s" % (n, k))
    ctx.close()


def test_refusal_keeps_the_checkpoints():
    """A rollout that may not keep a tape uses the buffer of the one before it, whether that
    was refused too or had a tape, and gradients do not depend on it."""
    sc, ctx = _batch(64)
    _, own = _batch(64)
    want = [_gradient(sc, own, 24, 5), _gradient(sc, own, 31, 5)]
    own.close()
    ctx.set_rollout_memory(0)
    for n, i in ((24, 0), (24, 0), (31, 1), (24, 0)):
        got = _gradient(sc, ctx, n, 5)
        for k, v in want[i].items():
            np.testing.assert_array_equal(got[k], v, err_msg="%d %s" % (n, k))
    ctx.set_rollout_memory(-1)
    for limit in (-1, 0, -1):
        ctx.set_rollout_memory(limit)
        got = _gradient(sc, ctx, 24, 5)
        for k, v in want[0].items():
            np.testing.assert_array_equal(got[k], v, err_msg=k)
    ctx.close()


@pytest.mark.parametrize("limit", [-1, 0])
def test_batched_timing_after_a_rollout(limit):
    """nans_batched_timing names the launch shape after a rollout as after a step, with a
    tape and with checkpoints; before either it refuses."""
    sc, ctx = _batch(4)
    ctx.set_rollout_memory(limit)
    with pytest.raises(runtime.NansError):
        ctx.batched_timing()
    ctx.rollout(7, 3)
    t = ctx.batched_timing()
    assert t["workgroups"] > 0 and t["threads_per_world"] == 128 and t["steps"] == 1 and t["elapsed_ms"] == 0.0
    ctx.step_batched(5)
    t = ctx.batched_timing()
    assert t["steps"] == 5 and t["elapsed_ms"] > 0.0
    ctx.close()
