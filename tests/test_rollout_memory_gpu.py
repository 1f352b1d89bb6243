"""What a rollout keeps on the device: the caller's bound of the tape of every step."""
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
