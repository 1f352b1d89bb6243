"""The batched step's launches: a world's steps run one after another inside one
launch, and a call longer than a launch's bound (256 steps) continues in another."""
import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu

STATE = ("pos", "vel", "angvel", "angles", "force", "torque")


@pytest.mark.parametrize("block,wave,warm", [(0, -1, False), (256, 16, False), (64, -1, True), (256, 16, True)])
def test_one_call_equals_many(block, wave, warm):
    """259 steps in one call (two launches) = one-step calls, then 2, then the rest:
    state and the recorded contacts of the last step, with worlds on workgroups and
    on waves, cold and warm-started."""
    sc = S.config3(6, nsteps=1)
    outs = []
    for calls in ([259], [1, 1, 1, 2, 254]):
        ctx = runtime.Context(sc.params)
        ctx.upload(sc)
        ctx.set_batched_block(block)
        ctx.set_wave_worlds(wave)
        ctx.set_warm_start(warm)
        ctx.record_contacts()
        for n in calls:
            ctx.step_batched(n)
        outs.append((ctx.download(), [ctx.contacts(w) for w in range(sc.nworlds)], ctx.stats()))
        ctx.close()
    for f in STATE:
        np.testing.assert_array_equal(outs[0][0][f], outs[1][0][f], err_msg=f)
    for a, b in zip(outs[0][1], outs[1][1]):
        assert a.tobytes() == b.tobytes()
    assert outs[0][2] == outs[1][2]
