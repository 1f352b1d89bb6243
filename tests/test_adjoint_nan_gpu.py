"""A rollout whose state leaves the numbers has no gradient: the adjoint says so, with the
step and the world, and does not report its replay as different from the rollout."""
import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tape", [True, False])
def test_nan_state_is_named(tape):
    """A body of world 2 starts with a NaN velocity, and one of world 3 at an infinite
    position, which stays equal to itself: 8 world-steps are NaN, the first is step 0 of
    world 2, through the tape and through checkpoints.  From a finite state the batch gives
    gradients again."""
    sc, bad = (S.config4(nworlds=4, nsteps=8) for _ in range(2))
    bad.vel[int(sc.offsets[2]) + 5] = np.nan
    bad.pos[int(sc.offsets[3]) + 7, 0] = np.inf
    ctx = runtime.Context(sc.params)
    ctx.upload(sc)
    ctx.record_contacts(not tape)
    d = np.ones((sc.nbodies, 3), np.float32)
    ctx.set_state(bad)
    ctx.rollout(8, 3)
    with pytest.raises(runtime.NansError) as e:
        ctx.adjoint(dl_pos=d)
    assert e.value.code == runtime.ERR_STATE
    assert "not a number in 8 world-steps, from step 0 of world 2 on" in str(e.value)
    ctx.set_state(sc)
    ctx.rollout(8, 3)
    assert all(np.isfinite(v).all() for v in ctx.adjoint(dl_pos=d).values())
    ctx.close()
