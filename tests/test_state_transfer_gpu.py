"""State in and out of a batch: staged for small batches, field by field for larger
ones; quaternions of set_state's angles, whenever they are asked for."""
import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

pytestmark = pytest.mark.gpu

STATE = ("pos", "vel", "angvel", "angles", "force", "torque")


def _scene(n):
    r = np.random.default_rng(n)
    g = r.uniform(1, 500, (n, 3)).astype(np.float32)
    sc = S._world(g, np.ones((n, 3), np.float32), np.ones(n, np.float32), np.zeros((0, 3)), np.zeros((0, 3)), [], [])
    for k in STATE:
        setattr(sc, k, r.normal(size=(n, 3)).astype(np.float32) * 30)
    return sc


@pytest.mark.parametrize("n", [1, 8192, 8193])
def test_state_round_trip(n):
    """set_state then download returns every field, also after another state was there,
    and the quaternions are those of the given angles (as an upload's), in both modes
    and after the angles have moved on."""
    sc, other = _scene(n), _scene(n)
    other.pos = other.pos + 1.0
    other.angles = other.angles * 0.5
    ref = runtime.Context(sc.params)
    ref.upload(sc)
    quat = ref.quaternions()
    ref.close()
    ctx = runtime.Context(sc.params)
    ctx.upload(other)
    ctx.set_state(sc)
    got = ctx.download()
    for k in STATE:
        np.testing.assert_array_equal(got[k], getattr(sc, k), err_msg=k)
    np.testing.assert_array_equal(ctx.quaternions(), quat)
    ctx.set_state(other)
    ctx.set_state(sc)
    ctx.step_plain(1)
    np.testing.assert_array_equal(ctx.quaternions(), quat)
    ctx.set_state(other)
    ctx.set_orientation_mode("quaternion")
    ctx.set_state(sc)
    np.testing.assert_array_equal(ctx.quaternions(), quat)
    ctx.close()
