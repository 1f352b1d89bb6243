"""State in and out of a batch: staged for small batches, field by field for larger
ones; quaternions of set_state's angles, whenever they are asked for."""
import ctypes

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


@pytest.mark.parametrize("n", [8192, 8193, 70_000])
def test_null_force_and_torque_are_zero_when_set_state_returns(n):
    """NULL force and torque overwrite the planes with zeros, and the call has synchronised
    when it returns: its stream is idle, and a call on another stream reads the zeros.
    With the warm start on, its emptied lists too."""
    import torch
    sc = _scene(n) if n < 10_000 else S.concat([_scene(7) for _ in range(n // 7)])
    ctx = runtime.Context(sc.params)
    ctx.upload(sc)
    ctx.set_warm_start(True)
    if n < 10_000:
        ctx.step_plain(1)  # the contact lists exist from here on
    one, other = torch.cuda.Stream(), torch.cuda.Stream()
    planes = {k: np.ascontiguousarray(getattr(sc, k).T) for k in STATE}
    ptr = lambda a: ctypes.c_void_p(a.ctypes.data)
    for _ in range(3):
        ctx.set_state(sc)
        np.testing.assert_array_equal(ctx.download()["force"], sc.force)
        b = runtime.BodiesSoa(*[ptr(planes[k]) for k in STATE[:4]], *([None] * 6))
        runtime.check(ctx.lib.nans_set_stream(ctx.h, ctypes.c_void_p(one.cuda_stream)))
        runtime.check(ctx.lib.nans_set_state(ctx.h, ctypes.byref(b)))
        assert one.query()
        runtime.check(ctx.lib.nans_set_stream(ctx.h, ctypes.c_void_p(other.cuda_stream)))
        got = ctx.download()
        for k in STATE[:4]:
            np.testing.assert_array_equal(got[k], getattr(sc, k), err_msg=k)
        assert not got["force"].any() and not got["torque"].any()
        runtime.check(ctx.lib.nans_set_stream(ctx.h, ctypes.c_void_p(one.cuda_stream)))
        ctx.set_warm_start(False)
        ctx.set_warm_start(True)
        assert one.query()
    ctx.close()
