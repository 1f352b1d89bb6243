"""Worlds of many overlapping bodies, bit for bit against the oracle: contact lists longer
than the solver's store of terms, which are then solved in parts, and boxes mixed with
spheres, whose pairs leave the lanes' EPA by different ways (nans_epa.hpp)."""
import numpy as np
import pytest

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

from test_step_gpu import _state_equal

pytestmark = pytest.mark.gpu

Z3, Z = np.zeros((0, 3), np.float32), np.zeros(0, np.float32)


def _params():
    return S.StepParams(dt=1.0 / 120.0, solver_iterations=10, restitution=0.2, friction=0.5)


def _heap(n, spread, seed):
    """Unit cubes whose centres lie in a small cube: (almost) every pair touches."""
    r = np.random.default_rng(seed)
    pos = (np.array([2.0, 3.0, 2.0]) + r.uniform(-spread, spread, (n, 3))).astype(np.float32)
    sc = S._world(pos, np.ones((n, 3), np.float32), np.ones(n, np.float32), Z3, Z3, Z, Z)
    sc.params = _params()
    return sc


def _mixed(nbox, nsph, seed):
    """Turned boxes and spheres thrown together: lanes, groups and the whole wave all have work."""
    r = np.random.default_rng(seed)
    at = lambda n: (np.array([2.0, 2.2, 2.0]) + r.uniform(-1.3, 1.3, (n, 3))).astype(np.float32)
    sc = S._world(at(nbox), r.uniform(0.6, 1.4, (nbox, 3)).astype(np.float32), np.ones(nbox, np.float32), at(nsph),
                  np.zeros((nsph, 3)), r.uniform(0.3, 0.6, nsph), np.ones(nsph))
    sc.angles[:nbox] = r.uniform(-180.0, 180.0, (nbox, 3)).astype(np.float32)
    sc.params = _params()
    return sc


# Bytes of a contact's terms (35 words), and an upper bound of the terms a step has room
# for: all of a CU's LDS in the plain step; in the batched one the radii and polytopes (12 KB
# a wave at most), and a contact record (20 words) per candidate in scratch.
TERMS = 140


def _room(path, n, npairs, threads):
    if path == "plain":
        return 160 * 1024 // TERMS
    return (4 * n + 12 * 1024 * max(threads, 64) // 64) // TERMS + 4 * npairs // 7


@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("path,threads", [("plain", 0), ("batched", 64), ("batched", 256)])
def test_contact_lists_solved_in_parts(oracle_mod, path, threads, warm):
    n = 72
    sc = _heap(n, 0.22, 11)
    ctx = runtime.Context(sc.params)
    ctx.upload(sc)
    ctx.set_batched_block(threads)
    ctx.set_warm_start(warm)
    ws = oracle_mod.WorldState(sc, 0, "f32")
    if warm:
        ws.enable_warm(16 * n + 64)
    npairs = n * (n - 1) // 2 + n
    longest = 0
    for k in range(4):
        before = ctx.stats()["contacts"]
        (ctx.step_plain if path == "plain" else ctx.step_batched)(1)
        ref = ws.run(1, contacts=True)
        count = ctx.stats()["contacts"] - before
        assert count == len(ref)
        longest = max(longest, count)
        _state_equal(ctx.download(), ws, 0, n, "%s step %d" % (path, k))
    assert longest > _room(path, n, npairs, threads)
    ctx.close()


@pytest.mark.parametrize("islands", [0, 1])
@pytest.mark.parametrize("path,threads,wave", [("plain", 0, 0), ("batched", 64, 0), ("batched", 128, 0),
                                               ("batched", 256, 0), ("batched", 512, 0), ("batched", 256, 64)])
def test_boxes_and_spheres(oracle_mod, path, threads, wave, islands):
    """More than 48 candidates a wave (the lanes' EPA) in the larger worlds, fewer in the
    smallest (the groups'); spheres only, boxes only, and both."""
    parts = [_mixed(30, 30, 1), _mixed(55, 5, 2), _mixed(3, 57, 3), _mixed(0, 40, 4), _mixed(40, 0, 5), _mixed(4, 3, 6)]
    sc = S.concat(parts)
    sc.params = _params()
    sc.params.fp64_islands = islands
    ctx = runtime.Context(sc.params)
    ctx.upload(sc)
    ctx.set_batched_block(threads)
    ctx.set_wave_worlds(wave)
    states = [oracle_mod.WorldState(sc, w, "f32") for w in range(sc.nworlds)]
    for k in range(3):
        before = ctx.stats()["contacts"]
        (ctx.step_plain if path == "plain" else ctx.step_batched)(1)
        got = ctx.download()
        total = 0
        for w, ws in enumerate(states):
            total += len(ws.run(1, contacts=True))
            _state_equal(got, ws, int(sc.offsets[w]), int(sc.offsets[w + 1]), "step %d world %d" % (k, w))
        assert ctx.stats()["contacts"] - before == total
    st = ctx.stats()
    assert st["epa_overflow"] == 0 and st["capacity_overflow"] == 0
    ctx.close()
    plain = runtime.Context(sc.params)  # its workgroups take few candidates: the groups' EPA throughout
    plain.upload(sc)
    plain.step_plain(3)
    assert st == plain.stats()
    plain.close()
