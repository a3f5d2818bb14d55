"""Calls that fail and the calls after them on the same world: what a failed call leaves readable is
whole, and the next call that can succeed gives what it gives in a world that never failed. A small limit
on the pairs of the narrow phase stands for the 2^26 - 1 that it takes."""
import numpy as np
import pytest

from nphysics_amd import abi, scenes
from tests.test_gpu_detection import _same, _shuffled, _worlds

pytestmark = pytest.mark.gpu

KEYS = ("pos", "rot", "linvel", "angvel")
MOST = (1 << 26) - 1


def _limit(nphys, w, pairs):
    assert nphys.load_library().nphys_test_most_pairs(w._h, pairs) == 0


def _refused(nphys, call):
    with pytest.raises(nphys.NphysError, match="too many broad-phase pairs"):
        call()


def _same_state(g, o, what):
    gs, os_ = g.get_state(), o.get_state()
    for key in KEYS:
        np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=f"{key}, {what}")


@pytest.mark.parametrize("n,known", [(60, True), (60, False), (400, True), (2100, True), (2100, False)])
def test_more_pairs_than_the_narrow_phase_takes(nphys, oracle_mod, n, known):
    """A crowd with more pairs than the limit, refused by the world's first detection or by a later one (whose
    buffers the last list fits): the pairs are all there, no contacts are, and bodies moved apart are detected again."""
    s = _shuffled(n, n, statics=0.0, spacing=0.3)
    g, o = _worlds(nphys, oracle_mod, s)
    o.collide()
    pairs = o.pairs()
    apart = s["pos"] * 10.0
    if known:
        g.collide()
        _same(g, o, "before")
    _limit(nphys, g, pairs.shape[0] - 1)
    for call in (g.collide, g.collide, lambda: g.step(1)):
        _refused(nphys, call)
        np.testing.assert_array_equal(g.pairs(), pairs)
        assert g.contacts()["depth"].shape[0] == 0 and g.manifolds()["count"].shape[0] == 0
    _same_state(g, o, "refused")
    for w in (g, o):
        w.set_state(pos=apart)
        w.collide()
    _same(g, o, "apart")
    _limit(nphys, g, MOST)
    for w in (g, o):
        w.set_state(pos=s["pos"])
    for k in range(2):
        for w in (g, o):
            w.step(1)
        _same(g, o, f"step {k + 1}")
        _same_state(g, o, f"step {k + 1}")


def test_step_refused_at_its_end(nphys, oracle_mod):
    """The detection that ends a step fails: the step after it begins with another one, and has the contacts."""
    s = scenes._empty(20)
    s["dims"][:, 0] = 0.5
    i = np.arange(20)
    s["pos"][:] = np.stack([1.5 * (i % 2), np.zeros(20), 4.0 * (i // 2)], 1)
    s["linvel"][:, 0] = np.where(i % 2 == 0, 20.0, -20.0)
    g, o = _worlds(nphys, oracle_mod, s)
    _limit(nphys, g, 1)
    _refused(nphys, lambda: g.step(1))
    o.step(1)
    _same_state(g, o, "first step")
    np.testing.assert_array_equal(g.pairs(), o.pairs())
    assert g.pairs().shape[0] == 10
    _limit(nphys, g, MOST)
    for k in range(3):
        g.step(1)
        o.step(1)
        _same(g, o, f"step {k + 2}")
        _same_state(g, o, f"step {k + 2}")
