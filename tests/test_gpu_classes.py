"""Colour classes at the edges of the launches that solve them: classes list the manifolds with several
contacts first (eight lanes each in a sweep, a quad in the position correction), then those with one (two
lanes, one lane), and classes of up to 1,024 lanes share a workgroup."""
import numpy as np
import pytest

from nphysics_amd import abi, scenes

pytestmark = pytest.mark.gpu


def _resting(nboxes, nballs, chain=False):
    """Boxes and balls apart from each other, a little inside the ground: one class of
    nboxes four-contact and nballs one-contact manifolds. chain: the last ball in a row with two more above the
    ground instead (with nballs 0, three balls more), which gives the class one of their two manifolds and a second class the other."""
    if chain:
        nballs = max(nballs - 1, 0) + 3
    n = nboxes + nballs
    side = int(np.ceil(np.sqrt(n)))
    s = scenes.boxes(nx=n, ny=1, nz=1)  # and the ground
    s["rot"][1:] = (0.0, 0.0, 0.0, 1.0)
    s["shape"][1 + nboxes:] = 0
    s["dims"][1 + nboxes:] = (0.5, 0.0, 0.0)
    i = np.arange(n)
    rng = np.random.default_rng(n)
    s["pos"][1:, 0] = 1.7 * (i % side) - 0.85 * side
    s["pos"][1:, 1] = 0.5 - rng.uniform(0.005, 0.03, n)
    s["pos"][1:, 2] = 1.7 * (i // side) - 0.85 * side
    s["linvel"][1:] = rng.uniform(-1.0, 1.0, (n, 3))
    s["angvel"][1:] = rng.uniform(-1.0, 1.0, (n, 3))
    if chain:
        s["pos"][-3:] = [(0.99 * k, 20.0, 0.0) for k in range(3)]
        s["linvel"][-3:] = 0.0
    return s


@pytest.mark.parametrize("variant", [0, 256, 512, 1024])
@pytest.mark.parametrize("nboxes,nballs", [(1, 0), (0, 1), (1, 1), (15, 33), (32, 129), (127, 4), (127, 5), (128, 0),
                                           (129, 0), (0, 512), (0, 513), (300, 700)])
def test_class_sizes(nphys, oracle_mod, nboxes, nballs, variant):
    s = _resting(nboxes, nballs, chain=variant > 0)  # the blocked variants are for two colours and more
    g = nphys.MechanicalWorld(integration_parameters=abi.default_params())
    o = oracle_mod.OracleWorld(abi.default_params(), precision=32, order=oracle_mod.ORDER_COLOURED)
    for w in (g, o):
        w.add_bodies(s)
    g.set_sweep_variant(variant)
    for k in range(3):
        g.step(1)
        o.step(1)
        gs, os_ = g.get_state(), o.get_state()
        for key in ("pos", "rot", "linvel", "angvel"):
            np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=f"{key}, step {k + 1}")
        assert g.counters()["ncolours"] == (2 if variant else 1)
        assert g.counters()["sweep_variant"] == variant


@pytest.mark.parametrize("crowd", [256, 300])
def test_many_colours_in_many_scenes(nphys, oracle_mod, crowd):
    """As many scenes as there can be, all but one of them empty, and in that one a crowd of as many colours as
    bodies: the blocked launches hold a class's place for each."""
    s = scenes._empty(crowd)
    s["dims"][:, 0] = 0.3
    s["pos"][:] = np.random.default_rng(crowd).uniform(-0.02, 0.02, (crowd, 3))
    s["scene"] = np.full(crowd, 32767, np.int32)
    g = nphys.MechanicalWorld(integration_parameters=abi.default_params())
    o = oracle_mod.OracleWorld(abi.default_params(), precision=32, order=oracle_mod.ORDER_COLOURED)
    for w in (g, o):
        w.add_bodies(s)
    g.set_sweep_variant(256)
    for k in range(2):
        for w in (g, o):
            w.step(1)
        gs, os_ = g.get_state(), o.get_state()
        for key in ("pos", "rot", "linvel", "angvel"):
            np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=f"{key}, step {k + 1}")
    assert crowd - 1 <= g.counters()["ncolours"] <= 511
    assert g.counters()["sweep_variant"] == 256


def _same_steps(nphys, oracle_mod, s, steps):
    g = nphys.MechanicalWorld(integration_parameters=abi.default_params())
    o = oracle_mod.OracleWorld(abi.default_params(), precision=32, order=oracle_mod.ORDER_COLOURED)
    for w in (g, o):
        w.add_bodies(s)
    for k in range(steps):
        g.step(1)
        o.step(1)
        gs, os_ = g.get_state(), o.get_state()
        for key in ("pos", "rot", "linvel", "angvel"):
            np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=f"{key}, step {k + 1}")
    return g.counters()


@pytest.mark.parametrize("nballs,above", [(1023, 0), (1024, 0), (1025, 0), (2047, 0), (2048, 0), (2049, 0), (100, 3995),
                                          (100, 3996)])
def test_colouring_edges(nphys, oracle_mod, nballs, above):
    """Up to 2,048 manifolds among 4,096 bodies one workgroup colours and orders them: the last sizes it takes
    and the first it does not, with `above` bodies that touch nothing."""
    s = _resting(0, nballs + above)
    s["pos"][1 + nballs:, 1] += 20.0
    _same_steps(nphys, oracle_mod, s, 2)


@pytest.mark.parametrize("grid", [(6, 6, 6), (9, 8, 9), (9, 9, 9), (10, 9, 9), (12, 9, 9)])
def test_colouring_of_stacks(nphys, oracle_mod, grid):
    """Cuboids inside their neighbours: some 600 to 2,700 manifolds of several colours, on both sides of the
    2,048 that one workgroup colours."""
    nx, ny, nz = grid
    _same_steps(nphys, oracle_mod, scenes.boxes(nx=nx, ny=ny, nz=nz, spacing=0.995), 3)
