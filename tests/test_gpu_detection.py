"""The pair searches against the CPU restatement's pairs, contacts and manifolds: body counts around
its 64-collider chunks, statics anywhere in the body order, scenes interleaved in the body order,
collision groups, segments that overflow, calm steps (kept segments) and the size at which worlds go over
to the search by boxes."""
import numpy as np
import pytest

from nphysics_amd import abi, scenes

pytestmark = pytest.mark.gpu


def _shuffled(n, seed, nscenes=1, statics=0.1, groups=False, spacing=0.9):
    """n balls and cuboids on a jittered lattice in random body order, a share of them static."""
    rng = np.random.default_rng(seed)
    s = scenes._empty(n)
    side = int(np.ceil(n ** (1 / 3)))
    k = rng.permutation(n)
    c = np.stack([k % side, k // side % side, k // (side * side)], 1) * spacing
    s["pos"][:] = c + rng.uniform(-0.2, 0.2, (n, 3))
    ball = rng.random(n) < 0.5
    s["shape"][:] = np.where(ball, 0, 1)
    s["dims"][:] = np.where(ball[:, None], np.stack([rng.uniform(0.2, 0.5, n), np.zeros(n), np.zeros(n)], 1),
                            rng.uniform(0.15, 0.4, (n, 3)))
    s["status"][:] = (rng.random(n) < statics).astype(np.int32)
    s["status"][0] = 0
    s["linvel"][:] = np.where(s["status"][:, None] == 0, rng.uniform(-0.5, 0.5, (n, 3)), 0.0)
    if nscenes > 1:
        s["scene"] = rng.integers(0, nscenes, n).astype(np.int32)
    if groups:
        s["collision_groups"] = np.array([abi.collision_groups(membership=[int(g)], whitelist=[0, int(g)])
                                          for g in rng.integers(0, 3, n)], np.uint32)
    return s


def _same(g, o, what):
    np.testing.assert_array_equal(g.pairs(), o.pairs(), err_msg=what)
    gc, oc = g.contacts(), o.contacts()
    np.testing.assert_array_equal(gc["bodies"], oc["bodies"], err_msg=what)
    np.testing.assert_array_equal(gc["depth"], np.asarray(oc["depth"]).astype(np.float32), err_msg=what)
    gm, om = g.manifolds(), o.manifolds()
    for k in ("bodies", "first", "count"):
        np.testing.assert_array_equal(gm[k], om[k], err_msg=what)


def _worlds(nphys, oracle_mod, s):
    p = dict(gravity=(0.0, 0.0, 0.0))
    g = nphys.MechanicalWorld(integration_parameters=abi.default_params(**p))
    o = oracle_mod.OracleWorld(abi.default_params(**p), precision=32, order=oracle_mod.ORDER_COLOURED)
    g.add_bodies(s)
    o.add_bodies(s)
    return g, o


@pytest.mark.parametrize("n,nscenes,groups", [(2, 1, False), (63, 1, False), (64, 1, True), (65, 1, False),
                                              (130, 1, False), (257, 5, False), (700, 3, True), (1500, 1, True),
                                              (1999, 40, True)])
def test_pairs_match_the_restatement(nphys, oracle_mod, n, nscenes, groups):
    s = _shuffled(n, n, nscenes, groups=groups)
    g, o = _worlds(nphys, oracle_mod, s)
    for k in range(4):
        g.step(1)
        o.step(1)
        _same(g, o, f"step {k + 1}")
    rng = np.random.default_rng(1)
    pos = s["pos"].copy()
    for k in range(4):  # few bodies moved: calm detections; then all of them
        few = rng.choice(n, max(1, n // 20) if k < 3 else n, replace=False)
        few = few[s["status"][few] == 0] if k % 2 else few  # with and without statics among them
        pos[few] += rng.uniform(-0.3, 0.3, (len(few), 3)).astype(np.float32)
        g.set_state(pos=pos)
        o.set_state(pos=pos)
        g.collide()
        o.collide()
        _same(g, o, f"move {k}")


def test_segment_overflow(nphys, oracle_mod):
    """300 small balls around body 0: its segment of 32 partners grows to hold them, in one detection,
    also after bodies came and went."""
    n = 301
    s = scenes._empty(n)
    s["dims"][:, 0] = 0.05
    rng = np.random.default_rng(5)
    d = rng.normal(size=(n, 3))
    s["pos"][:] = 3.02 * d / np.linalg.norm(d, axis=1, keepdims=True)
    s["pos"][0] = 0.0
    s["dims"][0, 0] = 3.0
    g, o = _worlds(nphys, oracle_mod, s)
    for far in (0.0, 10.0, 0.0):
        pos = s["pos"].copy()
        pos[1:] *= 1.0 + far
        g.set_state(pos=pos)
        o.set_state(pos=pos)
        g.collide()
        o.collide()
        _same(g, o, f"far {far}")
        assert (g.pairs()[:, 0] == 0).sum() == (300 if far == 0.0 else 0)


@pytest.mark.parametrize("n", [128, 129, 200, 400])
def test_crowd(nphys, oracle_mod, n):
    """Every body overlaps every other: n (n - 1) / 2 pairs, at and above the 8,192 pairs that a tile of the
    compaction sorts by kind in one go."""
    s = _shuffled(n, n, statics=0.0)
    s["pos"][:] = np.random.default_rng(n).uniform(-0.02, 0.02, (n, 3))
    g, o = _worlds(nphys, oracle_mod, s)
    g.collide()
    o.collide()
    _same(g, o, f"{n} bodies")
    assert g.pairs().shape[0] == n * (n - 1) // 2


@pytest.mark.parametrize("n,nscenes,groups", [(2047, 1, False), (2048, 1, True), (2049, 1, True), (4096, 1, False),
                                              (4097, 1, False), (9001, 1, True), (9001, 7, False)])
def test_search_by_boxes(nphys, oracle_mod, n, nscenes, groups):
    """Around the size at which a world goes over to the search by boxes, and with one and two levels of
    them; the order of the boxes ages over the steps."""
    s = _shuffled(n, 3, nscenes, groups=groups, spacing=1.0)
    g, o = _worlds(nphys, oracle_mod, s)
    for k in range(4):
        g.step(1)
        o.step(1)
        _same(g, o, f"{n} bodies, step {k + 1}")


@pytest.mark.parametrize("n", [40, 257, 300])
def test_crowd_steps(nphys, oracle_mod, n):
    """Steps of a crowd whose bodies all touch each other: n - 1 manifolds per body, so at least as many
    colours, below and above the 256 that the colour order is built for at first, and classes of a few manifolds."""
    s = _shuffled(n, n, statics=0.0)
    s["pos"][:] = np.random.default_rng(n).uniform(-0.02, 0.02, (n, 3))
    g, o = _worlds(nphys, oracle_mod, s)
    for k in range(2):
        g.step(1)
        o.step(1)
        gs, os_ = g.get_state(), o.get_state()
        for key in ("pos", "rot", "linvel", "angvel"):
            np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=f"{key}, step {k + 1}")
    assert g.counters()["ncolours"] >= (n - 1 if n < 257 else 257)


def _sliding(n, ccd):
    """Balls and cuboids on a ground without friction, a third of them sliding at 1 mm a step: their loose AABBs,
    10 mm wider, are replaced every tenth step or so, and from the thirtieth step on bodies come near each other."""
    s = scenes.boxes(nx=n, ny=1, nz=1)
    i = np.arange(n)
    side = int(np.ceil(np.sqrt(n)))
    ball = i % 2 == 0
    s["rot"][1:] = (0.0, 0.0, 0.0, 1.0)
    s["shape"][1:] = np.where(ball, 0, 1)
    s["dims"][1:] = np.where(ball[:, None], [0.5, 0.0, 0.0], [0.4, 0.5, 0.5])
    s["pos"][1:] = np.stack([1.3 * (i % side) - 0.65 * side, np.full(n, 0.519), 1.07 * (i // side) - 0.535 * side], 1)
    s["dims"][0] = (3.0 * side, 0.5, 3.0 * side)
    s["friction"][:] = 0.0
    s["linvel"][1:] = s["angvel"][1:] = 0.0
    s["linvel"][1:, 2] = np.where(np.random.default_rng(n).random(n) < 0.3, 0.06, 0.0)
    if ccd:
        s["ccd_enabled"] = (np.arange(n + 1) % 10 == 5).astype(np.int32)
    return s


@pytest.mark.parametrize("ccd", [False, True])
@pytest.mark.parametrize("n", [65, 700, 2100])
def test_calm_steps(nphys, oracle_mod, n, ccd):
    """Most detections replace no loose AABB and keep the pairs and their lists by kind; those that follow
    and do replace some begin as if they did not."""
    s = _sliding(n, ccd)
    g = nphys.MechanicalWorld(integration_parameters=abi.default_params())
    o = oracle_mod.OracleWorld(abi.default_params(), precision=32, order=oracle_mod.ORDER_COLOURED)
    for w in (g, o):
        w.add_bodies(s)
    steps = ""
    for k in range(40):
        before = g.counters()["pair_rebuilds"]
        for w in (g, o):
            w.step(1)
        steps += "x" if g.counters()["pair_rebuilds"] > before else "."
        _same(g, o, f"step {k + 1}")
        gs, os_ = g.get_state(), o.get_state()
        for key in ("pos", "rot", "linvel", "angvel"):
            np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=f"{key}, step {k + 1}")
    assert steps.count("......") >= 3 and steps.count("...x") >= 3, steps


@pytest.mark.parametrize("n", [65, 2100])
def test_calm_queries(nphys, oracle_mod, n):
    """Collision queries that move the bodies by less than their margins, and then one that moves static ones
    (alone) further: after the calm ones it begins as one of them."""
    s = _shuffled(n, n, statics=0.3)
    g, o = _worlds(nphys, oracle_mod, s)
    rng = np.random.default_rng(n)
    static = s["status"] == 1
    pos = s["pos"].copy()
    for far in (0.0, 0.0, 0.0, 0.0, 0.3, 0.0, 0.0, 0.0, 0.0):
        query = pos + rng.uniform(-2e-4, 2e-4, (n, 3)).astype(np.float32)
        if far:
            pos[static] += rng.uniform(-far, far, (int(static.sum()), 3)).astype(np.float32)
            query[static] = pos[static]
        for w in (g, o):
            w.set_state(pos=query)
            w.collide()
        _same(g, o, f"far {far}")
