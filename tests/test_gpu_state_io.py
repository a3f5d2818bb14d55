"""State in and out: set_state / get_state return every array exactly, at body counts around the
256-body blocks of the transfer kernels, for every choice of arrays set."""
import time

import numpy as np
import pytest

from nphysics_amd import abi, scenes

pytestmark = pytest.mark.gpu

KEYS = ("pos", "rot", "linvel", "angvel")


@pytest.mark.parametrize("n", [1, 2, 63, 255, 256, 257, 511, 1021])
def test_state_round_trip(nphys, n):
    s = scenes.boxes(nx=n, ny=1, nz=1)  # a static ground and n cuboids
    w = nphys.MechanicalWorld(integration_parameters=abi.default_params())
    w.add_bodies(s)
    want = w.get_state()
    for k in KEYS:
        np.testing.assert_array_equal(want[k], s[k].astype(np.float32), err_msg=k)
    rng = np.random.default_rng(n)
    for mask in (15, 1, 2, 4, 8, 5, 10):
        new = {k: rng.normal(size=want[k].shape).astype(np.float32) for i, k in enumerate(KEYS) if mask >> i & 1}
        w.set_state(**new)
        for k, v in new.items():
            want[k] = v.copy()
            if k in ("linvel", "angvel"):
                want[k][0] = 0.0  # the static ground keeps no velocity
        got = w.get_state()
        for k in KEYS:
            np.testing.assert_array_equal(got[k], want[k], err_msg=f"{k} after mask {mask}")
    # the bodies of a second insertion keep the first ones' state
    w.add_bodies({k: v[1:] for k, v in s.items()})
    got = w.get_state()
    for k in KEYS:
        np.testing.assert_array_equal(got[k][: n + 1], want[k], err_msg=k)
        np.testing.assert_array_equal(got[k][n + 1:], s[k][1:].astype(np.float32), err_msg=k)


def test_reads_of_a_filling_scene(nphys):
    """Contacts and pairs read at every call while their number grows by one in a hundred: all of them, and without
    a new staging buffer at each call (which took eight times as long as a read does: the median read is within
    three times that of a scene that stays)."""
    n = 27000
    s = scenes._empty(n)
    s["dims"][:, 0] = 0.15
    i = np.arange(n)
    s["pos"][:] = np.stack([0.3 * (i % 30), 0.3 * (i // 900), 0.3 * (i // 30 % 30)], 1)
    w = nphys.MechanicalWorld(integration_parameters=abi.default_params(gravity=(0.0, 0.0, 0.0)))
    w.add_bodies(s)

    def timed_reads(filled):
        pos = s["pos"].copy()
        pos[filled:, 1] += 5.0 * (4 + np.arange(n - filled))
        w.set_state(pos=pos)
        w.collide()
        t = time.perf_counter()
        contacts, pairs = w.contacts(), w.pairs()
        t = time.perf_counter() - t
        a, b = contacts["bodies"].min(1), contacts["bodies"].max(1)
        assert np.isin(b - a, (1, 30, 900)).all() and contacts["depth"].shape[0] <= pairs.shape[0]
        np.testing.assert_allclose(np.linalg.norm(contacts["normal"], axis=1), 1.0, rtol=1e-5)
        return t, contacts["depth"].shape[0]

    grows = [timed_reads(14000 + 150 * k) for k in range(20)]
    stays = [timed_reads(14000 + 150 * 19) for _ in range(20)]
    counts = [c for _, c in grows]
    assert all(a < b for a, b in zip(counts, counts[1:])) and counts[0] > 40000
    assert np.median([t for t, _ in grows]) < 3.0 * np.median([t for t, _ in stays])
