"""State in and out: set_state / get_state return every array exactly, at body counts around the
256-body blocks of the transfer kernels, for every choice of arrays set."""
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
