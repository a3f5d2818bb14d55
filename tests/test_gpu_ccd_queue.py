"""The impact queue where its slots fill more than one wave per group: above 262,144 CCD pairs a group
of the queue holds 128 slots or more."""
import numpy as np
import pytest

from nphysics_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num", [4, 9])
def test_cloud_of_swept_pairs(nphys, oracle_mod, num):
    """num^3 small balls and cuboids in one cloud: their swept boxes all overlap, so every pair has a slot
    (2,016 and 265,356 of the dynamic ones), and their relative velocities make a part of them hit."""
    s = scenes.ccd_room(num=num, rad=0.008, velocity=(90.0, 90.0, 90.0), height=-0.1, seed=num)
    rng = np.random.default_rng(num)
    s["linvel"][6:] += rng.uniform(-3.0, 3.0, (num ** 3, 3))
    s["angvel"][6:] = rng.uniform(-5.0, 5.0, (num ** 3, 3))
    g = nphys.MechanicalWorld(integration_parameters=abi.default_params())
    o = oracle_mod.OracleWorld(abi.default_params(), precision=32, order=oracle_mod.ORDER_COLOURED)
    for w in (g, o):
        w.add_bodies(s)
        w.step(1)
    gs, os_ = g.get_state(), o.get_state()
    for key in ("pos", "rot", "linvel", "angvel"):
        np.testing.assert_array_equal(gs[key], np.asarray(os_[key]).astype(np.float32), err_msg=key)
    assert g.counters()["npairs"] >= num ** 3 * (num ** 3 - 1) // 2
    assert g.counters()["ccd_impacts"] > 0
