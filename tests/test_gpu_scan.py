"""Prefix sums across tiles: pair lists and manifolds of scenes whose body, pair and manifold counts
stand at and around the scan's 2,048-word tiles and its 64-tile look-back window (and above the
262,144 colliders of 64 upper boxes), against the sorted
brute-force pair set of a line of touching balls."""
import numpy as np
import pytest

from nphysics_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 2047, 2048, 2049, 4097, 131071, 131072, 133121, 266305])
def test_line_of_balls(nphys, n):
    # ball k touches k-1 and k+1 only (0.3 m apart, radius 0.15; the next neighbour is 0.3 m away)
    s = scenes._empty(n)
    s["dims"][:, 0] = 0.15
    row, col = np.arange(n) // 512, np.arange(n) % 512
    col = np.where(row % 2 == 0, col, 511 - col)  # rows by turns, so that k and k+1 are neighbours
    s["pos"][:] = np.stack([0.3 * col, np.zeros(n), 2.0 * row], 1)
    w = nphys.MechanicalWorld(integration_parameters=abi.default_params(gravity=(0.0, 0.0, 0.0)))
    w.add_bodies(s)
    k = np.arange(n - 1)
    k = k[row[:-1] == row[1:]]
    want = np.stack([k, k + 1], 1)
    for _ in range(3):  # the scan state is reused from one call to the next
        w.collide()
        np.testing.assert_array_equal(w.pairs(), want)
        m = w.manifolds()
        np.testing.assert_array_equal(m["bodies"], want)
        np.testing.assert_array_equal(m["first"], np.arange(len(k)))
        assert w.contacts()["depth"].shape[0] == len(k)
