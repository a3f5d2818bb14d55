"""Weight gradients at the edges of their kernels' tiles: 16 rows a wave and 64 a workgroup in the pass, 32 rows a
stage and 256 a workgroup in the products, 16 partial sums read ahead. The tolerance is the BF16 level of
test_mlp.py: 2% in norm, and 3% in each group of parameters."""
import numpy as np
import pytest

from tests.test_mlp import random_params, random_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 17, 31, 33, 64, 65, 255, 257, 4096 + 33])
def test_gradients_of_ragged_batches(nphys, oracle_mod, n):
    from nphysics_amd import learned

    rng = np.random.default_rng(n)
    p = random_params(rng)
    net = learned.WarmStartNet(seed=5)
    net.params = p.astype(np.float32)
    X, T = random_rows(rng, p, n)
    g, loss = net.gradients(X, T)
    gr, lr = oracle_mod.mlp_gradients(net.params.astype(np.float64), X, T, emulate_bf16=True)
    assert loss == pytest.approx(lr, rel=2e-3)
    assert np.linalg.norm(g - gr) < 0.02 * np.linalg.norm(gr)
    for a, b in ((0, 3072), (3072, 3200), (3200, 19584), (19584, 19712), (19712, 20096), (20096, 20099)):
        assert np.linalg.norm(g[a:b] - gr[a:b]) <= 0.03 * np.linalg.norm(gr[a:b]) + 1e-7, (a, b)
    net.close()
