"""Loss and gradient of the warm-start network at the batch sizes where the
training launch changes its blocks and tiles per wave, each after a larger batch
whose partial rows stay in the scratch memory (needs an MI355X).  Against the
FP64 oracle with BF16 operands and by the bars of the existing gradient test;
targets three units off the outputs, so that no sample's error is small."""
import numpy as np
import pytest

import mlp_oracle as M
from vps import Projection, scenes

pytestmark = pytest.mark.gpu

BLOCKS = {"W1": slice(0, 512), "b1": slice(512, 576), "W2": slice(576, 4672),
          "b2": slice(4672, 4736), "W3": slice(4736, 4800), "b3": slice(4800, 4801)}


# 16 samples a tile, 4 waves a block, 256 blocks: 16,384 samples a tile per wave
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 4097, 16383, 16384, 16385, 32769, 49153])
def test_loss_and_gradient(n):
    g = Projection(scenes.small_3d(12, 8, 6))
    p = M.random_params(31).astype(np.float32)
    g.mlp_set_parameters(p)
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, 8)).astype(np.float32)
    t = (rng.normal(size=n) + 3).astype(np.float32)
    g.mlp_loss_and_grad(np.concatenate([X, X + 1]), np.concatenate([t, t]))
    loss, grad = g.mlp_loss_and_grad(X, t)
    lref, gref = M.loss_and_grad(p.astype(np.float64), X.astype(np.float64),
                                 t.astype(np.float64), bf=True)
    assert loss == pytest.approx(lref, rel=5e-3)
    for name, s in BLOCKS.items():
        assert np.linalg.norm(grad[s] - gref[s]) < 2e-2 * np.linalg.norm(gref[s]), name
    again, grad2 = g.mlp_loss_and_grad(X, t)
    assert again == loss and np.array_equal(grad, grad2)
    g.close()
