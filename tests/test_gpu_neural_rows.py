"""The training step's sums over gradient rows (one per 64 samples, sixteen runs of
them, eight reads at a time): one row, a partial one, runs of 7, 8 and 9 rows and the
most a batch has, against the float64 oracle with the bound of the other gradient test
(float32 accumulation, 1e-4 of the layer's largest)."""
import numpy as np
import pytest

from oracle import nn
from test_gpu_neural import _lighting

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('batch', [33, 64, 65, 112 * 64, 113 * 64 - 5, 128 * 64, 129 * 64, 256 * 64])
def test_gradient_rows(gpu, batch):
    from taichi_three_amd.neural import NeuralShading
    print(f'case: gradient of {batch} samples', flush=True)
    ns = NeuralShading(_lighting(), seed=5)
    X, Y = ns.samples(batch, seed=13)
    g = ns.gradient(X, Y).cpu().numpy().astype(np.float64)
    ref = nn.backward(ns.params.cpu().numpy().astype(np.float64), X.cpu().numpy().astype(np.float64),
                      Y.cpu().numpy().astype(np.float64))
    for name, shape, off in nn.layout():
        a, b = g[off:off + int(np.prod(shape))], ref[off:off + int(np.prod(shape))]
        assert np.abs(a - b).max() <= 1e-4 * (np.abs(b).max() + 1e-12), name
