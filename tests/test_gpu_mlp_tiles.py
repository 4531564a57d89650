"""The network's training kernels at the edges of their tiles (4 or 8 samples
per block, 128 slices of the samples, 16 rounds staged at a time, weights in
LDS or not) against the CPU oracle.  Tolerances as for the other sizes: FP32
sums of a few hundred terms."""
import numpy as np
import pytest

from cgxx_amd import learned
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(37, 128, 128, 13), (5, 64, 65, 1), (3, 193, 130, 70), (63, 256, 256, 64)])
@pytest.mark.parametrize("rows", [1, 3, 5, 127, 129, 1024, 1025, 1033, 2049])
def test_gradient_at_tile_edges(dims, rows):
    from cgxx_amd.cghip import Mlp

    rng = np.random.default_rng(rows)
    p = learned.init_params(dims, 1)
    p += (0.05 * rng.standard_normal(p.size)).astype(np.float32)
    X = rng.standard_normal((rows, dims[0])).astype(np.float32)
    T = rng.standard_normal((rows, dims[3])).astype(np.float32)
    with Mlp(dims, rows) as m:
        m.set_params(p)
        Y = m.forward(X)
        g, loss = m.gradient(X, T)
    _, _, Yr = mo.forward(p, dims, X)
    np.testing.assert_allclose(Y, Yr, rtol=2e-5, atol=2e-5 * np.abs(Yr).max())
    gr, lr = mo.gradient(p, dims, X, T)
    assert loss == pytest.approx(lr, rel=1e-5)
    np.testing.assert_allclose(g, gr, rtol=1e-3, atol=1e-4 * np.abs(gr).max())
