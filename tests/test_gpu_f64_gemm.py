"""The FP64 GEMM's tiles and k pieces: misfits and gradients at sizes on and off
the tile edges (64, 32 and 16 chains; 128, 64 and 32 rows; one and several k
pieces), both endpoint forms, against NumPy.

Tolerance: an FP64 sum of K products in any order is within K eps of the sum
of their magnitudes; misfit and gradient are sums of at most n + d <= 6200
terms, 6200 eps = 1.4e-12, of magnitudes within a factor of about 10 of the
largest result, so 1e-10 of the largest holds with room.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,B,dtype", [
    (33, 31, 1, np.float64),        # one 32 x 32 tile, ragged
    (64, 64, 16, np.float64),       # exact 64 x 16 tiles
    (700, 301, 17, np.float64),     # 32 x 32
    (2000, 129, 3, np.float32),     # at most 16 chains, long k
    (901, 1531, 100, np.float64),   # 32 x 32 in k pieces
    (1201, 2999, 130, np.float32),  # 64 x 32
    (3100, 3100, 257, np.float64),  # 64 x 64 and 128 x 64, ragged in every direction
    (2048, 4096, 512, np.float64),  # exact 64 x 64 tiles
])
@pytest.mark.parametrize("premult", [0, 1])
def test_f64_gemm_tiles(n, d, B, dtype, premult):
    from hmclab_amd._lib import PRIOR_NORMAL
    from hmclab_amd.engine import Problem

    rng = np.random.default_rng(n + d + B)
    G = rng.normal(size=(n, d)).astype(dtype)
    data, var = rng.normal(size=n), rng.uniform(0.5, 2.0, size=n)
    X = rng.normal(size=(B, d))
    p = Problem(d, precision="f64", engine="gemm")
    p.set_option("endpoint_premult", premult)
    p.set_dense(G, data, var)
    p.add_prior(PRIOR_NORMAL, np.zeros(d), np.ones(d))
    r = X @ G.astype(np.float64).T - data
    chi = 0.5 * np.sum(r * r / var, axis=1) + 0.5 * np.sum(X * X, axis=1)
    grad = (r / var) @ G.astype(np.float64) + X
    got = p.misfit_batch(X)
    assert np.max(np.abs(got - chi)) <= 1e-10 * np.max(np.abs(chi))
    got = p.gradient_batch(X)
    assert np.max(np.abs(got - grad)) <= 1e-10 * np.max(np.abs(grad))
    p.close()
