"""bf16 training pass of the surrogate at the edges of its tiles: one 32 x 32
tile, ragged dimensions, long products (a loading wave beside the computing
one) and 64 x 64 blocks.

Tolerances: operands are rounded to bf16 (2^-9 relative each), so a gradient
built from a chain of four such products is off by a few times 2^-9 of its
norm; 3e-2 is the bound the small-size comparison uses as well.  The planes
the Adam step writes are roundings of the new weights, so an evaluation from
them equals one from planes rebuilt out of the read-back weights exactly.
"""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu
SHAPES = [(31, 64, 64), (64, 64, 128), (2049, 320, 192), (700, 512, 320), (4100, 128, 64)]


def _inputs(D, H, B):
    rng = np.random.default_rng(D + H + B)
    P = dict(W1=rng.normal(size=(H, D)) / np.sqrt(D), b1=0.1 * rng.normal(size=H), W2=rng.normal(size=(H, H)) / np.sqrt(H),
             b2=0.1 * rng.normal(size=H), w3=rng.normal(size=H) / np.sqrt(H), b3=np.float64(0.1))
    return P, rng.normal(size=(B, D)), rng.normal(size=B), rng.normal(size=(B, D))


@pytest.mark.parametrize("D,H,B", SHAPES)
def test_bf16_gradients_at_tile_edges(D, H, B):
    from hmclab_amd.surrogate import Surrogate

    P, X, y, T = _inputs(D, H, B)
    s = Surrogate(D, H)
    s.set_params(P)
    loss, g = s.loss_and_grads(X, y, T)
    lo, go = M.loss_and_grads(P, X, y, T)
    assert abs(loss - lo) <= 3e-2 * abs(lo)
    for k in ("W1", "b1", "W2", "b2", "w3"):
        assert np.linalg.norm(g[k] - go[k]) <= 3e-2 * np.linalg.norm(go[k]), k


@pytest.mark.parametrize("D,H,B", SHAPES)
def test_planes_follow_the_adam_step(D, H, B):
    from hmclab_amd.surrogate import Surrogate

    P, X, y, T = _inputs(D, H, 3 * B)
    s = Surrogate(D, H)
    s.set_params(P)
    s.train(X, y, T, epochs=1, batch=B, learning_rate=1e-2, normalize=False)
    fresh = Surrogate(D, H)
    fresh.set_params(s.get_params())
    f0, g0 = s.evaluate(X[:B])
    f1, g1 = fresh.evaluate(X[:B])
    assert np.array_equal(f0, f1) and np.array_equal(g0, g1)
    assert not np.array_equal(s.get_params()["W1"], np.asarray(P["W1"], dtype=np.float32))
