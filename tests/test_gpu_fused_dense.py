"""Small dense float64 targets on the fused engine (several proposals per
launch): the same seeded chains on the GEMM engine, and the same proposals one
launch at a time, at sizes on and off the row slices (64), the parts of a row
over the waves, the columns of H a thread may hold (8, 16, 32), and past the
largest size that takes this path (192 parameters).

Tolerance: both engines sum in float64, in different orders; a proposal is at
most 5 stages whose rounding (about (n + d) eps, 1e-13 relative) grows with
the condition of the trajectory, here a short one (eps sqrt(lambda) < 1): 1e-9
of the largest magnitude holds with room for 6 proposals.  One launch for all
proposals and one each run the same code on the same numbers: equal bits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(n, d, B, engine, premult, calls, tiles=-1, trace=0, thinning=1, tune=False):
    from hmclab_amd._lib import PRIOR_NORMAL
    from hmclab_amd.engine import Chains, Problem

    rng = np.random.default_rng(1000 * n + d)
    p = Problem(d, precision="f64", engine=engine)
    if engine == "fused":
        p.set_option("premult_trajectory", premult)
    if tiles > 0:
        p.set_option("fused_tile_chains", tiles)
    if n:
        p.set_dense(rng.normal(size=(n, d)) / np.sqrt(n + d), rng.normal(size=n), rng.uniform(0.5, 2.0, size=n))
    p.add_prior(PRIOR_NORMAL, rng.normal(size=d), rng.uniform(0.5, 2.0, size=d))
    ch = Chains(p, B)
    ch.set_state(rng.normal(size=(B, d)))
    if trace:
        ch.set_trace(trace)
    if tune:
        ch.set_tuning_history(sum(calls))
    step, accepted, k = np.full(B, 0.3), np.zeros(B, dtype=np.int64), 0
    for m in calls:
        step, acc = ch.run(m, 5, step, autotune=tune, seed=11, first_proposal=k, thinning=thinning)
        accepted += acc
        k += m
    res = [*ch.get_state(), step, accepted]
    rng = np.random.default_rng(7)   # one proposal from given momenta: end state and energies
    prop = ch.propose(rng.normal(size=(B, d)), np.full(B, 0.3), np.zeros(B), 5, trajectory=True)
    res += [prop[key] for key in ("X1", "P1", "H0", "H1")]
    if trace:
        res += ch.read_trace(0, ch.trace_count())
    if tune:
        res += ch.tuning_history()
    p.close()
    return res


@pytest.mark.parametrize("n,d,B,premult", [
    (5, 1, 1, 1),         # one parameter, one wave of eight with work
    (40, 63, 3, 0),       # a slice short of a wave
    (70, 64, 5, 1),       # 8 columns of H per part
    (100, 65, 300, 1),    # two slices, 32 columns, two chains per workgroup
    (129, 65, 2, 0),      # odd rows of both products
    (30, 128, 2, -1),     # n < d: residual form
    (200, 129, 257, -1),  # three slices, H from memory, a lone last chain
    (150, 192, 2, 0),     # the largest of this path
    (150, 193, 2, 1),     # past it
    (0, 20, 4, -1),       # no data
])
def test_fused_dense_sizes(n, d, B, premult):
    one = _run(n, d, B, "fused", premult, [6])
    each = _run(n, d, B, "fused", premult, [1] * 6)
    for a, b in zip(one, each):
        assert np.array_equal(a, b)
    want = _run(n, d, B, "gemm", premult, [6])
    assert np.array_equal(one[3], want[3])
    for a, b in zip(one, want):
        assert np.max(np.abs(a - b)) <= 1e-9 * max(np.max(np.abs(b)), 1.0)


@pytest.mark.parametrize("tiles", [1, 2])
def test_fused_dense_trace_and_tuning(tiles):
    """Thinned traces and tuning histories over several launches."""
    kw = dict(tiles=tiles, trace=4, thinning=3, tune=True)
    one = _run(90, 70, 5, "fused", 1, [10], **kw)
    parts = _run(90, 70, 5, "fused", 1, [4, 1, 5], **kw)
    assert one[8].shape == (4, 5, 70) and one[10].shape == (10, 5)
    for a, b in zip(one, parts):
        assert np.array_equal(a, b)
    want = _run(90, 70, 5, "gemm", 1, [10], trace=4, thinning=3, tune=True)
    for a, b in zip(one, want):
        assert np.max(np.abs(a - b)) <= 1e-9 * max(np.max(np.abs(b)), 1.0)


def test_fused_dense_trace_capacity():
    """A trace that runs full: the proposals before are done, the call fails."""
    from hmclab_amd._lib import PRIOR_NORMAL
    from hmclab_amd.engine import Chains, Problem

    p = Problem(10, precision="f64", engine="fused")
    p.add_prior(PRIOR_NORMAL, np.zeros(10), np.ones(10))
    ch = Chains(p, 2)
    ch.set_state(np.zeros((2, 10)))
    ch.set_trace(3)
    with pytest.raises(Exception, match="trace capacity"):
        ch.run(5, 5, 0.3, seed=1)
    assert ch.trace_count() == 3
    X, chi = ch.read_trace(0, 3)
    assert np.allclose(X[2], ch.get_state()[0], rtol=0, atol=0)
    p.close()


@pytest.mark.parametrize("B", [1, 256, 257, 512, 513])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_fused_tile_rule(B, precision):
    """The chains per workgroup that the number of chains picks, on a sparse and
    a dense operator: equal bits with one chain per workgroup."""
    import scipy.sparse as sp
    from hmclab_amd._lib import PRIOR_NORMAL
    from hmclab_amd.engine import Chains, Problem

    n, d = 75, 210
    rng = np.random.default_rng(B)
    G = rng.normal(size=(n, d)) / np.sqrt(n) * (rng.uniform(size=(n, d)) < 0.2)
    x0 = rng.normal(size=(B, d))
    for setter in (lambda p: p.set_csr(sp.csr_matrix(G), np.ones(n), 0.5), lambda p: p.set_dense(G, np.ones(n), 0.5)):
        out = []
        for tiles in (0, 1):
            p = Problem(d, precision=precision, engine="fused")
            p.set_option("fused_tile_chains", tiles)
            setter(p)
            p.add_prior(PRIOR_NORMAL, np.zeros(d), np.ones(d))
            ch = Chains(p, B)
            ch.set_state(x0)
            step, acc = ch.run(3, 4, 0.2, seed=5)
            out.append((*ch.get_state(), acc))
            p.close()
        assert out[0][2].sum() > 0
        for a, b in zip(*out):
            assert np.array_equal(a, b)
