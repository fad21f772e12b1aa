"""The neighbor searches with one query a wavefront, at strips of less than,
exactly and just over 64 points, at the longest lists, and on both sides of the
number of queries where nn2 changes kernels: bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(2, 1), (63, 62), (64, 15), (65, 63),
                                 (129, 5), (1500, 63), (4097, 16)])
@pytest.mark.parametrize("ordered", [True, False])
def test_predecessors_bit_exact(oracle, nngp, n, m, ordered):
    print(f"knn wave n={n} m={m} ordered={ordered}", flush=True)
    rng = np.random.default_rng(n + m)
    c = rng.uniform(size=(n, 2))
    if ordered:
        c = c[np.argsort(c[:, 0], kind="stable")]
    for got, want in ((nngp.mkNNIndxCB(c, m), oracle.mkNNIndxCB(c, m)),
                      (nngp.mkNNIndx(c, m), oracle.mkNNIndx(c, m))):
        for key in ("nnIndx", "nnIndxLU", "nnDist"):
            assert np.array_equal(got[key], want[key]), key


@pytest.mark.parametrize("n,k,q", [(1, 1, 3), (64, 64, 5), (65, 64, 70),
                                   (3000, 17, 400), (3000, 15, 49152),
                                   (3000, 15, 49153)])
def test_nn2_bit_exact(oracle, nngp, n, k, q):
    print(f"nn2 wave n={n} k={k} q={q}", flush=True)
    rng = np.random.default_rng(n + k)
    c = rng.uniform(size=(n, 2))
    c0 = rng.uniform(-0.2, 1.2, size=(q, 2))  # some outside every strip
    i_ref, d_ref = oracle.nn2(c, c0, k)
    i_got, d_got = nngp.nn2(c, c0, k)
    assert np.array_equal(i_got, i_ref) and np.array_equal(d_got, d_ref)
