"""The neighbor searches with one query a wavefront, at strips of less than,
exactly and just over 64 points, at the longest lists, and on both sides of the
number of queries where nn2 changes kernels: bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(2, 1), (63, 62), (64, 15), (65, 63),
                                 (129, 5), (1500, 63), (4097, 16),
                                 (8192, 5), (8193, 5)])
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
                                   (3000, 15, 49153), (3000, 1, 8192),
                                   (3000, 1, 8193), (3000, 5, 24577)])
def test_nn2_bit_exact(oracle, nngp, n, k, q):
    print(f"nn2 wave n={n} k={k} q={q}", flush=True)
    rng = np.random.default_rng(n + k)
    c = rng.uniform(size=(n, 2))
    c0 = rng.uniform(-0.2, 1.2, size=(q, 2))  # some outside every strip
    i_ref, d_ref = oracle.nn2(c, c0, k)
    i_got, d_got = nngp.nn2(c, c0, k)
    assert np.array_equal(i_got, i_ref) and np.array_equal(d_got, d_ref)


@pytest.mark.parametrize("side", [7, 40, 95])
def test_equal_coordinates_and_signed_zeros(oracle, nngp, side):
    """Lattices in random order, on both sides of the number of points up to
    which the strip index is counted instead of sorted: equal x and equal y, 0
    and -0, and doubled sites."""
    print(f"knn lattice {side} x {side}", flush=True)
    g = np.arange(side) - side // 2
    c = np.array([(x, y) for x in g for y in g], float) / 8.0
    rng = np.random.default_rng(side)
    c = np.vstack([c, c[rng.integers(0, len(c), 9)]])
    c = rng.permutation(c)
    c[(c == 0) & (rng.random(c.shape) < 0.5)] = -0.0
    for got, want in ((nngp.mkNNIndxCB(c, 6), oracle.mkNNIndxCB(c, 6)),
                      (nngp.mkNNIndx(c, 6), oracle.mkNNIndx(c, 6))):
        for key in ("nnIndx", "nnIndxLU", "nnDist"):
            assert np.array_equal(got[key], want[key]), key
    q = rng.uniform(-side / 16, side / 16, size=(50, 2))
    i_ref, d_ref = oracle.nn2(c, q, 9)
    i_got, d_got = nngp.nn2(c, q, 9)
    assert np.array_equal(i_got, i_ref) and np.array_equal(d_got, d_ref)


def test_more_sites_than_one_launch_holds(nngp):
    """2^26 + 5 sites, m = 1: one grid of a wavefront a site would be 2^32
    threads and more.  Sites in pairs 2k, 2k + 1 at (k, y_k) and
    (k + 1/4, y_k), y random: an odd site's nearest predecessor is its twin, as
    every other site is at least 3/4 off in x.  Even sites at both ends and on
    both sides of 2^25 and 2^26 are checked by hand."""
    n = (1 << 26) + 5
    print(f"knn n={n} m=1", flush=True)
    i = np.arange(n, dtype=np.int32)
    c = np.empty((n, 2), order="F")
    c[:, 0] = (i >> 1) + 0.25 * (i & 1)
    y = np.random.default_rng(7).uniform(0.0, 8192.0, (n + 1) // 2)
    c[:, 1] = y[i >> 1]
    got = nngp.mkNNIndx(c, 1)
    idx, dist = got["nnIndx"], got["nnDist"]
    lu = got["nnIndxLU"]
    assert np.array_equal(lu[1:n], i[:-1]) and lu[0] == 0
    assert lu[n] == 0 and (lu[n + 1:] == 1).all()
    assert idx.size == n - 1  # entry s - 1 is site s's
    assert np.array_equal(idx[0::2], i[0:n - 1:2])
    assert (dist[0::2] == 0.25).all()
    for s in [2, 4, 100, n - 3, n - 1] + [
            b + d for b in (1 << 25, 1 << 26) for d in (-2, 0, 2)]:
        lo = max(0, s - 200000)  # farther than 8192 in x
        d = np.hypot(c[lo:s, 0] - c[s, 0], c[lo:s, 1] - c[s, 1])
        k = int(np.argmin(d))
        assert idx[s - 1] == lo + k, s
        assert abs(dist[s - 1] - d[k]) <= 1e-12 * d[k], s
