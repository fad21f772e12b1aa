"""The per-lane updateBF kernel that keeps finished rows of the factor in LDS
(launch mode 2), at the sizes where its template sizes, its kept rows and its
ways of reading the covariate rows change, against the CPU oracle."""
import numpy as np
import pytest

from conftest import uniform_coords

pytestmark = pytest.mark.gpu

RTOL = 1e-10


# m at both ends of every kernel size (10, 12, 15, 16); p = 0 and 1: one pair
# a covariate row, 2 and 3: two pairs, 5: rows read by single values
@pytest.mark.parametrize("m,p,cov,theta", [
    (9, 0, 0, [1.0, 0.1, 6.0]), (10, 5, 1, [1.5, 0.3, 2.0]),
    (11, 1, 3, [1.0, 0.1, 5.0]), (12, 3, 2, [1.0, 0.1, 9.0, 2.5]),
    (13, 2, 0, [2.0, 0.2, 12.0]), (15, 5, 2, [1.0, 0.1, 9.0, 1.5]),
    (15, 1, 1, [1.5, 0.3, 2.0]), (16, 3, 0, [2.0, 0.2, 12.0]),
    (16, 0, 3, [1.0, 0.2, 5.0]),
])
def test_rows_in_lds_match_the_oracle(oracle, nngp, m, p, cov, theta):
    """B, F, log det, Q(r, r) within 1e-10 at one site more than a full block
    and at fewer sites than one block."""
    for n in (m + 3, 64 * 9 + 1):
        print(f"lane mode 2 n={n} m={m} p={p} cov={cov}", flush=True)
        c = uniform_coords(n, 900 + m + p)
        rng = np.random.default_rng(m + 100 * p)
        X = np.column_stack([np.ones(n), rng.normal(size=(n, p - 1))]) \
            if p else None
        beta = np.linspace(1.0, -1.0, p) if p else np.zeros(1)
        y = (X @ beta if p else 0.0) + rng.normal(size=n)
        nn = oracle.mkNNIndxCB(c, m)
        lu = nn["nnIndxLU"]
        B0, F0, ld0 = oracle.updateBF(c.T.reshape(-1).copy(), nn["nnIndx"], lu,
                                      n, m, theta, cov)
        with nngp.Model(c, nn["nnIndx"], lu, m, cov, X, y) as md:
            md.set_shape(0, 64, 2)
            out = md.update(theta, slot=0, beta=beta)
            B, F = md.get_bf(0)
        assert np.max(np.abs(F - F0) / F0) < RTOL
        assert np.max(np.abs(B - B0)) < RTOL * np.max(np.abs(B0))
        assert abs(out["logDet"] - ld0) < RTOL * max(abs(ld0), 1.0)
        if p:
            r = X @ beta - y
            q0 = oracle.Q(B0, F0, r, r, nn["nnIndx"], lu)
            assert abs(out["qResid"] - q0) < RTOL * abs(q0)


# The solve's verdict reaches the caller from a lane of a partly filled second
# wave: sample 70 of 77 alone has no nugget, and the new site's two nearest
# neighbors coincide, so its second pivot is exactly 4 - 2 * 2 = 0.
@pytest.mark.parametrize("m", [10, 15, 16])
@pytest.mark.parametrize("cov", [0, 1, 3])
def test_kriging_reports_the_one_singular_sample(nngp, m, cov):
    n, S, q = 400, 77, 3
    c = uniform_coords(n, 77 + m)
    rng = np.random.default_rng(m)
    c[201] = c[200]
    X = np.ones((n, 1))
    y = rng.normal(size=n)
    c0 = c[[50, 200, 300]] + 1e-6
    nn0 = np.array([np.argsort(((c - s) ** 2).sum(1), kind="stable")[:m]
                    for s in c0])
    assert set(nn0[1, :2]) == {200, 201}
    theta = np.repeat([[4.0], [0.5], [3.0]], S, axis=1)
    beta = np.zeros((1, S))
    z = rng.normal(size=q * S)
    args = (X, y, c, n, 1, m, np.ones((q, 1)), c0, q, nn0, beta)
    ok = nngp.rNNGPPredict(*args, theta, S, cov, z=z)["p.y.0"]
    assert np.isfinite(ok).all()
    theta[1, 70] = 0.0
    with pytest.raises(nngp.NngpError) as e:
        nngp.rNNGPPredict(*args, theta, S, cov, z=z)
    assert e.value.status == nngp.NNGP_ERR_NOT_PD


@pytest.mark.parametrize("cov,tail", [(0, []), (1, []), (2, [1.5]), (3, [])])
def test_grid_reports_a_singular_training_site(nngp, cov, tail):
    """A training site whose two nearest neighbors coincide: alpha = 0 is
    singular there, alpha = 0.1 is not."""
    n, m = 500, 15
    c = uniform_coords(n, 31)
    c[201] = c[200]
    c[202] = c[200] + 1e-6
    rng = np.random.default_rng(5)
    ho = np.array([np.arange(0, 40), np.arange(400, 440)])
    with nngp.CvGrid(rng.normal(size=n), np.ones((n, 1)), c, m, ho,
                     [2.0, 1.0], cov, shape=(0, 64, 2)) as g:
        assert np.isfinite(g.run([[3.0, 0.1] + tail])["scores"]).all()
        with pytest.raises(nngp.NngpError) as e:
            g.run([[3.0, 0.1] + tail, [3.0, 0.0] + tail])
        assert e.value.status == nngp.NNGP_ERR_NOT_PD


# The spherical is one formula of a selected argument: 0 beyond the range, the
# sill at distance 0.  On a lattice of spacing 1/8 with a range of 1/4 and
# doubled sites the distances 0 and exactly 1/phi both occur.
@pytest.mark.parametrize("m,shape", [(4, (0, 64, 0)), (15, (0, 64, 2)),
                                     (16, (0, 64, 2)), (16, (0, 256, 0)),
                                     (20, (2, 256, 0)), (40, (1, 64, 0))])
def test_spherical_at_its_edges(oracle, nngp, m, shape):
    print(f"spherical edges m={m} shape={shape}", flush=True)
    g = np.arange(18) / 8.0
    c = np.array([(x, y) for x in g for y in g])
    rng = np.random.default_rng(m)
    c = np.vstack([c, c[rng.integers(0, len(c), 60)]])
    c = c[np.argsort(c[:, 0], kind="stable")]
    n = len(c)
    nn = oracle.mkNNIndxCB(c, m)
    theta = [1.5, 0.3, 4.0]
    B0, F0, ld0 = oracle.updateBF(c.T.reshape(-1).copy(), nn["nnIndx"],
                                  nn["nnIndxLU"], n, m, theta, 1)
    X, y = np.ones((n, 1)), rng.normal(size=n)
    with nngp.Model(c, nn["nnIndx"], nn["nnIndxLU"], m, 1, X, y) as md:
        md.set_shape(*shape)
        out = md.update(theta, slot=0, beta=np.zeros(1))
        B, F = md.get_bf(0)
    assert np.max(np.abs(F - F0) / F0) < RTOL
    assert np.max(np.abs(B - B0)) < RTOL * np.max(np.abs(B0))
    assert abs(out["logDet"] - ld0) < RTOL * max(abs(ld0), 1.0)


@pytest.mark.parametrize("cov,n,p", [(0, 4013, 1), (1, 4013, 3), (2, 4013, 5),
                                     (0, 65536, 5), (1, 65537, 5),
                                     (2, 65601, 3)])
def test_mixed_m16_forms_agree(nngp, cov, n, p):
    """m = 16 in mixed precision: the form with the covariance in registers runs
    one wave a SIMD, with the covariate rows read by pairs (p = 1, 3) or one by
    one (p = 5), and above 65,536 sites without pairs two waves.  B and F are
    those of the form that evaluates C again, bit for bit."""
    print(f"mixed m=16 cov={cov} n={n} p={p}", flush=True)
    m = 16
    c = uniform_coords(n, 7 + cov)
    rng = np.random.default_rng(n + p)
    X = np.column_stack([np.ones(n), rng.normal(size=(n, p - 1))])
    beta = np.linspace(1.0, -1.0, p)
    y = X @ beta + rng.normal(size=n)
    nn = nngp.mkNNIndxCB(c, m)
    theta = [2.0, 0.2, 12.0 if cov != 1 else 3.0] + ([1.5] if cov == 2 else [])
    with nngp.Model(c, nn["nnIndx"], nn["nnIndxLU"], m, cov, X, y,
                    precision=1) as md:
        md.set_shape(0, 64, 0)
        ref = md.update(theta, slot=0, beta=beta)
        B0, F0 = md.get_bf(0)
        for th in (64, 128, 256):
            md.set_shape(0, th, 3)
            out = md.update(theta, slot=0, beta=beta)
            B, F = md.get_bf(0)
            assert np.array_equal(B, B0) and np.array_equal(F, F0), th
            for key in ("logDet", "qResid"):
                assert abs(out[key] - ref[key]) < 1e-12 * abs(ref[key]), key
