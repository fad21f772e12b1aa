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
