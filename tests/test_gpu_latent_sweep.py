"""The latent sweep's kernels where a site has more children than a group of
lanes holds, and where phases are larger than the walking block or get a grid
of their own: chains within 1e-9 of the oracle's under the same stream."""
import numpy as np
import pytest

from test_gpu_latent import _args, _colour_order, _compare

pytestmark = pytest.mark.gpu


def problem(n, m, seed, ordered):
    """Sites in x order, or in random order (the first sites then have up to
    about a hundred children each)."""
    from oracle import oracle as O
    rng = np.random.default_rng(seed)
    c = rng.random((n, 2))
    if ordered:
        c = c[np.argsort(c[:, 0], kind="stable")]
    r = O.mkNNIndx(c, m)
    U = O.mkUIndx(n, m, r["nnIndx"], r["nnIndxLU"], 2)
    X = np.column_stack([np.ones(n), rng.standard_normal(n)])
    y = X @ [1.0, -2.0] + np.sin(6 * c[:, 0]) + 0.5 * rng.standard_normal(n)
    return dict(c=c, nn=r["nnIndx"], lu=r["nnIndxLU"], U=U, X=X, y=y, n=n,
                m=m, p=2, cov=0)


@pytest.mark.parametrize("n,m,ordered,sweep", [
    (5, 2, True, "site"), (2500, 12, False, "site"), (9000, 15, True, "site"),
    (16000, 8, True, "coloured")])
def test_chain_matches_oracle(oracle, n, m, ordered, sweep):
    import spnngp_amd as nn
    P = problem(n, m, 60 + m, ordered)
    S = 6
    most = int(P["U"]["u.indx.lu"][n:].max())
    print(f"[sweep] n={n} m={m} {sweep}, up to {most} children", flush=True)
    assert ordered or most > 24
    rng = np.random.default_rng(7)
    normals, unifs = rng.standard_normal(S * (n + 12)), rng.random(S * 8)
    visit = None if sweep == "site" else _colour_order(P)
    args = _args(P, S)
    a_or = list(args)
    a_or[5] = P["c"].T.reshape(-1).copy()
    want = oracle.sNNGP(*a_or[:21], a_or[23], a_or[24], S,
                        oracle.TapeRng(normals, unifs), visit=visit)
    got = nn.sNNGP(*args, rng=oracle.TapeRng(normals, unifs), sweep=sweep)
    _compare(got, want)
