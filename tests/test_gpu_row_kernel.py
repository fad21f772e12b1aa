"""The 16-lane-row kernel where its entries and its launch can go wrong: the
Matern table's piece and octave borders and both ends of its range, against
the CPU oracle at the parity bound of the FP64 path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-10


def spread_coords(n, seed):
    """x-ordered sites whose distances run over many octaves: geometric gaps
    from 1e-11 to 10 along x, a jitter in y of the size of the gap, and every
    16th site a duplicate of the one before it."""
    rng = np.random.default_rng(seed)
    gap = 10.0 ** rng.uniform(-11, 1, n)
    gap[::16] = 0.0
    x = np.cumsum(gap)
    y = gap * rng.normal(size=n)
    y[::16] = np.roll(y, 1)[::16]
    return np.column_stack([x, y])


@pytest.mark.parametrize("m,nu,phi", [(3, 0.7, 1.0), (12, 1.2, 7.0),
                                      (16, 2.2, 1e-4), (17, 0.35, 40.0),
                                      (32, 1.9, 0.3)])
def test_matern_table_over_its_whole_range(oracle, nngp, m, nu, phi):
    """phi d from below 2^-30 (the series' side of the table) over every
    octave to beyond 64 (the other side), exact zeros among them.  n = 1001
    leaves a ragged last group of four sites.  B, F and the log determinant
    within 1e-10 of the oracle."""
    n, theta = 1001, [1.0, 0.5, phi, nu]
    print(f"matern table m={m} nu={nu} phi={phi}", flush=True)
    c = spread_coords(n, 30 + m)
    nn = oracle.mkNNIndx(c, m)
    lu = nn["nnIndxLU"]
    B0, F0, ld0 = oracle.updateBF(c.T.reshape(-1).copy(), nn["nnIndx"], lu, n,
                                  m, theta, 2)
    with nngp.Model(c, nn["nnIndx"], lu, m, 2) as md:
        for threads in (64, 256):
            md.set_shape(2, threads, 0)
            out = md.update(theta, slot=0)
            B, F = md.get_bf(0)
            assert np.max(np.abs(F - F0) / F0) < RTOL
            assert np.max(np.abs(B - B0)) < RTOL * np.max(np.abs(B0))
            assert abs(out["logDet"] - ld0) < RTOL * abs(ld0)
