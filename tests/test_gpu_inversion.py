"""Inversion at the edges of its forms against sqminl (the oracle's restatement, bit-identical to
the reference): matrices inverted in LDS (up to 128 rows) and in panels of 16 pivots (one, two or
more rows per thread), sizes around the panel and the tile, with and without a rank defect.
FP64 throughout; the panels sum in another order, which moves the result by about cond * 1e-16:
for these well-conditioned matrices (unit diagonal, off-diagonal sums below 1) 1e-12 covers it."""
import numpy as np
import pytest

import mpgpu
from helpers import packed_to_dense

pytestmark = pytest.mark.gpu


def _context(n):
    """A context of n variable parameters whose matrix the test sets: one record that touches every
    parameter makes them variable, the matrix is then filled by mupdat."""
    ii, gg = [0], [0.0]
    for e in range(n):
        ii += [0, 1, 0, e + 1]
        gg += [0.0, 1.0, 1.0, 1.0]
    P = mpgpu.Pede(matsto=mpgpu.FULL, metsol=mpgpu.INVERSION, mreqenf=1, mcount=1)
    # records of at most 100 equations, each with one local parameter
    rp, io, go = [0], [], []
    for a in range(0, n, 100):
        io.append(0)
        go.append(0.0)
        for e in range(a, min(n, a + 100)):
            io += [0, 1, 0, 2 * e + 1]
            go += [0.0, 1.0, 1.0, 1.0]
        rp.append(len(io))
    P.add_records(np.array(rp, np.int64), np.array(io, np.int32), np.array(go, np.float32))
    P.build_structure()
    assert P.nall == n
    P.loopn()
    return P


@pytest.mark.parametrize("n,defect", [(3, 0), (64, 0), (128, 0), (128, 3), (129, 0), (144, 5), (250, 0), (1023, 0), (1024, 2),
                                      (1100, 0), (2047, 0), (2100, 4)])
def test_inversion_forms(orc, n, defect):
    rng = np.random.default_rng(n)
    P = _context(n)
    A0 = packed_to_dense(P.matrix_packed(), n)
    # a few couplings per row, diagonal dominant; `defect` rows are exact copies of others
    B = np.zeros((n, n))
    for _ in range(3):
        k = rng.permutation(n)
        B[np.arange(n), k] += rng.uniform(-0.15, 0.15, n)
    B = np.tril(B + B.T, -1)
    B = B + B.T + np.diag(rng.uniform(1.0, 3.0, n))
    for q in range(defect):
        a, b = 2 * q, n - 1 - 2 * q
        B[b, :] = B[a, :]
        B[:, b] = B[:, a]
        B[b, b] = B[a, a]
    D = np.tril(B - A0)
    i, j = np.nonzero(D)
    P.mupdat(i + 1, j + 1, D[i, j])
    p = P.matrix_packed()
    rhs = rng.normal(size=n)
    inv, xo, rank = orc.sqminl(p, rhs)
    x, st = P.solve(rhs)
    assert st["nrank"] == rank == n - defect
    got = P.matrix_packed()
    assert np.abs(got - inv).max() <= 1e-12 * np.abs(inv).max()
    assert np.abs(x - xo).max() <= 1e-12 * np.abs(xo).max()
    P.close()
