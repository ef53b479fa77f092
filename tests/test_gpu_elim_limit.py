"""MINRES with eliminated constraints that ends at its iteration limit: the solution of the unfinished
iteration depends on the order of every sum, so that order is fixed.  The golden file has every 60th
parameter as the pass and solve with one order gave it (records one at a time, whole block rows, band
solves by substitution, reflections in four launches).  Another order of one of these sums alone
moves the solution of this system by 5e-4 to 3e-3 (measured one at a time); the same order repeats it
bit for bit, so the tolerance is for the last bits only."""
import os
import numpy as np
import pytest

import mpgpu
from helpers import packed_to_dense
from test_gpu_parity import _dense_constraints, _pede

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "minres_elim_limit.txt")
LAYERS, NX, NY = 20, 13, 3


def _context(itnlim):
    rp, ii, gg, _ = mpgpu.pixel_records(5, LAYERS, NX, NY, NX * NY * 900, 8, 30, wx=100.0 / NX, wy=100.0 / NY, sigma=0.002)
    P = mpgpu.Pede(matsto=mpgpu.SPARSE, metsol=mpgpu.MINRES, mreqenf=5, mcount=1, mbandw=6, mrestl=1e-14, itnlim=itnlim,
                   withmultipliers=0)
    P.add_records(rp, ii, gg)
    lab = np.array(mpgpu.pixel_weak_labels(LAYERS, NX, NY), dtype=np.int32)
    P.set_steering_parameters(lab, np.zeros(len(lab)), np.array(mpgpu.pixel_presigma(lab)))
    P.add_constraints(mpgpu.pixel_constraints(LAYERS, NX, NY))
    P.build_structure()
    P.loopn(1, 1, 0.0)
    return P


def test_solution_at_the_iteration_limit():
    P = _context(2000)
    x, st = P.solve()
    assert st["istop"] == 5 and st["itn"] == 2000
    want = [line.split() for line in open(GOLDEN)]
    at = np.array([int(k) for k, _ in want])
    gold = np.array([float.fromhex(v) for _, v in want])
    assert np.linalg.norm(x[at] - gold) <= 1e-10 * np.linalg.norm(gold)
    y, _ = P.solve()
    assert np.array_equal(x, y)
    P.close()


@pytest.mark.parametrize("ncon", [127, 128, 129, 132])
def test_many_eliminated_constraints(ncon):
    """Around 128 constraints, where the reflections go from two launches each to four: against the
    dense KKT solve of the same matrix, the bars of test_minres_elimination."""
    nl, nx, ny = 44, 2, 1
    rp, ii, gg, _ = mpgpu.pixel_records(47, nl, nx, ny, 3000, 20, nl + 2, wx=10.0, wy=20.0)
    weak = mpgpu.pixel_weak_labels(nl, nx, ny)
    cons = mpgpu.pixel_constraints(nl, nx, ny)[:ncon]
    cons = [(2e-3 * (j % 7), s, l, f) for j, (_, s, l, f) in enumerate(cons)]
    P = _pede(rp, ii, gg, weak, mpgpu.pixel_presigma(weak), cons, matsto=mpgpu.SPARSE, metsol=mpgpu.MINRES, mreqenf=5,
              mcount=1, mbandw=6, mrestl=1e-12, itnlim=5000, withmultipliers=0)
    assert P.ncon == 0 and P.nall == P.nvar
    P.loopn()
    x, st = P.solve()
    A = packed_to_dense(P.matrix_packed(), P.nvar)
    b, _ = P.vector()
    C, d = _dense_constraints(P, cons)
    assert C.shape[0] == ncon
    K = np.block([[A, C.T], [C, np.zeros((ncon, ncon))]])
    xr = np.linalg.solve(K, np.concatenate([b, d]))[:P.nvar]
    sig = np.sqrt(np.abs(np.diag(np.linalg.inv(K))[:P.nvar]))
    assert st["istop"] in (1, 2)
    assert np.abs(C @ x - d).max() < 1e-10 * max(1.0, np.abs(C).max() * np.abs(x).max())
    assert np.max(np.abs(x - xr) / sig) < 1e-4
    P.close()
