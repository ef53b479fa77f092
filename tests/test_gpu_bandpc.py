"""The band preconditioner's application against the oracle's (lltdec / equdecs / equslvs, pinned
bitwise to the reference): MINRES with either one on the same matrix stops with the same code after
nearly the same number of iterations and at the same solution.  At the edges of the sub-chunk form
(bands of 2 to 9 rows, up to 128 constraints, one chunk of rows or several, incomplete chunks) and
just beyond it, where the chunk kernels without sub-chunks and the sequential constraint block
remain; with constraint blocks whose factor is formed by one wavefront (up to 110 constraints, 64
and more in two registers a lane) and in memory.  The bars are those of test_minres_sparse_constraints."""
import numpy as np
import pytest

import mpgpu
from helpers import packed_to_dense
from test_gpu_parity import _oracle_band_precond, _pede

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nl,nx,ny,hits,mbandw", [
    (3, 2, 2, 3, 6),        # 72 rows: one chunk
    (4, 5, 3, 5, 2),        # 360 rows, 12 constraints
    (4, 5, 3, 5, 9),
    (4, 5, 3, 5, 10),       # 9 boundary values: chunk kernels without sub-chunks
    (22, 2, 2, 12, 6),      # 66 constraints
    (44, 2, 1, 20, 6),      # 132 constraints: sequential constraint block
])
def test_band_preconditioner_is_the_oracles(orc, nl, nx, ny, hits, mbandw):
    _against_oracle(orc, nl, nx, ny, hits, mbandw, 3 * nl)


# (A band of 3 rows on the detector of four layers makes MINRES break down, stop code 6, in the oracle
# too: two solves that stop there are 2e-4 to 4e-3 parameter errors apart, so it is tested on the longer
# detector.)
@pytest.mark.parametrize("nl,nx,ny,hits,mbandw", [(22, 2, 2, 12, 3), (4, 5, 3, 5, 4), (4, 5, 3, 5, 5), (4, 5, 3, 5, 7), (4, 5, 3, 5, 8)])
def test_every_boundary_width(orc, nl, nx, ny, hits, mbandw):
    _against_oracle(orc, nl, nx, ny, hits, mbandw, 3 * nl)


# (110 constraints: the last factor formed in LDS; 128: the last in sub-chunk form, whose inverse
# needs more than 64 KB of LDS)
@pytest.mark.parametrize("ncon", [64, 65, 108, 110, 111, 126, 128, 129])
def test_many_constraints(orc, ncon):
    _against_oracle(orc, 44, 2, 1, 20, 6, ncon)


def _against_oracle(orc, nl, nx, ny, hits, mbandw, ncon):
    rp, ii, gg, _ = mpgpu.pixel_records(3 + nl, nl, nx, ny, 1500 * nx * ny, hits, nl + 2, wx=20.0 / nx, wy=20.0 / ny)
    weak = mpgpu.pixel_weak_labels(nl, nx, ny)
    P = _pede(rp, ii, gg, weak, mpgpu.pixel_presigma(weak), mpgpu.pixel_constraints(nl, nx, ny)[:ncon], matsto=mpgpu.SPARSE,
              metsol=mpgpu.MINRES, mreqenf=5, mcount=1, mbandw=mbandw, mrestl=1e-10, withmultipliers=1)
    assert P.ncon == ncon
    P.loopn()
    x, st = P.solve()
    A = packed_to_dense(P.matrix_packed(), P.nall)
    b, _ = P.vector()
    sig = np.sqrt(np.abs(np.diag(np.linalg.inv(A))[:P.nvar]))
    xo, so, io, _ = orc.minres(P.nall, lambda v: A @ v, _oracle_band_precond(orc, A, P.nvar, P.ncon, mbandw), b, 1e-10,
                               precon=True)
    assert st["istop"] == so
    assert abs(io - st["itn"]) <= max(3, io // 20), (io, st["itn"])
    assert np.max(np.abs(x[:P.nvar] - xo[:P.nvar]) / sig) < 1e-4
    P.close()
