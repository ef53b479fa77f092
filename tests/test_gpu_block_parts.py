"""GPU: the group-block product with block rows of several parts (rows of 0 to more than 128
off-diagonal blocks, part lengths with and without remainder), for groups of equal and of mixed
sizes, against the dense product of the stored matrix."""
import numpy as np
import pytest

import mpgpu
from helpers import packed_to_dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [None, 2, 16 + 4, 32 + 8])
@pytest.mark.parametrize("mixed", [False, True])
def test_block_product_of_split_rows(monkeypatch, variant, mixed):
    if variant is not None:
        monkeypatch.setenv("MPGPU_SPMV_VARIANT", str(variant))
    rp, ii, gg, _ = mpgpu.pixel_records(7, 20, 5, 4, 9000, 10, 20, slope_sigma=1.0, dz=2.5)
    P = mpgpu.Pede(matsto=mpgpu.SPARSE, metsol=mpgpu.MINRES, mreqenf=2, mcount=1)
    P.add_records(rp, ii, gg)
    if mixed:                                   # every third label and each label 7 k fixed
        lab = np.unique(ii[(ii > 0)])
        lab = lab[lab > 10]
        lab = lab[(lab % 3 == 0) | (lab % 7 == 0)]
        P.set_steering_parameters(lab, np.zeros(len(lab)), np.full(len(lab), -1.0))
    P.build_structure()
    gfirst, brow, bcol, boff, _ = P.block_structure()
    size = np.diff(gfirst)
    assert (size.min() < size.max()) == mixed
    off = np.diff(brow) - 1
    assert off.min() == 0 and off.max() > 2 * 64 and ((off > 64) & (off % 8 != 0)).any()
    P.loopn()
    n = P.nall
    x = np.random.default_rng(5).normal(size=n)
    y = P.avprod(x)
    A = packed_to_dense(P.matrix_packed(), n)
    # each of the n products and sums of an element is rounded once, in both orders of the sum
    assert (np.abs(y - A @ x) <= 4 * n * np.finfo(float).eps * (np.abs(A) @ np.abs(x))).all()
    P.close()
