"""Records in row form (equations that each touch one group of at most 8
parameters, at most 5 local parameters, 128 equations, 4 equations per group) against the oracle,
at the edges of what has that form and just beyond, where the other record kernel takes over:
equations per wavefront (64, 66, 128, 130), group sizes, local parameters, equations per group
(an odd one leaves half a unit empty), fixed parameters inside a group, FP64 payloads, rejected
records, and lists of a matrix block short and long (few modules, many records).  The bar is that
of the other parity tests: FP64 arithmetic, only the order of sums differs, 1e-10 relative."""
import numpy as np
import pytest

import labels as LB
import mpgpu
from test_gpu_parity import _compare_pass

pytestmark = pytest.mark.gpu


def _records(seed, nmod, gsize, nloc, nrec, hits, per_hit, dtype):
    rng = np.random.default_rng(seed)
    rp, ii, gg = [0], [], []
    for _ in range(nrec):
        ii.append(0)
        gg.append(0.0)
        for m in rng.choice(nmod, hits, replace=False):
            for e in range(per_hit):
                l = rng.uniform(0.5, 1.5, nloc) * rng.choice([-1.0, 1.0], nloc)
                g = rng.uniform(0.5, 1.5, gsize) * rng.choice([-1.0, 1.0], gsize)
                if gsize > 2 and per_hit > 1:
                    g[e % 2] = 0.0                       # a derivative left out, as Mille does
                k = np.flatnonzero(g)
                ii += [0, *range(1, nloc + 1), 0, *(100 * (int(m) + 1) + k + 1)]
                gg += [rng.normal() * (20.0 if rng.random() < 0.02 else 1.0), *l, 0.5, *g[k]]
        # an equation without global parameters
        ii += [0, 1, 0]
        gg += [0.1, 1.0, 0.7]
        rp.append(len(ii))
    return np.array(rp, np.int64), np.array(ii, np.int32), np.array(gg, dtype)


CASES = [
    # modules, group, local, records, hits, equations per hit, payload
    (6, 1, 1, 200, 3, 1, np.float32),
    (10, 2, 2, 300, 5, 1, np.float32),
    (12, 3, 3, 300, 9, 2, np.float64),
    (40, 6, 4, 60, 31, 2, np.float32),      # 63 equations
    (40, 6, 4, 60, 32, 2, np.float32),      # 65
    (70, 6, 4, 40, 63, 2, np.float32),      # 127
    (70, 6, 4, 40, 64, 2, np.float32),      # 129: not in row form
    (12, 7, 5, 200, 8, 3, np.float32),
    (12, 8, 5, 200, 8, 4, np.float64),
    (12, 6, 4, 100, 8, 5, np.float32),      # five equations per group: not in row form
    (12, 9, 4, 100, 8, 2, np.float32),      # nine parameters per group: not in row form
    (12, 6, 6, 100, 8, 2, np.float32),      # six local parameters: not in row form
    (5, 6, 4, 1500, 4, 2, np.float32),      # lists of 900 pairs per block
]


@pytest.mark.parametrize("matsto", [mpgpu.SPARSE, mpgpu.FULL])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c[:6]))
def test_row_form_pass(orc, case, matsto):
    nmod, gsize, nloc, nrec, hits, per_hit, dtype = case
    rp, ii, gg = _records(sum(case[:6]), nmod, gsize, nloc, nrec, hits, per_hit, dtype)
    # a parameter inside every third group is fixed at a start value
    fixed = [100 * (m + 1) + gsize // 2 + 1 for m in range(0, nmod, 3)] if gsize > 1 else []
    P = mpgpu.Pede(matsto=matsto, metsol=mpgpu.MINRES, mreqenf=1, mcount=1, lhuber=3, lfitbb=0)
    P.add_records(rp, ii, gg)
    if fixed:
        P.set_steering_parameters(fixed, 0.05 * np.ones(len(fixed)), -np.ones(len(fixed)))
    P.build_structure()
    lab, var = P.labels()[:2]
    l2, v2 = LB.label_maps(rp, ii, gg.astype(float), steer_labels=fixed, presigma=[-1.0] * len(fixed), mreqenf=1, mcount=1)[:2]
    assert np.array_equal(lab, l2) and np.array_equal(var, v2)
    par = P.parameters()
    par[var > 0] = 1e-3 * np.arange(P.nvar)
    P.set_parameters(par)
    _compare_pass(P, orc, rp, ii, gg, lab, var, chicut=0.0)
    s, _, _ = _compare_pass(P, orc, rp, ii, gg, lab, var, nloopn=2, lhuber=3, chicut=1.2)
    _compare_pass(P, orc, rp, ii, gg, lab, var, nloopn=2, lhuber=3, icalcm=0)
    P.close()
