"""GPU: bordered-band local fits at the limits of the kernel's phases, against the oracle: bands of
64 and 65 rows, of 10 and 11 columns, with and without border, equations of 9 and 10 local
parameters and of 64 and 65 words, a repeated label, fixed parameters, and a local inverse that does
not fit in LDS.  The bar is that of the other parity tests (FP64, only the order of sums differs)."""
import numpy as np
import pytest

import labels as LB
import mpgpu
from test_gpu_parity import _band_side, _compare_pass

pytestmark = pytest.mark.gpu


def _records(seed, nrec, npl, nbdr, window, nglob, repeat, dtype):
    """Border parameters 1 .. nbdr and one offset per plane: a measurement per plane with nglob
    global parameters of its module, and an equation of the border and `window` offsets."""
    rng = np.random.default_rng(seed)
    rp, ii, gg = [0], [], []
    for _ in range(nrec):
        ii.append(0)
        gg.append(0.0)
        for p in range(npl):
            g = 100 * (p + 1 + 200 * int(rng.integers(2))) + np.arange(1, nglob + 1)
            if repeat and p % 3 == 0:
                g = np.append(g, g[0])
            ii += [0, nbdr + p + 1, 0, *g]
            gg += [rng.normal(), rng.uniform(0.5, 1.5), 0.5, *rng.uniform(0.5, 1.5, len(g))]
        for p in range(npl - window + 1):
            ii += [0, *range(1, nbdr + 1), *range(nbdr + p + 1, nbdr + p + window + 1), 0]
            gg += [0.1 * rng.normal(), *(rng.uniform(0.5, 1.5, nbdr + window) * rng.choice([-1.0, 1.0], nbdr + window)), 0.3]
        rp.append(len(ii))
    return np.array(rp, np.int64), np.array(ii, np.int32), np.array(gg, dtype)


CASES = [
    # records, planes, border, window, globals per equation, repeated label, payload
    (200, 14, 2, 3, 2, False, np.float32),
    (100, 64, 0, 3, 2, False, np.float32),
    (100, 65, 2, 3, 2, False, np.float32),
    (100, 40, 2, 11, 1, False, np.float32),
    (60, 60, 2, 12, 1, False, np.float32),
    (200, 20, 4, 5, 6, False, np.float64),
    (200, 24, 4, 6, 6, False, np.float32),
    (40, 12, 2, 3, 61, False, np.float32),
    (40, 12, 2, 3, 62, False, np.float32),
    (200, 12, 2, 3, 3, True, np.float32),
    (40, 100, 2, 3, 2, False, np.float32),
]


@pytest.mark.parametrize("matsto", [mpgpu.FULL, mpgpu.SPARSE])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c[:6]))
def test_band_pass_sizes(orc, case, matsto):
    rp, ii, gg = _records(sum(case[:5]), *case)
    assert _band_side(LB.decode(rp, ii, gg), ii, 0) > 0
    fixed = [102, 302] if case[4] > 1 else [100]
    P = mpgpu.Pede(matsto=matsto, metsol=mpgpu.MINRES, mreqenf=1, mcount=1, lhuber=3)
    P.add_records(rp, ii, gg)
    P.set_steering_parameters(fixed, 0.05 * np.ones(len(fixed)), -np.ones(len(fixed)))
    P.build_structure()
    lab, var = P.labels()[:2]
    l2, v2 = LB.label_maps(rp, ii, gg.astype(float), steer_labels=fixed, presigma=[-1.0] * len(fixed), mreqenf=1, mcount=1)[:2]
    assert np.array_equal(lab, l2) and np.array_equal(var, v2)
    par = P.parameters()
    par[var > 0] = 0.3 / case[4] * np.sin(np.arange(P.nvar))
    P.set_parameters(par)
    s, _, _ = _compare_pass(P, orc, rp, ii, gg, lab, var)
    assert s["naccept"] > 0
    _compare_pass(P, orc, rp, ii, gg, lab, var, nloopn=2, lhuber=3, chicut=1.2)
    P.close()
