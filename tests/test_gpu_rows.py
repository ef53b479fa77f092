"""Records in row form (equations that each touch one group of at most 8
parameters, at most 5 local parameters, 128 equations, 4 equations per group) against the oracle,
at the edges of what has that form and just beyond, where the other record kernel takes over:
equations per wavefront (64, 66, 128, 130), group sizes, local parameters, equations per group
(an odd one leaves half a unit empty), fixed parameters inside a group, FP64 payloads, rejected
records, and lists of a matrix block short and long (few modules, many records).  The bar is that
of the other parity tests: FP64 arithmetic, only the order of sums differs, 1e-10 relative."""
import re

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


# which records of the cases have row form
IN_ROW_FORM = [True] * 6 + [False] + [True] * 2 + [False] * 3 + [True]


def paths(err):
    """(records in row form, batches, records of the record kernel, batches) from the build's MPGPU_VERBOSE line"""
    m = re.findall(r"records in row form: (\d+) in (\d+) batches, by the record kernel: (\d+) in (\d+)", err)
    return tuple(map(int, m[-1]))


@pytest.mark.parametrize("matsto", [mpgpu.SPARSE, mpgpu.FULL])
@pytest.mark.parametrize("k", range(len(CASES)))
def test_which_records_have_row_form(monkeypatch, capfd, k, matsto):
    nmod, gsize, nloc, nrec, hits, per_hit, dtype = CASES[k]
    rp, ii, gg = _records(sum(CASES[k][:6]), nmod, gsize, nloc, nrec, hits, per_hit, dtype)
    monkeypatch.setenv("MPGPU_VERBOSE", "1")
    P = mpgpu.Pede(matsto=matsto, metsol=mpgpu.MINRES, mreqenf=1, mcount=1, lfitbb=0)
    P.add_records(rp, ii, gg)
    P.build_structure()
    P.close()
    row, _, gen, _ = paths(capfd.readouterr().err)
    assert (row, gen) == ((nrec, 0) if IN_ROW_FORM[k] else (0, nrec))


def _mixed(seed, nmod=24, nrec=600):
    """records of both forms on the same modules: two thirds with 4 local parameters, the others with 6"""
    a = _records(seed, nmod, 6, 4, nrec * 2 // 3, 8, 2, np.float32)
    b = _records(seed + 1, nmod, 6, 6, nrec - nrec * 2 // 3, 8, 2, np.float32)
    cut = lambda r: [(r[1][x:y], r[2][x:y]) for x, y in zip(r[0][:-1], r[0][1:])]
    recs = cut(a) + cut(b)
    np.random.default_rng(seed + 2).shuffle(order := np.arange(len(recs)))
    rp = np.concatenate([[0], np.cumsum([len(recs[k][0]) for k in order])]).astype(np.int64)
    return rp, np.concatenate([recs[k][0] for k in order]), np.concatenate([recs[k][1] for k in order])


@pytest.mark.parametrize("matsto", [mpgpu.SPARSE, mpgpu.FULL])
@pytest.mark.parametrize("batches", [False, True])
def test_records_of_both_forms(orc, monkeypatch, capfd, matsto, batches):
    """Both gathers (or the gather and the atomic additions) add to the same blocks, vector and counters, in one
    batch and with a buffer so small that each takes several."""
    rp, ii, gg = _mixed(11, nrec=3600 if batches else 600)
    n = len(rp) - 1
    monkeypatch.setenv("MPGPU_VERBOSE", "1")
    if batches:
        monkeypatch.setenv("MPGPU_UPDATE_BUFFER_GB", "0.001")       # 2^20 doubles, the least that is taken
    P = mpgpu.Pede(matsto=matsto, metsol=mpgpu.MINRES, mreqenf=1, mcount=1, lhuber=3, lfitbb=0)
    P.add_records(rp, ii, gg)
    P.build_structure()
    row, nb, gen, nb2 = paths(capfd.readouterr().err)
    assert (row, gen) == (n * 2 // 3, n - n * 2 // 3)
    assert (nb > 1) == batches and (nb2 > 1) == (batches and matsto == mpgpu.SPARSE)
    lab, var = P.labels()[:2]
    par = P.parameters()
    par[var > 0] = 1e-3 * np.arange(P.nvar)
    P.set_parameters(par)
    _compare_pass(P, orc, rp, ii, gg, lab, var, chicut=0.0)
    _compare_pass(P, orc, rp, ii, gg, lab, var, nloopn=2, lhuber=3, chicut=1.2)
    _compare_pass(P, orc, rp, ii, gg, lab, var, nloopn=2, lhuber=3, icalcm=0)
    P.close()


@pytest.mark.parametrize("matsto", [mpgpu.SPARSE, mpgpu.FULL])
@pytest.mark.parametrize("nloc", [4, 6])
def test_small_buffer(monkeypatch, capfd, orc, matsto, nloc):
    """Several batches of records of one form (6 local parameters: the record kernel and the gather of its
    updates, in full storage one launch of atomic additions)."""
    rp, ii, gg = _records(5 + nloc, 24, 6, nloc, 2500, 8, 2, np.float32)
    monkeypatch.setenv("MPGPU_VERBOSE", "1")
    monkeypatch.setenv("MPGPU_UPDATE_BUFFER_GB", "0.001")
    P = mpgpu.Pede(matsto=matsto, metsol=mpgpu.MINRES, mreqenf=1, mcount=1, lfitbb=0)
    P.add_records(rp, ii, gg)
    P.build_structure()
    row, nb, gen, nb2 = paths(capfd.readouterr().err)
    assert (row, gen) == ((2500, 0) if nloc == 4 else (0, 2500))
    assert nb > 1 if nloc == 4 else nb2 > 1 or matsto == mpgpu.FULL
    lab, var = P.labels()[:2]
    _compare_pass(P, orc, rp, ii, gg, lab, var)
    P.close()


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
