"""Serving engine: concurrent jobs on one GPU give the same result as the job run alone, and
every job reports its latency."""
import numpy as np
import pytest

import mpgpu

pytestmark = pytest.mark.gpu


def _job(seed, nl, nx, ny, ntr):
    rp, ii, gg, _ = mpgpu.pixel_records(seed, nl, nx, ny, ntr, 4, 8, wx=100.0 / nx, wy=100.0 / ny)
    weak = mpgpu.pixel_weak_labels(nl, nx, ny)
    params = (np.array(weak), np.zeros(len(weak)), np.array(mpgpu.pixel_presigma(weak)))
    return (rp, ii, gg), params, mpgpu.pixel_constraints(nl, nx, ny)


def test_alone_vs_in_the_mix():
    rec, par, cons = _job(1, 6, 4, 3, 3000)
    opt = dict(matsto=mpgpu.FULL, metsol=mpgpu.DECOMPOSITION, mreqenf=5, mcount=1)
    S = mpgpu.Server(nworkers=4, budget_bytes=8 << 30)
    j = S.submit(rec, par, cons, **opt)
    rc, st, lab0, x0 = S.wait(j, capacity=100000)
    assert rc == 0 and st["nvar"] > 0 and st["latency_ms"] > 0
    others = [_job(10 + k, 5 + k % 3, 3 + k % 2, 3, 1500 + 200 * k) for k in range(6)]
    ids = []
    for k, (r2, p2, c2) in enumerate(others):
        o2 = dict(opt) if k % 2 == 0 else dict(matsto=mpgpu.SPARSE, metsol=mpgpu.MINRES, mbandw=6, mreqenf=5, mcount=1,
                                                mrestl=1e-10)
        ids.append(S.submit(r2, p2, c2, **o2))
        if k == 2:
            jm = S.submit(rec, par, cons, **opt)
    for i in ids:
        rc2, st2, _, _ = S.wait(i)
        assert rc2 == 0, st2
    rc, st, lab1, x1 = S.wait(jm, capacity=100000)
    assert rc == 0
    assert np.array_equal(lab0, lab1)
    # the two runs differ only in the order of the FP64 atomic additions of the matrix build
    # (1e-16 relative per element), amplified by the condition of the system (~1e8 here)
    assert np.max(np.abs(x1 - x0)) <= 1e-7 * np.max(np.abs(x0))
    S.close()


def test_group_block_job_bitwise_alone_vs_in_the_mix():
    """Group-block storage has no FP64 atomics on the path of a pixel job: the matrix and the
    vector are summed per block in processing order (the vector values ride in the records'
    updates), the product, the preconditioner and the MINRES reductions use fixed orders, and
    the product variants the autotuner picks between are bit-identical.  The same job alone and
    among concurrent jobs gives the bit-identical solution."""
    rec, par, cons = _job(3, 6, 4, 3, 3000)
    opt = dict(matsto=mpgpu.SPARSE, metsol=mpgpu.MINRES, mbandw=6, mreqenf=5, mcount=1, mrestl=1e-12)
    S = mpgpu.Server(nworkers=4, budget_bytes=8 << 30)
    rc, st, lab0, x0 = S.wait(S.submit(rec, par, cons, **opt), capacity=100000)
    assert rc == 0 and st["nvar"] > 0
    others = [_job(20 + k, 5 + k % 3, 3 + k % 2, 3, 1500 + 300 * k) for k in range(6)]
    ids = []
    for k, (r2, p2, c2) in enumerate(others):
        ids.append(S.submit(r2, p2, c2, **opt))
        if k == 2:
            jm = S.submit(rec, par, cons, **opt)
    for i in ids:
        rc2, st2, _, _ = S.wait(i)
        assert rc2 == 0, st2
    rc, st, lab1, x1 = S.wait(jm, capacity=100000)
    assert rc == 0
    assert np.array_equal(lab0, lab1)
    assert np.array_equal(x0, x1)
    S.close()


def test_budget_rejects_oversized_job():
    """A job larger than the whole budget ends with status 30 (the worker that takes it sizes
    it); the server keeps serving the next ones."""
    rec, par, cons = _job(2, 4, 3, 3, 500)
    S = mpgpu.Server(nworkers=1, budget_bytes=1 << 20)
    j = S.submit(rec, par, cons, matsto=mpgpu.FULL, metsol=mpgpu.DECOMPOSITION, mreqenf=5, mcount=1)
    rc, st, _, _ = S.wait(j)
    assert rc == 30 and st["status"] == 30
    S.close()
    S = mpgpu.Server(nworkers=2, budget_bytes=8 << 30)
    j = S.submit(rec, par, cons, matsto=mpgpu.FULL, metsol=mpgpu.DECOMPOSITION, mreqenf=5, mcount=1)
    rc, st, lab, x = S.wait(j, capacity=10000)
    assert rc == 0 and st["nvar"] == len(lab) > 0
    S.close()


def _sized_jobs():
    """jobs of every method and storage, and records with and without row form"""
    from test_gpu_rows import _records
    rec, par, cons = _job(5, 6, 4, 3, 4000)
    no_rows = _records(9, 30, 6, 6, 2000, 8, 2, np.float32)
    single = _records(10, 400, 1, 3, 4000, 20, 1, np.float32)
    dense, dpar, dcons = _job(6, 8, 6, 4, 2000)
    full = dict(matsto=mpgpu.FULL, mreqenf=5, mcount=1)
    block = dict(matsto=mpgpu.SPARSE, metsol=mpgpu.MINRES, mreqenf=5, mcount=1, mbandw=6, mrestl=1e-10)
    out = []
    for m in (mpgpu.INVERSION, mpgpu.DECOMPOSITION, mpgpu.CHOLESKY_FP32_IR, mpgpu.LAPACK_PACKED, mpgpu.MINRES):
        out.append((rec, par, cons, dict(full, metsol=m)))
        out.append((dense, dpar, dcons, dict(full, metsol=m)))
    out.append((dense, dpar, dcons, dict(full, metsol=mpgpu.CHOLESKY_FP32_IR, fp32_min_n=100)))
    for r in (no_rows, single):
        out.append((r, None, None, dict(full, metsol=mpgpu.INVERSION, default_presigma=1.0)))
        out.append((r, None, None, dict(block, default_presigma=1.0)))
    for w in (0, 1):
        out.append((rec, par, cons, dict(block, withmultipliers=w)))
        out.append((dense, dpar, dcons, dict(block, withmultipliers=w)))
    return out


def test_memory_charged_to_a_job_covers_what_it_uses(monkeypatch, capfd):
    import re
    monkeypatch.setenv("MPGPU_VERBOSE", "1")
    S = mpgpu.Server(nworkers=1, budget_bytes=60 << 30)
    capfd.readouterr()
    for rec, par, cons, opt in _sized_jobs():
        rc, st, _, _ = S.wait(S.submit(rec, par, cons, **opt))
        assert rc == 0, (rc, opt)
    S.close()
    lines = re.findall(r"charged (\d+) bytes \(least (\d+)\), in use at most (\d+)", capfd.readouterr().err)
    assert len(lines) == len(_sized_jobs())
    # (64 MB of every estimate are for what does not grow with the job: not for these to hide in)
    for line, (_, _, _, opt) in zip(lines, _sized_jobs()):
        charged, least, peak = map(int, line)
        assert peak <= charged - (64 << 20), opt


def test_job_whose_least_part_fits_the_budget_runs():
    """More memory than the budget would only make the job faster: it is accepted as long as what it cannot do
    without fits, and refused below that."""
    rec, par, cons = _job(5, 8, 8, 6, 20000)
    opt = dict(matsto=mpgpu.FULL, metsol=mpgpu.INVERSION, mreqenf=5, mcount=1)
    n = 6 * 8 * 8 * 6 + 3 * 8
    words = len(rec[1])
    least = 12 * words + 64 * 20000 + 8 * n * (n + 1) + 200 * n + (64 << 20)
    for budget, want in ((int(1.001 * least), 0), (int(0.9 * least), 30)):
        S = mpgpu.Server(nworkers=2, budget_bytes=budget)
        rc, st, _, _ = S.wait(S.submit(rec, par, cons, **opt))
        assert rc == want
        S.close()
