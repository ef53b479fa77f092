"""Device memory of contexts: sizes of large blocks, free blocks given back when an allocation fails,
bounds of what is kept, a context that runs out of memory, and what a pass does without when memory is
short.  MPGPU_MEMORY_LIMIT_MB sets the most bytes a context may have in use (read when it is made and
when its options are set), so that an allocation fails without filling the card."""
import os
import re

import numpy as np
import pytest

import mpgpu
from test_gpu_rows import _records

pytestmark = pytest.mark.gpu
LINE = r"device memory after (.*): (\d+) bytes in use, (\d+) at most, (\d+) kept, (\d+) of ended contexts"


@pytest.fixture
def memory(monkeypatch, capfd):
    """the lines of the calls since the last one: (call, in use, at most, kept, of ended contexts)"""
    monkeypatch.setenv("MPGPU_VERBOSE", "1")
    capfd.readouterr()
    return lambda: [(m[0], *map(int, m[1:])) for m in re.findall(LINE, capfd.readouterr().err)]


def _context(matsto, metsol, seed=3, modules=40, tracks=400, nloc=4, **opt):
    rp, ii, gg = _records(seed, modules, 6, nloc, tracks, 8, 2, np.float32)
    P = mpgpu.Pede(matsto=matsto, metsol=metsol, mreqenf=1, mcount=1, **opt)
    P.add_records(rp, ii, gg)
    labels = np.array([100 * (m + 1) + k + 1 for m in range(modules) for k in range(6)], np.int32)
    P.set_steering_parameters(labels, np.zeros(len(labels)), np.full(len(labels), 0.1))
    P.build_structure()
    return P


def _iteration(P):
    P.loopn()
    return P.solve()[0]


def test_large_blocks_have_their_own_size(memory):
    """One more parameter takes n + 1 more words of a packed matrix of 288 MB, not another step of
    the size classes (32 MB there) that are for blocks which may be kept."""
    used = []
    for n in (8688, 8689):
        P = mpgpu.Pede(matsto=mpgpu.FULL, metsol=mpgpu.INVERSION, mreqenf=0, mcount=1)
        labels = np.arange(1, n + 1, dtype=np.int32) + 1000
        P.add_records(np.array([0, 6]), np.array([0, 0, 1, 0, 1001, 1002], np.int32),
                      np.array([0.0, 0.1, 1.0, 0.5, 1.0, 1.0], np.float32))
        P.set_steering_parameters(labels, np.zeros(n), np.full(n, 0.1))
        P.build_structure()
        assert P.nvar == n
        used.append(memory()[0][1])
        P.close()
    assert 0 < used[1] - used[0] < 1 << 20


@pytest.mark.parametrize("matsto,metsol", [(mpgpu.FULL, mpgpu.INVERSION), (mpgpu.SPARSE, mpgpu.MINRES)])
def test_kept_blocks_are_given_back_when_memory_is_short(memory, monkeypatch, matsto, metsol):
    """With the context's own maximum as limit the same calls give the same numbers: free blocks of the
    context, and those of ended ones, make room."""
    P = _context(matsto, metsol)
    x = _iteration(P)
    lines = memory()
    P.close()
    assert len(lines) == 2 and lines[1][3] > 0          # blocks were kept
    monkeypatch.setenv("MPGPU_MEMORY_LIMIT_MB", repr(lines[1][2] / (1 << 20)))
    Q = _context(matsto, metsol)
    y = _iteration(Q)
    lines2 = memory()
    Q.close()
    # (with full storage the records may then be left to atomic additions)
    assert np.array_equal(x, y) if matsto == mpgpu.SPARSE else np.allclose(x, y, rtol=1e-9, atol=1e-9 * np.abs(x).max())
    assert lines2[1][2] <= lines[1][2] and lines2[1][1] + lines2[1][3] <= lines[1][2]


def test_out_of_memory_is_an_error_and_the_next_context_works(memory, monkeypatch):
    P = _context(mpgpu.SPARSE, mpgpu.MINRES)
    x = _iteration(P)
    used = memory()[0][1]
    P.close()
    monkeypatch.setenv("MPGPU_MEMORY_LIMIT_MB", repr(0.5 * used / (1 << 20)))
    with pytest.raises(mpgpu.MpgpuError) as e:
        _context(mpgpu.SPARSE, mpgpu.MINRES)
    assert e.value.code == 30
    monkeypatch.delenv("MPGPU_MEMORY_LIMIT_MB")
    Q = _context(mpgpu.SPARSE, mpgpu.MINRES)
    assert np.array_equal(_iteration(Q), x)
    Q.close()


def test_contexts_reuse_memory_within_its_bounds(memory):
    """Contexts of other sizes in turn: what one leaves is used by the next ones with the same results,
    at most 2 GB are kept by a context and 4 GB of ended ones."""
    first = {}
    for turn in range(3):
        for modules in (20, 90, 45):
            P = _context(mpgpu.FULL, mpgpu.INVERSION, modules=modules, seed=modules)
            x = _iteration(P)
            P.close()
            assert np.array_equal(first.setdefault(modules, x), x)
    lines = memory()
    assert len(lines) == 18
    assert max(q[3] for q in lines) <= 2 << 30 and max(q[4] for q in lines) <= 4 << 30
    assert lines[-1][4] > 0 and lines[-1][4] <= 2 * max(q[4] for q in lines[:6])


def _pass_of(P):
    P.loopn()
    return P.vector()[0], P.matrix_packed()


def test_units_of_a_pass_make_room_for_the_solve(memory, monkeypatch):
    """The units of records in row form are scratch memory of a pass: when a solve does not find the memory
    it needs they go, and the next pass makes them again."""
    args = dict(modules=150, tracks=4000)
    P = _context(mpgpu.FULL, mpgpu.INVERSION, **args)
    x = _iteration(P)
    (_, _, peak1, _, _), (_, use2, peak2, _, _) = memory()
    P.loopn()
    units = 4000 * 8 * 128
    limit = peak2 - units // 2
    assert limit > peak1
    monkeypatch.setenv("MPGPU_MEMORY_LIMIT_MB", repr(limit / (1 << 20)))
    P.set_options()
    y, _ = P.solve()
    line = memory()[-1]
    assert np.array_equal(x, y) and line[1] <= use2 - units
    P.loopn()
    assert np.array_equal(P.solve()[0], x)
    P.close()


def test_pass_without_room_for_units(memory, monkeypatch):
    """With full storage the record kernel takes the records when there is no memory for their units (the
    bar of the other passes: only the order of sums differs)."""
    P = _context(mpgpu.FULL, mpgpu.INVERSION, modules=150, tracks=4000)
    use = memory()[0][1]
    v, A = _pass_of(P)
    monkeypatch.setenv("MPGPU_MEMORY_LIMIT_MB", repr((use - 4000 * 8 * 64) / (1 << 20)))
    P.set_options()
    P.solve()                           # takes the units' memory
    w, B = _pass_of(P)
    assert not np.array_equal(A, B)     # (atomic additions)
    assert np.abs(v - w).max() <= 1e-10 * np.abs(v).max() and np.abs(A - B).max() <= 1e-10 * np.abs(A).max()
    monkeypatch.delenv("MPGPU_MEMORY_LIMIT_MB")
    P.set_options()
    w, B = _pass_of(P)
    assert np.array_equal(v, w) and np.array_equal(A, B)
    P.close()


def test_full_storage_without_room_for_lists(monkeypatch, capfd):
    """... and from the start when the lists would take more than half of what the matrix and its solve
    leave."""
    monkeypatch.setenv("MPGPU_VERBOSE", "1")
    P = _context(mpgpu.FULL, mpgpu.INVERSION, modules=20, tracks=4000)
    v, A = _pass_of(P)
    err = capfd.readouterr().err
    assert "records in row form: 4000 in 1 batches, by the record kernel: 0 in 0" in err
    use = int(re.findall(LINE, err)[0][1])
    P.close()
    monkeypatch.setenv("MPGPU_MEMORY_LIMIT_MB", repr(use / (1 << 20)))
    P = _context(mpgpu.FULL, mpgpu.INVERSION, modules=20, tracks=4000)
    w, B = _pass_of(P)
    assert "records in row form: 0 in 0 batches, by the record kernel: 4000 in 1" in capfd.readouterr().err
    assert np.abs(v - w).max() <= 1e-10 * np.abs(v).max() and np.abs(A - B).max() <= 1e-10 * np.abs(A).max()
    P.close()


@pytest.mark.parametrize("modules,defect", [(22, False), (22, True), (150, False)])
def test_inversion_without_room_for_the_square_matrix(memory, monkeypatch, modules, defect):
    """The square copy of the matrix (16 n^2 / 2 bytes) does not fit beside the packed one and its copy: one
    pivot at a time in the packed matrix, with the same pivots, so the same rank, and the same solution and
    inverse but for rounding.  (defect: parameters that nothing determines.)"""
    def context():
        # (6 local parameters: no units whose memory could be had instead)
        P = _context(mpgpu.FULL, mpgpu.INVERSION, modules=modules, tracks=1000, nloc=6)
        P.loopn()
        if defect:
            # the last module's rows and columns away
            A = P.matrix_packed()
            n = P.nall
            i = np.arange(n - 6, n)
            rows = np.concatenate([np.full(k + 1, k) for k in i])
            cols = np.concatenate([np.arange(k + 1) for k in i])
            P.mupdat(rows + 1, cols + 1, -A[rows * (rows + 1) // 2 + cols])
        return P

    P = context()
    x, st = P.solve()
    err, gcor = P.errors()
    P.close()
    use = memory()[1][1]
    n, packed = P.nall, 4 * P.nall * (P.nall + 1)
    Q = context()
    assert Q.nall == n > 128
    monkeypatch.setenv("MPGPU_MEMORY_LIMIT_MB", repr((use + packed + 4 * n * n) / (1 << 20)))
    Q.set_options()
    y, st2 = Q.solve()
    e2, g2 = Q.errors()
    Q.close()
    assert st["nrank"] == st2["nrank"] == n - (6 if defect else 0)
    # REAL(4) errors; the condition of these systems is below 1e4
    assert np.abs(x - y).max() <= 1e-10 * np.abs(x).max()
    assert np.allclose(err, e2, rtol=1e-6) and np.allclose(gcor, g2, rtol=1e-5, atol=1e-6)
