"""Device memory of contexts: sizes of large blocks, free blocks given back when an allocation fails,
bounds of what is kept, and a context that runs out of memory.  MPGPU_MEMORY_LIMIT_MB sets the most
bytes a context may have in use, so that an allocation fails without filling the card."""
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


def _context(matsto, metsol, seed=3, modules=40, tracks=400, **opt):
    rp, ii, gg = _records(seed, modules, 6, 4, tracks, 8, 2, np.float32)
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
    assert np.array_equal(x, y)
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
