"""Distance rows copied to the host around the sizes where the copy changes
(pages asked for from 32 KiB, one or two 4 MiB pieces, more than two), into
ordinary memory at odd addresses, into pinned memory, and several rows of a
serving launch at once.  Every word is compared; the words beside the row keep
their values."""
import contextlib
import ctypes
import sys

import numpy as np
import pytest

from hip_rt import hip
from mlmq_tpds_withl3_amd import Solver
from mlmq_tpds_withl3_amd._lib import check
from mlmq_tpds_withl3_amd.serve import Server

pytestmark = pytest.mark.gpu
UNREACHED = 0x7FFFFFFF
PIECE = (4 << 20) // 4


def say(msg):
    print(f"[gpu-row-copy] {msg}", flush=True)
    sys.stdout.flush()


@contextlib.contextmanager
def pinned(n):
    """n words of pinned memory, each -7."""
    p = ctypes.c_void_p()
    assert hip().hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(4 * n), ctypes.c_uint(0)) == 0
    row = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_int32)), shape=(n,))
    row[:] = -7
    yield row
    assert hip().hipHostFree(p) == 0


def stars(n):
    """Vertex i % 1000 == 0 has an edge of weight i + 1 from vertex 0."""
    heads = np.arange(1000, n, 1000)
    row = np.full(n + 1, len(heads), dtype=np.int64)
    row[0] = 0
    expect = np.full(n, UNREACHED, dtype=np.int32)
    expect[0] = 0
    expect[heads] = heads + 1
    return row, heads.astype(np.int32), (heads + 1).astype(np.int32), expect


@pytest.mark.parametrize("n", [1, 1001, 8191, 8193, PIECE - 1, PIECE, PIECE + 1, 2 * PIECE, 2 * PIECE + 1, 3 * PIECE + 7])
def test_sizes(n):
    say(f"{n} words")
    row, col, w, expect = stars(n)
    s = Solver(0)
    s.load_csr(row, col, w)
    s.solve(0, timeout_s=20.0)
    assert np.array_equal(s.dist(), expect)
    # at an odd word of a larger array
    around = np.full(n + 64, -7, dtype=np.int32)
    check(s._L.mlmq_copy_dist(s._h, around[33:].ctypes.data), s._h)
    assert np.array_equal(around[33:33 + n], expect)
    assert (around[:33] == -7).all() and (around[33 + n:] == -7).all()
    with pinned(n + 2) as row:
        check(s._L.mlmq_copy_dist(s._h, row[1:].ctypes.data), s._h)
        assert np.array_equal(row[1:-1], expect)
        assert row[0] == -7 and row[-1] == -7
    s.close()


def test_rows_of_a_launch():
    say("rows of a serving launch")
    s = Server(0, hbm_budget=1 << 30, timeout_s=20.0)
    graphs = [stars(n) for n in (1001, PIECE + 5, 2 * PIECE + 9)]
    for g in graphs:
        s.add_graph(g[:3])
    which = np.array([2, 0, 1, 0, 2, 1, 1], dtype=np.int32)
    rows = [np.full(len(graphs[g][3]), -1, dtype=np.int32) for g in which]
    with pinned(len(rows[3])) as rows[3]:
        res, _ = s.run(np.zeros(len(which)), which, np.zeros(len(which), dtype=np.int32), dist_out=rows)
        assert (res["status"] == 0).all()
        for g, row in zip(which, rows):
            assert np.array_equal(row, graphs[g][3])
    s.close()
