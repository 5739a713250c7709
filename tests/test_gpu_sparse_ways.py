"""Which way the device sparse() takes: few triples, triples in no order and
columns too long go to the radix sort, runs of one column to the wavefront per
column.  Every input is bitwise the oracle's sparse() whichever it is: around
the least number of triples, in wide matrices, with runs that a look at a part
of the triples shows and the whole does not have, and the other way round."""
import ctypes

import numpy as np
import pytest

import oracle as O
from feasm import _lib as L
from feasm import core
from test_gpu_device_entry_points import DeviceBuffers
from test_gpu_sparse_runs import check, runs

pytestmark = pytest.mark.gpu

LEAST = 1 << 16  # triples from which runs are looked for


def values(rng, n):
    return rng.uniform(-1.0, 1.0, n) * 10.0 ** rng.integers(-8, 9, n)


def in_runs(rng, nt, n, length):
    J = np.repeat(rng.integers(1, n + 1, -(-nt // length)), length)[:nt]
    return rng.integers(1, n + 1, nt), J


@pytest.mark.parametrize("nt", [LEAST - 1, LEAST, LEAST + 1, 3 * LEAST + 17])
@pytest.mark.parametrize("length", [1, 3, 4, 5, 24, 64, 100])
def test_run_lengths_around_the_least_number(ctx, nt, length):
    rng = np.random.default_rng(nt + length)
    I, J = in_runs(rng, nt, 700, length)
    check(ctx, I, J, values(rng, nt), 700, 700)


@pytest.mark.parametrize("longest", [1, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 3000])
@pytest.mark.parametrize("filler", [False, True])
def test_column_lengths(ctx, longest, filler):
    """Few triples of a wide matrix; and among enough others."""
    rng = np.random.default_rng(longest)
    n = 40
    lengths = rng.integers(0, longest + 1, n)
    lengths[[0, 7, n - 1]] = 0, longest, longest
    I, J, V = runs(rng, np.arange(1, n + 1), lengths, max(1, longest // 3))
    if filler:
        i, j = in_runs(rng, LEAST, 900, 24)
        I, J, V = np.r_[I, i], np.r_[J, j + 50], np.r_[V, values(rng, LEAST)]
        check(ctx, I, J, V, 1100, 1000)
    else:
        check(ctx, I, J, V, max(1, longest // 3) + 2, n + len(V) + 3)


def test_runs_only_where_one_looks(ctx):
    """Every fourth stretch of 64 is looked at: runs there and nowhere else, and the reverse."""
    rng = np.random.default_rng(8)
    nt = 64 * 1024
    J = rng.integers(1, 3001, nt).reshape(-1, 64)
    for looked in (True, False):
        K = J.copy()
        at = (np.arange(1024) % 4 == 0) == looked
        K[at] = np.repeat(rng.integers(1, 3001, (int(at.sum()), 2)), 32, axis=1)
        check(ctx, rng.integers(1, 3001, nt), K.ravel(), values(rng, nt), 3000, 3000)


@pytest.mark.parametrize("columns", [1, 20])
def test_few_columns(ctx, columns):
    rng = np.random.default_rng(columns)
    nt = 2 * LEAST
    J = np.repeat(np.arange(1, columns + 1), nt // columns)
    check(ctx, rng.integers(1, 5001, len(J)), J, values(rng, len(J)), 5000, 5000)


@pytest.mark.parametrize("bad", ["row", "column", "column of few"])
def test_indices_out_of_range(ctx, hiprt, bad):
    rng = np.random.default_rng(5)
    I, J = in_runs(rng, LEAST + 100 if bad != "column of few" else 500, 400, 24)
    i0, j0 = (I - 1).astype(np.int32), (J - 1).astype(np.int32)
    n = 400 if bad != "column of few" else 1000
    if bad == "row":
        i0[333] = n
    else:
        j0[333] = -1
    buf = DeviceBuffers(hiprt)
    try:
        d = [buf.upload(a) for a in (i0, j0, values(rng, len(i0)))]
        h = ctypes.c_void_p()
        rc = L.lib().feasm_sparse_device(ctx.h, len(i0), *d, n, n, ctypes.byref(h))
    finally:
        buf.free()
    assert rc == L.EDOF and not h.value


@pytest.mark.parametrize("length", [30, 200, 256, 257, 500, 600, 1024])
@pytest.mark.parametrize("span", [(1 << 21) - 2, (1 << 21) + 5, (1 << 23) - 2, (1 << 23) + 5, (1 << 26) + 1])
def test_rows_far_apart_beside_others(ctx, length, span):
    """Some columns have rows too far apart for 31-bit keys (20 bits and more
    beside the place in the column), the others do not."""
    rng = np.random.default_rng(length)
    I, J, V = runs(rng, np.arange(1, 9), [length] * 8, 50)
    far = [np.flatnonzero(J == c)[-1] for c in (2, 5, 8)]
    I[far] = span
    I[np.flatnonzero(J == 3)[0]] = span  # at the front of a column
    i, j = in_runs(rng, LEAST, 900, 24)
    order = rng.permutation(2)
    parts = [(I, J, V), (i, j + 8, values(rng, LEAST))]
    I, J, V = (np.concatenate([parts[k][x] for k in order]) for x in range(3))
    check(ctx, I, J, V, span, 910)


@pytest.mark.parametrize("lengths", [[1025], [1024, 1025, 5000], [3000] * 9, [40000]])
@pytest.mark.parametrize("where", ["first", "last", "spread"])
def test_long_columns_beside_others(ctx, lengths, where):
    """Columns of more than 1024 triples are sorted apart from the others."""
    rng = np.random.default_rng(len(lengths))
    n = 5000
    at = {"first": np.arange(len(lengths)), "last": n - 1 - np.arange(len(lengths)),
          "spread": 3 + 500 * np.arange(len(lengths))}[where]
    I, J, V = runs(rng, at + 1, lengths, 700)
    i, j = in_runs(rng, LEAST, n, 24)
    parts = [(I, J, V), (i, j, values(rng, LEAST))]
    for order in ([0, 1], [1, 0]):
        a, b, c = (np.concatenate([parts[k][x] for k in order]) for x in range(3))
        check(ctx, a, b, c, n, n)


@pytest.mark.parametrize("share", [1, 3])
def test_most_triples_in_long_columns(ctx, share):
    """Up to half of the triples in long columns, and more than that."""
    rng = np.random.default_rng(share)
    nt = 40000 * share
    I, J = rng.integers(1, 901, nt), np.repeat(rng.integers(1, 8, nt // 16), 16)
    i, j = in_runs(rng, LEAST, 900, 24)
    check(ctx, np.r_[i, I], np.r_[j + 50, J], values(rng, nt + LEAST), 900, 1000)


def test_row_out_of_range_in_a_long_column(ctx, hiprt):
    rng = np.random.default_rng(6)
    i, j = in_runs(rng, LEAST, 400, 24)
    i0 = np.r_[i, rng.integers(1, 401, 2000)].astype(np.int32) - 1
    j0 = np.r_[j, np.full(2000, 17)].astype(np.int32) - 1
    i0[-5] = 400
    buf = DeviceBuffers(hiprt)
    try:
        d = [buf.upload(a) for a in (i0, j0, values(rng, len(i0)))]
        h = ctypes.c_void_p()
        rc = L.lib().feasm_sparse_device(ctx.h, len(i0), *d, 400, 400, ctypes.byref(h))
    finally:
        buf.free()
    assert rc == L.EDOF and not h.value
