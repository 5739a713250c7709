"""The device sparse() on triples that come in runs of one column (the
wavefront-per-column way) and at its limits, where it hands over to the radix
sort: bitwise the oracle's sparse() -- the same left fold in input order."""
import ctypes

import numpy as np
import pytest

import oracle as O
from feasm import _lib as L
from feasm import core
from test_gpu_device_entry_points import DeviceBuffers

pytestmark = pytest.mark.gpu


def check(ctx, I, J, V, m, n):
    got = core.sparse(ctx, I, J, V, m, n).csc_arrays(1)
    ref = O.sparse(I, J, V, m, n)
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)


def runs(rng, columns, lengths, rows, span=0):
    """Shuffled runs: column j gets lengths[j] triples in runs of up to 24."""
    parts = []
    for j, total in zip(columns, lengths):
        while total > 0:
            k = int(min(total, rng.integers(5, 25)))
            parts.append((np.full(k, j), rng.integers(0, rows, k) + 1))
            total -= k
    rng.shuffle(parts)
    J = np.concatenate([p[0] for p in parts])
    I = np.concatenate([p[1] for p in parts])
    if span:  # one far row in every column
        last = {j: t for t, j in enumerate(J)}
        I[list(last.values())] = span
    return I, J, rng.uniform(-1.0, 1.0, len(I)) * 10.0 ** rng.integers(-8, 9, len(I))


@pytest.mark.parametrize("longest", [1, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 3000])
def test_column_lengths(ctx, longest):
    rng = np.random.default_rng(longest)
    n = 40
    lengths = rng.integers(0, longest + 1, n)
    lengths[[0, 7, n - 1]] = 0, longest, longest  # an empty first column, and full ones
    I, J, V = runs(rng, np.arange(1, n + 1), lengths, max(1, longest // 3))
    check(ctx, I, J, V, max(1, longest // 3) + 2, n + 3)


@pytest.mark.parametrize("length,span", [(200, (1 << 23) - 2), (200, (1 << 23) + 5), (600, (1 << 21) - 2),
                                         (600, (1 << 21) + 5)])
def test_row_spans(ctx, length, span):
    rng = np.random.default_rng(3)
    I, J, V = runs(rng, np.arange(1, 6), [length] * 5, 50, span)
    check(ctx, I, J, V, span, 6)


def test_single_triples_and_one_long_run(ctx):
    rng = np.random.default_rng(4)
    I, J = rng.integers(1, 30, 5000), rng.integers(1, 50, 5000)
    check(ctx, I, J, rng.uniform(-1, 1, 5000), 30, 50)  # no runs
    check(ctx, I, np.full(5000, 2), rng.uniform(-1, 1, 5000), 30, 50)  # one column
    check(ctx, I[:1], J[:1], np.array([0.0]), 30, 50)
    check(ctx, np.repeat(I[:8], 6), np.repeat(J[:8], 6), np.zeros(48), 30, 50)  # explicit zeros stay


def test_indices_out_of_range_in_runs(ctx, hiprt):
    I, J, V = runs(np.random.default_rng(5), np.arange(1, 9), [100] * 8, 40)
    for bad in ("row", "column"):
        i0, j0 = (I - 1).astype(np.int32), (J - 1).astype(np.int32)
        if bad == "row":
            i0[333] = 40
        else:
            j0[333] = 8
        buf = DeviceBuffers(hiprt)
        try:
            d = [buf.upload(a) for a in (i0, j0, V)]
            h = ctypes.c_void_p()
            rc = L.lib().feasm_sparse_device(ctx.h, len(V), *d, 40, 8, ctypes.byref(h))
        finally:
            buf.free()
        assert rc == L.EDOF and not h.value
