"""Reductions over rows and columns of any extent and alignment, against the oracle at the bars of
tests/test_gpu_parity.py: short rows on each of their lane counts, rows with a partial last unit,
narrow columns read as one flat array (with and without chunks, over the widths whose whole rows fill
the workgroup differently), wide columns with a partial last unit, and each one's redo of the values
(NaN, signed zeros, infinities, ties, overflowing sums) that the fast order may not decide."""
from __future__ import annotations

import numpy as np
import pytest

from cases import REDUCE, Arr, Case, _red_shape
from test_gpu_parity import check_case
from test_gpu_sum_overflow import _check, _lines

pytestmark = pytest.mark.gpu

OPS = REDUCE + ["argmax"]
ROWS = [(1, 1), (5, 2), (7, 3), (64, 5), (33, 31), (70, 32), (9, 33), (65, 77), (17, 128), (18, 129),
        (7, 511), (6, 512), (5, 513), (3, 1001), (2, 9001)]
# (outer, len, inner): narrow columns, then wide ones
COLS = [(1, 1, 3), (1, 700, 1), (3, 40, 2), (1, 5000, 3), (1, 60000, 10), (2, 300, 77), (1, 9000, 77),
        (1, 64, 129), (1, 3000, 171), (1, 40, 255), (1, 6000, 254), (2, 100, 256), (1, 90, 257),
        (1, 1000, 261), (2, 30, 1027), (1, 5000, 515), (1, 17, 300), (2, 63, 1003)]


def _cases():
    out = []
    for i, s in enumerate(ROWS):
        for op in OPS:
            for d in ("special", "ties"):
                out.append(Case(f"{op}_rows_{s}_{d}", op, "fwd", [Arr(s, d, 10 + i)], _red_shape(s, 1, 0),
                                (1, 0, 0.0), "i64" if op == "argmax" else "f32"))
    # argmax rows on each side of their lane counts' lines
    for i, s in enumerate([(99, 16), (99, 17), (99, 64), (8192, 65), (8192, 128), (8193, 65), (8193, 128), (8193, 129)]):
        for d in ("special", "ties"):
            out.append(Case(f"argmax_rows_{s}_{d}", "argmax", "fwd", [Arr(s, d, 30 + i)], _red_shape(s, 1, 0),
                            (1, 0, 0.0), "i64"))
    for i, s in enumerate(COLS):
        for op in OPS:
            for d in ("special", "normal"):
                out.append(Case(f"{op}_cols_{s}_{d}", op, "fwd", [Arr(s, d, 40 + i)], _red_shape(s, 1, 0),
                                (1, 0, 0.0), "i64" if op == "argmax" else "f32"))
    for i, s in enumerate([(3, 5), (9, 33), (65, 77), (18, 129), (5, 513), (3, 1001)]):
        for op in REDUCE:
            for d in ("normal", "ties", "special"):
                out.append(Case(f"{op}_rows_bwd_{s}_{d}", op, "bwd", [Arr(s, d, 70 + i, requires_grad=True)],
                                _red_shape(s, 1, 0), (1, 0, 0.0)))
    for i, s in enumerate([(2, 40, 3), (1, 300, 77), (1, 90, 257)]):
        for op in REDUCE:
            out.append(Case(f"{op}_cols_bwd_{s}", op, "bwd", [Arr(s, "ties", 80 + i, requires_grad=True)],
                            _red_shape(s, 1, 0), (1, 0, 0.0)))
    # max/min backward over rows on each thread count and loop trip of its kernel, and past them
    for i, s in enumerate([(3, 1025), (3, 2047), (5, 2048), (3, 2049), (2, 4099), (2, 16387), (2, 32768), (2, 32769),
                           (257, 32769), (70, 128), (70, 1024)]):
        for op in ("max", "min"):
            for d in ("ties", "special"):
                out.append(Case(f"{op}_rows_bwd_{s}_{d}", op, "bwd", [Arr(s, d, 90 + i, requires_grad=True)],
                                _red_shape(s, 1, 0), (1, 0, 0.0)))
    return out


CASES = _cases()


@pytest.mark.parametrize("c", CASES, ids=[c.id for c in CASES])
def test_ragged_reduction(c):
    check_case(c)


@pytest.mark.parametrize("op", ["sum", "mean"])
@pytest.mark.parametrize("n, count, dim", [(30, 24, 1), (77, 24, 1), (300, 12, 1), (1001, 12, 1),
                                           (60, 12, 0), (3000, 10, 0), (20000, 6, 0), (500, 259, 0)])
def test_overflowing_sums(op, n, count, dim):
    """Sums whose order decides a non-finite outcome follow the reference's order."""
    print(f"{op} {n} x {count} dim {dim}", flush=True)
    x = _lines(n, count, np.random.RandomState(n))
    _check(x if dim == 1 else np.ascontiguousarray(x.T), op, dim)


@pytest.mark.parametrize("off", [1, 3])
@pytest.mark.parametrize("shape, dim", [((40, 77), 1), ((6, 1000), 1), ((50, 12), 0), ((40, 300), 0)])
def test_misaligned_input(shape, dim, off):
    from plast_amd import runtime as rt
    from plast_amd.abi import KernelParams
    print(f"{shape} dim {dim} offset {off}", flush=True)
    n = int(np.prod(shape))
    x = np.random.RandomState(n + off).randn(n + off).astype(np.float32)
    X = rt.DeviceTensor.from_numpy(x)
    v = rt.DeviceTensor(shape, base=X, offset=off, zero=False)
    out = rt.DeviceTensor((shape[1 - dim],), zero=False)
    for op in ("sum", "max"):
        rt.forward(op, [v], out, KernelParams(dim, 0, 0.0))
        h = x[off:].reshape(shape)
        if op == "max":
            assert np.array_equal(out.numpy(), h.max(axis=dim))
        else:
            bar = 1e-5 * np.abs(h).astype(np.float64).sum(axis=dim)
            assert np.all(np.abs(out.numpy() - h.astype(np.float64).sum(axis=dim)) <= bar)


@pytest.mark.parametrize("op", ["max", "min"])
@pytest.mark.parametrize("shape", [(40, 9), (20, 300), (7, 1500), (5, 3000), (2, 40000)])
def test_extreme_backward_strided_and_constant(shape, op):
    """Max/min backward in its one read over a window of a wider matrix whose gradient is a window of
    another, and over rows of one value, all of it ties: every element gets dout / n, and what lies
    between the rows stays as it was."""
    from plast_amd import abi, runtime as rt
    from plast_amd.abi import KernelParams
    print(f"{op} {shape}", flush=True)
    rows, cols = shape
    rng = np.random.RandomState(cols)
    x = rng.randint(-2, 3, (rows, cols + 5)).astype(np.float32)
    x[0] = x[rows // 2] = 1.0
    d0 = rng.randn(rows, cols + 9).astype(np.float32)
    dout = rng.randn(rows).astype(np.float32)
    X, D = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor.from_numpy(d0)
    gt = abi.make_tensor(D.ptr + 7 * 4, shape, (cols + 9, 1), rt.FLOAT32)
    v = abi.make_tensor(X.ptr + 3 * 4, shape, (cols + 5, 1), rt.FLOAT32, rt.GPU, True, gt)
    out = rt.DeviceTensor((rows,), requires_grad=True)
    rt.lib().arena_memcpy_h2d_hip(out.grad.ptr, dout.ctypes.data, dout.nbytes)
    p = KernelParams(1, 0, 0.0)
    rt.forward(op, [v], out, p)
    rt.backward(op, [v], out, p)
    w = x[:, 3:3 + cols]
    tie = w == getattr(w, op)(1)[:, None]
    want = d0.copy()
    add = (dout / tie.sum(1, dtype=np.float32)).astype(np.float32)
    want[:, 7:7 + cols] = np.where(tie, d0[:, 7:7 + cols] + add[:, None], d0[:, 7:7 + cols])
    assert np.array_equal(D.numpy(), want)
