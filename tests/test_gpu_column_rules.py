"""Leading-axis reductions on each side of the sizes where their kernel changes (launch_rules.hpp):
one-launch slices, the flat array, one and four columns a lane, one and several chunks. Forwards
against the oracle at the bars of tests/test_gpu_parity.py; the one-pass epilogue and the gradient
of a broadcast operand against the sum of their terms in 64 bits (1e-5 of the terms' magnitudes)."""
from __future__ import annotations

import numpy as np
import pytest

from cases import REDUCE, Arr, Case, _red_shape
from test_gpu_parity import check_case

pytestmark = pytest.mark.gpu

# (outer, len, inner)
COLS = [(1, 47, 64), (1, 48, 65), (1, 6144, 12), (1, 6145, 12), (130, 100, 10), (257, 100, 10),
        (1024, 128, 9), (1025, 128, 8), (1025, 256, 3), (20000, 3, 10), (2048, 5, 65), (2047, 5, 65),
        (16, 1000, 30), (1, 2048, 257), (1, 5800, 1001), (3, 900, 300)]


@pytest.mark.parametrize("i, s, op", [(i, s, op) for i, s in enumerate(COLS) for op in REDUCE + ["argmax"]])
def test_forward(i, s, op):
    check_case(Case(f"{op}_cols_{s}", op, "fwd", [Arr(s, "special", 140 + i)], _red_shape(s, 1, 0),
                    (1, 0, 0.0), "i64" if op == "argmax" else "f32"))


ROWS = [(23, 300), (24, 301), (63, 3), (64, 3), (1536, 301), (1537, 30), (1537, 64), (2049, 64),
        (2048, 16), (700, 512), (4096, 128), (4097, 100), (6000, 1000)]


@pytest.mark.parametrize("rows, cols", ROWS)
def test_epilogue_and_gradients(rows, cols):
    from plast_amd import runtime as rt
    print(f"[{rows}, {cols}]", flush=True)
    rng = np.random.RandomState(rows + cols)
    g, z = (rng.randn(rows, cols).astype(np.float32) for _ in range(2))
    G, Z, DC, DB = rt.DeviceTensor.from_numpy(g), rt.DeviceTensor.from_numpy(z), rt.DeviceTensor((rows, cols)), rt.DeviceTensor((cols,))
    L = rt.lib()
    L.relu_grad_modulate_bias_grad_hip(G.ptr, Z.ptr, DC.ptr, DB.ptr, rows * cols, cols, 0.25)
    L.check("epilogue")
    dc = g * np.where(z > 0, np.float32(1), np.float32(0.25))
    assert np.array_equal(DC.numpy(), dc)

    def close(got, terms):
        terms = terms.astype(np.float64)
        assert np.all(np.abs(got - terms.sum(0)) <= 1e-5 * np.abs(terms).sum(0))
    close(DB.numpy(), dc)
    b = rng.uniform(0.5, 1.5, cols).astype(np.float32)
    out = rt.DeviceTensor((rows, cols), requires_grad=True)
    L.arena_memcpy_h2d_hip(out.grad.ptr, g.ctypes.data, g.nbytes)
    for op, terms in (("add", g), ("mul", g * z), ("div", -(g * z) / (b * b))):
        B = rt.DeviceTensor.from_numpy(b, requires_grad=True)
        rt.backward(op, [Z, B], out)
        close(B.grad.numpy(), terms)
