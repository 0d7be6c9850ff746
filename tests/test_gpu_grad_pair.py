"""Both gradients of a binary op in one pass, against the oracle bit for bit: sizes around a float4 and
a workgroup, signed zeros (the B-gradient of sub and div starts from 0 - g inside the reference's SIMD
blocks), one tensor as both operands, gradients that share a buffer, and one gradient wanted alone."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from cases import BINARY, Arr, Case, assert_bits
from test_gpu_parity import check_case

pytestmark = pytest.mark.gpu

SHAPES = [(1,), (3,), (4,), (9,), (1023,), (1025,), (3, 5, 7), (64, 65), (257, 1024)]


def _cases():
    out = []
    for i, s in enumerate(SHAPES):
        for op in BINARY:
            for ga, gb in ((True, True), (True, False), (False, True)):
                dist = "special" if op != "div" else "normal"
                out.append(Case(f"{op}_{s}_{ga}_{gb}", op, "bwd",
                                [Arr(s, dist, 10 + i, requires_grad=ga),
                                 Arr(s, "pos" if op == "div" else dist, 30 + i, requires_grad=gb)], s,
                                grad_init=50 + i if ga and gb else None))
    for op in BINARY:
        out.append(Case(f"{op}_same", op, "bwd", [Arr((33,), "pos", 7, requires_grad=True)] * 2, (33,),
                        same_input=True))
    return out


CASES = _cases()


@pytest.mark.parametrize("c", CASES, ids=[c.id for c in CASES])
def test_pair(c):
    check_case(c)


def test_overlapping_gradients_run_in_turn():
    """b's gradient starts four elements into a's: the second pass adds to what the first left."""
    from plast_amd import runtime as rt
    n = 1000
    rng = np.random.RandomState(0)
    x, y, g, d = (rng.randn(n + 4).astype(np.float32) for _ in range(4))
    a, b = rt.DeviceTensor.from_numpy(x[:n]), rt.DeviceTensor.from_numpy(y[:n])
    out = rt.DeviceTensor((n,), requires_grad=True)
    rt.lib().arena_memcpy_h2d_hip(out.grad.ptr, g.ctypes.data, 4 * n)
    D = rt.DeviceTensor.from_numpy(d)
    grads = [rt.DeviceTensor((n,), base=D, offset=o, zero=False) for o in (0, 4)]
    for t, gr in zip((a, b), grads):
        t.t.requires_grad = True
        t.t.grad = C.pointer(gr.t)
    rt.backward("mul", [a, b], out)
    want = d.copy()
    want[:n] += g[:n] * y[:n]
    want[4:n + 4] += g[:n] * x[:n]
    assert_bits(D.numpy(), want, "shared gradient buffer")
