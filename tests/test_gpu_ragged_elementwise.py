"""Elementwise launches whose rows are no whole float4, whose buffers start off a 16-byte boundary, or
whose transposed operand leaves ragged tiles, against the oracle bit for bit (tests/test_gpu_parity.py's
bars): the flat kernel's partial last unit and its gathers over one, two and more outer axes, the
tile kernel's edges, and a fused chain on each side of the sizes where it changes kernel."""
from __future__ import annotations

import numpy as np
import pytest

from cases import Arr, Case, _bshape, assert_bits
from test_gpu_parity import check_case

pytestmark = pytest.mark.gpu

FLAT = [((1,), (1,)), ((3,), (3,)), ((1025,), (1025,)), ((7, 3), (3,)), ((5, 2), (5, 1)),
        ((33, 1001), (1001,)), ((33, 1001), (33, 1)), ((4, 9, 7), (9, 1)), ((4, 9, 7), (4, 1, 7)),
        ((3, 5, 2, 7), (3, 1, 2, 1)), ((2, 3, 4, 5, 3), (2, 1, 4, 1, 3))]
# (batch, p, q): a's last two axes are swapped, so the tile runs over (q, p)
TILES = [(1, 521, 1009), (9, 257, 231), (3, 66, 2731), (100, 5, 1049)]


def _cases():
    out = []
    for i, (sa, sb) in enumerate(FLAT):
        for op in ("add", "sub", "mul", "div"):
            b = Arr(sb, "pos" if op == "div" else "special", 60 + i, requires_grad=True)
            a = Arr(sa, "special", 30 + i, requires_grad=True)
            out.append(Case(f"{op}_fwd_{sa}_{sb}", op, "fwd", [a, b], _bshape(sa, sb)))
            out.append(Case(f"{op}_bwd_{sa}_{sb}", op, "bwd", [a, b], _bshape(sa, sb), exact=sa == sb))
    for i, s in enumerate(TILES):
        v = (s[0], s[2], s[1])
        for sb in ((1, v[1], 1), (s[0], 1, v[2]), v):
            out.append(Case(f"add_tile_{s}_{sb}", "add", "fwd",
                            [Arr(s, "special", 90 + i, transpose=(1, 2)), Arr(sb, "normal", 95 + i)],
                            v))
    return out


CASES = _cases()


@pytest.mark.parametrize("c", CASES, ids=[c.id for c in CASES])
def test_ragged(c):
    check_case(c)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("n", [4, 5, 4096, 4099])
def test_misaligned_buffers(n, off):
    from plast_amd import runtime as rt
    print(f"n {n} offset {off}", flush=True)
    rng = np.random.RandomState(n + off)
    x, y = (rng.randn(n + 8).astype(np.float32) for _ in range(2))
    X, Y, O = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor.from_numpy(y), rt.DeviceTensor((n + 8,))
    views = [rt.DeviceTensor((n,), base=t, offset=o, zero=False)
             for t, o in ((X, off), (Y, 0), (O, 4 - off))]
    rt.forward("mul", views[:2], views[2])
    want = np.zeros(n + 8, np.float32)
    want[4 - off:4 - off + n] = x[off:off + n] * y[:n]
    assert_bits(O.numpy(), want, "mul into a misaligned view")


# either side of 2^18 elements (one element a lane below) and of 2^19 (the ragged tile above)
@pytest.mark.parametrize("shape", [(1, 1, 262144), (1, 1, 262145), (1, 511, 513), (1, 723, 724),
                                   (1, 724, 729), (3, 417, 425), (2, 301, 1024), (1, 801, 1003)])
def test_chain_sizes(shape):
    """(permute(a) + b) * c, then neg: the chain on whichever kernel takes its size = its ops."""
    from plast_amd import ops, runtime as rt
    b, m, n = shape
    print(f"chain {shape}", flush=True)
    rng = np.random.RandomState(b * 7 + m)
    a = rt.DeviceTensor.from_numpy(rng.randn(b, n, m).astype(np.float32))
    at = ops.transpose(a, 1, 2)
    bb = rt.DeviceTensor.from_numpy(rng.uniform(0.5, 1.5, (1, m, 1)).astype(np.float32))
    c = rng.uniform(0.5, 1.5, (b, 1, n)).astype(np.float32)
    c[..., -5:] = 0.0  # zeros of both signs, whose negation tells the NEG rule's tail
    cc = rt.DeviceTensor.from_numpy(c)
    tape = ops.make_tape([("LOAD", 0, 0, 0, 0.0), ("ADD", 1, 1, 0, 0.0), ("MUL", 1, 2, 0, 0.0),
                          ("NEG", 0, 0, 0, 0.0)], 3)
    got = ops.fused(tape, [at, bb, cc], shape).numpy()
    mid = ops.binary("mul", ops.binary("add", at, bb), cc)
    want = ops.unary("neg", mid).numpy()
    assert_bits(got, want, "fused against unfused")
