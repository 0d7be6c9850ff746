"""Reductions over several axes that do not merge into one (a bias gradient over batch and space, a
whole-tensor reduction of a permuted view), and gradients written along a permuted operand's own
memory order, against the oracle at the bars of tests/test_gpu_parity.py: runs of whole and broken
float4, one run or many per wave, segments with a finalize, an innermost kept axis, and the values
(signed zeros, infinities, NaN, ties) whose order decides max, min and argmax."""
from __future__ import annotations

import pytest

from cases import REDUCE, Arr, Case, _bshape
from plast_amd.abi import DIM_ALL
from test_gpu_parity import check_case

pytestmark = pytest.mark.gpu

# (a, b): b's gradient sums over every axis where b has extent 1
BCAST = [
    ((5, 3, 8), (1, 3, 1)),            # runs shorter than a wave's unit
    ((7, 4, 33), (1, 4, 1)),           # broken float4
    ((64, 6, 260), (1, 6, 1)),         # one wave per segment, several runs per segment
    ((300, 2, 1028), (1, 2, 1)),       # few outputs: segments and the finalize
    ((9, 5, 3, 7), (1, 5, 1, 1)),      # the two innermost merge
    ((6, 5, 4, 3, 8), (1, 5, 1, 3, 1)),  # three reduced axes
    ((40, 3, 50, 64), (1, 3, 1, 64)),  # innermost kept: columns over two reduced axes
    ((40, 3, 50, 5), (1, 3, 1, 5)),    # the same in scalar columns
    ((200, 2, 100, 12), (1, 2, 1, 12)),
]


def _bcast(op, sa, sb, i, dist="normal"):
    dist_b = "pos" if op == "div" else dist
    return Case(f"{op}_{sa}_{sb}_{dist}", op, "bwd",
                [Arr(sa, dist, 900 + i, requires_grad=True),
                 Arr(sb, dist_b, 950 + i, requires_grad=True)], _bshape(sa, sb), exact=False)


CASES = [_bcast(op, sa, sb, i) for i, (sa, sb) in enumerate(BCAST)
         for op in ("add", "sub", "mul", "div")]
CASES += [_bcast("mul", sa, sb, 20 + i, "special") for i, (sa, sb) in enumerate(BCAST)]
# a's gradient follows a's own memory: the last two axes swapped, whole and partial tiles
CASES += [Case(f"{op}_permuted_{s}", op, "bwd",
               [Arr(s, "normal", 300 + i, transpose=(1, 2), requires_grad=True),
                Arr((1, s[2], 1), "pos" if op == "div" else "normal", 330 + i, requires_grad=True)],
               (s[0], s[2], s[1]), exact=False)
          for i, s in enumerate([(2, 64, 128), (3, 65, 70), (1, 5, 9), (4, 100, 36)])
          for op in ("add", "mul", "div")]
# a whole-tensor reduction of a view whose innermost axis stays in place
CASES += [Case(f"{op}_all_{s}_{d}", op, "fwd", [Arr(s, d, 400 + i, transpose=(0, 1))], (1,),
               (DIM_ALL, 0, 0.0), "i64" if op == "argmax" else "f32")
          for i, s in enumerate([(5, 7, 8), (5, 7, 9), (130, 65, 64), (3, 5, 3000)])
          for d in ("normal", "special", "ties") for op in REDUCE + ["argmax"]]


@pytest.mark.parametrize("c", CASES, ids=[c.id for c in CASES])
def test_multi_axis(c):
    check_case(c)
