"""What a Graph runs follows its DAG: slots, operands, parameters and node pointers changed between
passes are used by the next one, as the loop over the nodes that the passes stand for reads them
each time. The slots are host callbacks, so no GPU is needed."""
from __future__ import annotations

import ctypes as C

import pytest

from plast_amd import abi
from plast_amd import graph as graph_module
from plast_amd.graph import Graph


class _Lib:
    def error_count(self):
        return 0


@pytest.fixture()
def dag(monkeypatch):
    monkeypatch.setattr(graph_module, "lib", lambda: _Lib())
    log = []
    slots = {k: abi.ForwardKernel(lambda i, o, p, k=k: log.append((k, p.dim))) for k in "abcd"}

    def node(forward, backward, dim=0):
        n = abi.Node()
        n.op.gpu_forward = C.cast(slots[forward], C.c_void_p).value
        n.op.gpu_backward = C.cast(slots[backward], C.c_void_p).value
        n.params = abi.KernelParams(dim, 0, 0.0)
        return n
    nodes = [node("a", "b"), node("c", "d")]
    ptrs = (C.POINTER(abi.Node) * 2)(*[C.pointer(n) for n in nodes])
    g = Graph()
    g.dag = abi.DAG()
    g.dag.nodes, g.dag.count, g.dag.capacity = ptrs, 2, 2

    def run(kind):
        log.clear()
        getattr(g, kind)()
        return list(log)
    return g, nodes, ptrs, node, slots, run


def test_order(dag):
    run = dag[-1]
    for _ in range(2):
        assert run("forward") == [("a", 0), ("c", 0)]
        assert run("backward") == [("d", 0), ("b", 0)]


def test_changes_between_passes(dag):
    g, nodes, ptrs, node, slots, run = dag
    run("forward")
    nodes[0].op.gpu_forward = C.cast(slots["d"], C.c_void_p).value
    nodes[1].params = abi.KernelParams(7, 0, 0.0)
    assert run("forward") == [("d", 0), ("c", 7)]
    nodes[1].op.gpu_backward = C.cast(slots["a"], C.c_void_p).value
    assert run("backward") == [("a", 7), ("b", 0)]
    other = node("b", "c", 3)
    ptrs[0] = C.pointer(other)
    assert run("forward") == [("b", 3), ("c", 7)]
    g.dag.count = 1
    assert run("forward") == [("b", 3)]
    more = (C.POINTER(abi.Node) * 1)(C.pointer(nodes[1]))
    g.dag.nodes = more
    assert run("backward") == [("a", 7)]
    g.dag.count = 0
    assert run("forward") == []
