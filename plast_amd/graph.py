"""Build and run op DAGs over device tensors through the library's `Op` table.

Standalone stand-in for the reference's L1 executor (src/core/node.c:3-32, src/core/graph.c:30-65)
and for its scheduler's fusion hook (src/scheduler/scheduler.c:16-52, fusion.c:209-224): nodes are
`Node` structs with GPU slots from plast_hip_get_op_impl, ordered by the same depth-first
topological sort, optionally rewritten by plast_hip_fuse_elementwise_chains, then executed by
calling each node's gpu_forward slot.
"""
from __future__ import annotations

import ctypes as C

from . import abi
from .abi import KernelParams
from .runtime import DeviceTensor, lib


class Graph:
    def __init__(self):
        self.nodes: list[abi.Node] = []
        self._keep = []       # ctypes objects the C side points into
        self._arena_bufs = bufs = []

        # the fusion pass allocates its nodes and tapes through this callback; it refers to the list
        # alone, so that a dropped graph (and the tensors it keeps) goes at once and not at the next
        # garbage collection
        def alloc(arena, size, align):
            buf = C.create_string_buffer(int(size) + int(align))
            bufs.append(buf)
            addr = C.addressof(buf)
            return (addr + align - 1) // align * align

        self._alloc_cb = abi.ArenaAllocFn(alloc)
        self.dag = None
        self._run = None      # what _bound() made of the DAG

    # --- construction
    def node(self, op: str, inputs, output: DeviceTensor, p: KernelParams | None = None) -> DeviceTensor:
        L = lib()
        n = abi.Node()
        arr = (abi.TensorP * len(inputs))(*[C.pointer(t.t) for t in inputs])
        self._keep.append(arr)
        # the nodes point into these tensors' structs and device memory: keep the owners alive
        # as long as the graph (a collected DeviceTensor frees its buffer)
        self._keep.extend(inputs)
        self._keep.append(output)
        n.inputs = C.cast(arr, abi.TensorPP)
        n.output = C.pointer(output.t)
        n.op = L.plast_hip_get_op_impl(abi.OP[op.upper()])
        n.op_type = abi.OP[op.upper()]
        n.num_inputs = len(inputs)
        n.params = p or KernelParams(0, 0, 0.0)
        self.nodes.append(n)
        output.t.creator = C.addressof(n)
        return output

    def build(self, root: DeviceTensor, fuse: bool = False) -> int:
        """Topologically order the nodes reachable from root's creator (graph.c:30-39); with
        fuse=True run the elementwise-chain pass. Returns the number of chains fused."""
        by_addr = {C.addressof(n): n for n in self.nodes}
        order: list[abi.Node] = []
        seen: set[int] = set()

        def visit(addr):
            seen.add(addr)
            n = by_addr[addr]
            for i in range(n.num_inputs):
                cr = n.inputs[i].contents.creator
                if cr and cr not in seen and cr in by_addr:
                    visit(cr)
            order.append(n)

        visit(root.t.creator)
        ptrs = (C.POINTER(abi.Node) * len(order))(*[C.pointer(n) for n in order])
        self._keep.append(ptrs)
        dag = abi.DAG()
        dag.nodes = ptrs
        dag.count = len(order)
        dag.capacity = len(order)
        dag.arena = None
        self.dag = dag
        fused = 0
        if fuse:
            fused = lib().plast_hip_fuse_elementwise_chains(C.byref(dag), self._alloc_cb)
            lib().check("plast_hip_fuse_elementwise_chains")
        self._run = None
        return int(fused)

    def op_types(self) -> list[str]:
        return [abi.OP_NAMES[self.dag.nodes[i].contents.op_type] for i in range(self.dag.count)]

    def _calls(self):
        """(forward slot, backward slot, inputs, output, params) of every node of the DAG, in order:
        the objects ctypes would otherwise make anew for each field on every pass (2 us a node of
        the 5 a small pass took). Each lies over the node's own memory, its slots included, so a
        node changed after build() is run as changed."""
        slot = abi.Node.op.offset
        calls = []
        for i in range(self.dag.count):
            n = self.dag.nodes[i].contents
            calls.append((abi.ForwardKernel.from_buffer(n, slot + abi.Op.gpu_forward.offset),
                          abi.BackwardKernel.from_buffer(n, slot + abi.Op.gpu_backward.offset),
                          n.inputs, n.output, n.params))
        return calls

    def _bound(self):
        """The calls, bound on the first pass and again when the DAG holds other nodes: its head (the
        node array and the count) and the array are compared with what they held then."""
        run = self._run
        if run is not None:
            dag, head, was_head, nodes, was_nodes, calls = run
            if dag is self.dag and head() == was_head and nodes() == was_nodes:
                return calls
        dag = self.dag
        size = dag.count * C.sizeof(C.c_void_p)
        head = memoryview((C.c_char * abi.DAG.capacity.offset).from_buffer(dag)).tobytes
        nodes = memoryview((C.c_char * size).from_address(C.addressof(dag.nodes.contents)) if size
                           else (C.c_char * 0)()).tobytes
        self._run = dag, head, head(), nodes, nodes(), self._calls()
        return self._run[5]

    def forward(self) -> None:
        """dag_forward (graph.c:57-60): each node's GPU forward slot in order."""
        for f, _, inputs, output, p in self._bound():
            f(inputs, output, p)
        L = lib()
        if L.error_count():
            L.raise_error("dag forward")

    def backward(self) -> None:
        """dag_backward (graph.c:62-65): GPU backward slots in reverse order."""
        for _, f, inputs, output, p in reversed(self._bound()):
            f(inputs, output, p)
        L = lib()
        if L.error_count():
            L.raise_error("dag backward")
