"""Calls recorded into a graph by a library whose workspace is still empty: the launches that split
their work over partials keep the split there, and give the eager call's results bit for bit. The
library is a copy of the build with a state of its own."""
from __future__ import annotations

import shutil

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture()
def cold(tmp_path):
    from plast_amd import runtime as rt
    base = rt.lib()
    path = tmp_path / "cold.so"
    shutil.copy(base.path, path)
    L = rt.load_library(path)
    assert L.plast_hip_workspace_bytes(0) == 0
    rt.use_library(L)
    yield L
    rt.use_library(base)


def _replayed(L, call, outs):
    """The outputs of the captured call, the same bits from two replays, from the eager call and from
    a second capture, with the workspace that the eager call left."""
    def clear():
        for t in outs:
            L.zeros_hip(t.p, int(np.prod(t.shape)))

    def capture():
        assert L.plast_hip_capture_begin() == 0
        call()
        g = L.plast_hip_capture_end()
        L.check("capture")
        return g

    def replay(g):
        clear()
        assert L.plast_hip_graph_launch(g) == 0
        return [t.numpy() for t in outs]

    g = capture()
    assert L.plast_hip_workspace_bytes(0) == 0
    got = [replay(g), replay(g)]
    clear()
    call()
    got.append([t.numpy() for t in outs])
    warm = capture()
    got += [replay(warm), replay(g)]
    for h in (g, warm):
        L.plast_hip_graph_destroy(h)
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    return got[0]


@pytest.mark.parametrize("shape, small", [((300, 2, 1028), (1, 2, 1)), ((200, 2, 100, 12), (1, 2, 1, 12)),
                                          ((300, 2, 1027), (1, 2, 1))])
def test_gradient_over_several_axes(cold, shape, small):
    from plast_amd import runtime as rt
    print(f"cold capture {shape}", flush=True)
    rng = np.random.RandomState(1)
    a = rt.DeviceTensor.from_numpy(rng.randn(*shape).astype(np.float32))
    b = rt.DeviceTensor.from_numpy(rng.randn(*small).astype(np.float32), requires_grad=True)
    out = rt.DeviceTensor(shape, requires_grad=True)
    g = rng.randn(*shape).astype(np.float32)
    cold.arena_memcpy_h2d_hip(out.grad.ptr, g.ctypes.data, g.nbytes)
    got = _replayed(cold, lambda: rt.backward("mul", [a, b], out), [b.grad])[0]
    terms = (g * a.numpy()).astype(np.float64)
    axes = tuple(i for i, n in enumerate(small) if n == 1)
    want = terms.sum(axes, keepdims=True).reshape(got.shape)
    bar = 1e-5 * np.abs(terms).sum(axes, keepdims=True).reshape(got.shape)
    assert np.all(np.abs(got - want) <= bar)


@pytest.mark.parametrize("shape", [(100, 255), (60000, 8), (127, 129)])
def test_narrow_columns(cold, shape):
    from plast_amd import runtime as rt
    from plast_amd.abi import KernelParams
    print(f"cold capture {shape}", flush=True)
    x = np.random.RandomState(2).randn(*shape).astype(np.float32)
    X, out = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor((shape[1],))
    got = _replayed(cold, lambda: rt.forward("sum", [X], out, KernelParams(0, 0, 0.0)), [out])[0]
    assert np.all(np.abs(got - x.astype(np.float64).sum(0)) <= 1e-5 * np.abs(x).astype(np.float64).sum(0))


def test_step_of_ragged_rows(cold):
    from plast_amd import runtime as rt
    N, C = 40, 3001
    print(f"cold capture step {N}x{C}", flush=True)
    rng = np.random.RandomState(3)
    x = (rng.randn(N, C) * 2).astype(np.float32)
    lab = rng.randint(0, C, N).astype(np.int32)
    g = np.full(N, np.float32(1 / N), np.float32)
    X, Y, G = (rt.DeviceTensor.from_numpy(v) for v in (x, lab, g))
    st, loss, dx = rt.DeviceTensor((N, 2)), rt.DeviceTensor((N,)), rt.DeviceTensor((N, C))
    db, mean = rt.DeviceTensor((C,)), rt.DeviceTensor((1,))
    got = _replayed(cold, lambda: cold.softmax_cross_entropy_step_hip(
        X.ptr, Y.ptr, G.ptr, st.ptr, loss.ptr, dx.ptr, db.ptr, mean.ptr, N, C), [loss, dx, st, db, mean])
    x64 = x.astype(np.float64)
    m = x64.max(1, keepdims=True)
    lse = np.log(np.exp(x64 - m).sum(1))
    assert np.allclose(got[0], lse - (x64 - m)[np.arange(N), lab], rtol=0, atol=1e-5 * (1 + lse.max()))
    p = np.exp(x64 - m - lse[:, None])
    p[np.arange(N), lab] -= 1.0
    assert np.all(np.abs(got[1] - p / N) <= 1e-5 * (np.abs(p) + 1e-2) / N)
