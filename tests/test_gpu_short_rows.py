"""Cross-entropy and softmax over short rows (2, 8, 32 or 64 lanes a row in a wave's registers) and over
rows of any length and alignment, on each side of the lengths where the kernel changes, against the
oracle at the bars of tests/test_gpu_ce_step.py and tests/test_gpu_softmax.py: clean rows and the
special ones (NaN, infinities, zero maxima, extreme spreads), more rows than the step's workgroups
hold at once, and results that repeat bit for bit. A gradient's scale has the floor 1e-2 * g: its
bar is then at least 1e-7 * g, the rounding of g * (p - 1) for p next to 1 (an ulp of p is 6e-8; the
same floor as 1e-2 / N where g = 1 / N)."""
from __future__ import annotations

import numpy as np
import pytest

from cases import assert_bits, check_ce_rows
from test_gpu_ce_step import _oracle, _special_rows, _step
from test_gpu_ce_step import test_step_matches_oracle as step_case
from test_gpu_softmax import test_softmax_forward_and_backward as softmax_case

pytestmark = pytest.mark.gpu

ROW = [1, 2, 3, 4, 5, 10, 31, 32, 33, 127, 128, 129, 511, 512, 513, 1001, 1024, 1025, 2047, 2048, 2049,
       2050, 4097, 8191]


@pytest.mark.parametrize("C", ROW)
def test_cross_entropy_op(C):
    """The op's forward and its accumulating and overwriting backward; the special rows need C > 3."""
    from plast_amd import ops, runtime as rt
    from plast_amd.abi import KernelParams
    N = 203
    print(f"ce op {N}x{C}", flush=True)
    rng = np.random.RandomState(C)
    x = (rng.randn(N, C) * 2).astype(np.float32)
    if C > 3:
        _special_rows(x)
    lab = rng.randint(0, C, N).astype(np.int32)
    g = rng.uniform(0.1, 1.0, N).astype(np.float32)
    X, Lb = rt.DeviceTensor.from_numpy(x, requires_grad=True), rt.DeviceTensor.from_numpy(lab)
    loss, stats = ops.softmax_cross_entropy(X, Lb, requires_grad=True)
    rt.lib().arena_memcpy_h2d_hip(loss.grad.ptr, g.ctypes.data, g.nbytes)
    rt.backward("softmax_cross_entropy", [X, Lb, stats], loss)
    wst, wloss, wdx = _oracle(x, lab, g)
    first = X.grad.numpy()
    check_ce_rows(x, lab, g, stats.numpy(), loss.numpy(), first, wst, wloss, wdx, 1e-2 * g)
    assert_bits(np.isnan(first), np.isnan(wdx), "NaN positions of dlogits")
    rt.backward("softmax_cross_entropy", [X, Lb, stats], loss)
    assert_bits(X.grad.numpy(), first + first, "accumulated gradient")
    rt.backward("softmax_cross_entropy", [X, Lb, stats], loss, KernelParams(0, 1, 0.0))
    assert_bits(X.grad.numpy(), first, "overwritten gradient")


@pytest.mark.parametrize("special", [False, True], ids=["clean", "special_rows"])
@pytest.mark.parametrize("N, C", [(1, 4), (9, 5), (700, 10), (301, 31), (77, 33), (130, 128), (41, 300),
                                  (25, 513), (19, 1025), (300, 2046), (21, 2049), (33, 4099), (12, 9001),
                                  (10, 32767)])
def test_step(N, C, special):
    step_case(N, C, special)


@pytest.mark.parametrize("special", [False, True], ids=["clean", "special_rows"])
@pytest.mark.parametrize("N, C", [(255, 10), (256, 10), (257, 10), (258, 4), (259, 5), (260, 33), (261, 130),
                                  (262, 300), (263, 513), (264, 1025), (256, 2048), (257, 2048)])
def test_step_row_counts(N, C, special):
    """Each side of one row per CU (256), beyond which short rows share waves."""
    step_case(N, C, special)


def test_short_step_repeats():
    """The bias gradient of short rows is the same bits on every call, with a workgroup per row too."""
    from plast_amd import runtime as rt
    rng = np.random.RandomState(9)
    for N, C in ((200, 2048), (37, 12)):
        x, lab = (rng.randn(N, C) * 2).astype(np.float32), rng.randint(0, C, N).astype(np.int32)
        X, Lb = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor.from_numpy(lab)
        g = np.full(N, 1.0 / N, np.float32)
        first = _step(rt, X, Lb, g)
        for _ in range(20):
            for a, b in zip(_step(rt, X, Lb, g), first):
                assert_bits(a, b, "a later call")


@pytest.mark.parametrize("N, C", [(40000, 12), (20000, 77), (6000, 700), (3000, 2000), (1100, 2051)])
def test_step_many_rows(N, C):
    """Several row groups per wave: every row against the oracle, the same bits twice for short rows."""
    from plast_amd import runtime as rt
    print(f"ce step {N}x{C}", flush=True)
    rng = np.random.RandomState(C)
    x = (rng.randn(N, C) * 2).astype(np.float32)
    x[N // 2, :] = 0.0     # a zero maximum, and an infinite logit, in later groups
    x[N - 3, 1] = -np.inf
    lab = rng.randint(0, C, N).astype(np.int32)
    g = rng.uniform(0.1, 1.0, N).astype(np.float32)
    X, Lb = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor.from_numpy(lab)
    st, loss, dx, db = _step(rt, X, Lb, g)
    wst, wloss, wdx = _oracle(x, lab, g)
    check_ce_rows(x, lab, g, st, loss, dx, wst, wloss, wdx, 1e-2 * g)
    ok = np.isfinite(wdx).all(0)
    want = wdx.astype(np.float64).sum(0)
    bar = 1e-5 * np.abs(wdx.astype(np.float64)).sum(0) + 1e-12
    assert np.all(np.abs(db - want)[ok] <= bar[ok])
    if C <= 2048:
        for a, b in zip(_step(rt, X, Lb, g), (st, loss, dx, db)):
            assert_bits(a, b, "a second call")


@pytest.mark.parametrize("log", [False, True], ids=["softmax", "log_softmax"])
@pytest.mark.parametrize("C", ROW + [16381, 16388, 20001])
def test_softmax_rows(C, log):
    softmax_case((23, C), log)


@pytest.mark.parametrize("log", [False, True], ids=["softmax", "log_softmax"])
@pytest.mark.parametrize("C", [c for c in ROW if c <= 1025] + [767, 768, 769])
def test_softmax_many_rows(C, log):
    """Rows enough for a wave each, or a share of one."""
    softmax_case((2101, C), log)


@pytest.mark.parametrize("log", [False, True], ids=["softmax", "log_softmax"])
@pytest.mark.parametrize("N", [1279, 1280, 1535, 1536, 1699, 1700, 2047, 2048])
def test_softmax_row_counts(N, log):
    """Each side of the row counts where a wave takes over from a workgroup."""
    softmax_case((N, 77), log)
    softmax_case((N, 300), log)


@pytest.mark.parametrize("log", [False, True], ids=["softmax", "log_softmax"])
@pytest.mark.parametrize("N, C", [(2175, 3), (2176, 301), (3071, 301), (3072, 3), (300, 511), (300, 514),
                                  (1024, 1023), (1025, 1026), (1025, 1343), (1025, 1345), (2048, 1022),
                                  (2049, 1022), (10894, 770), (10895, 770), (9, 4), (9, 16), (9, 20),
                                  (767, 20), (768, 300), (767, 300)])
def test_softmax_lines(N, C, log):
    """Each side of the lines between three passes, a wave and a workgroup's registers: rows that are
    no whole float4, and rows that share a 128-byte line with their neighbours."""
    softmax_case((N, C), log)


def _offset(rt, x, off):
    """x at `off` floats past a 16-byte boundary."""
    base = rt.DeviceTensor.from_numpy(np.concatenate([np.zeros(off, np.float32), x.ravel()]))
    return rt.DeviceTensor(x.shape, base=base, offset=off, zero=False)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("N, C", [(7, 100), (2100, 100), (7, 2052), (7, 17000)])
def test_misaligned_rows(N, C, off):
    """Rows of whole float4 in buffers that do not start on one, forward and backward: the bits of the
    aligned call where the rows are a wave's or share one (any alignment is the same kernel), the fp64
    softmax for the others (1e-5 of each value and of its gradient's terms)."""
    from plast_amd import abi, runtime as rt
    from plast_amd.abi import KernelParams
    print(f"softmax {N}x{C} offset {off}", flush=True)
    rng = np.random.RandomState(C + off)
    x, dy, d0 = (rng.randn(N, C).astype(np.float32) for _ in range(3))
    p = KernelParams(1, 0, 0.0)

    def run(at):
        X, Y, DY, D = _offset(rt, x, at), _offset(rt, np.zeros_like(x), (4 - at) % 4), _offset(rt, dy, at), _offset(rt, d0, at)
        tx = abi.make_tensor(X.ptr, x.shape, None, rt.FLOAT32, rt.GPU, True, D.t)
        ty = abi.make_tensor(Y.ptr, x.shape, None, rt.FLOAT32, rt.GPU, True, DY.t)
        rt.forward("softmax", [tx], ty, p)
        rt.backward("softmax", [tx], ty, p)
        return Y.numpy(), D.numpy()
    y, d = run(off)
    h = x.astype(np.float64)
    e = np.exp(h - h.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    assert np.all(np.abs(y - want) <= 1e-5 * want)
    t = dy * want
    term = want * (dy - t.sum(1, keepdims=True))
    scale = np.abs(d0) + want * (np.abs(dy) + np.abs(t).sum(1, keepdims=True))
    assert np.all(np.abs(d - (d0 + term)) <= 1e-5 * scale)
    if N > 2047 and C <= 768:
        for a, b in zip((y, d), run(0)):
            assert_bits(a, b, "aligned")


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("N, C", [(300, 100), (9, 100), (40, 2052), (12, 8192)])
def test_misaligned_cross_entropy(N, C, off):
    """The step and the op's backward over rows of whole float4 that start off a 16-byte boundary."""
    from plast_amd import abi, runtime as rt
    print(f"ce {N}x{C} offset {off}", flush=True)
    rng = np.random.RandomState(C + off)
    x = (rng.randn(N, C) * 2).astype(np.float32)
    _special_rows(x)
    lab = rng.randint(0, C, N).astype(np.int32)
    g = rng.uniform(0.1, 1.0, N).astype(np.float32)
    wst, wloss, wdx = _oracle(x, lab, g)
    X, DX = _offset(rt, x, off), _offset(rt, np.zeros_like(x), off)
    Lb, G = rt.DeviceTensor.from_numpy(lab), rt.DeviceTensor.from_numpy(g)
    st, loss, db = rt.DeviceTensor((N, 2)), rt.DeviceTensor((N,)), rt.DeviceTensor((C,))
    L = rt.lib()
    L.softmax_cross_entropy_step_hip(X.ptr, Lb.ptr, G.ptr, st.ptr, loss.ptr, DX.ptr, db.ptr, None, N, C)
    L.check("step")
    check_ce_rows(x, lab, g, st.numpy(), loss.numpy(), DX.numpy(), wst, wloss, wdx, 1e-2 * g)
    ok = np.isfinite(wdx).all(0)
    bar = 1e-5 * np.abs(wdx.astype(np.float64)).sum(0) + 1e-12
    assert np.all(np.abs(db.numpy() - wdx.astype(np.float64).sum(0))[ok] <= bar[ok])
    D = _offset(rt, np.zeros_like(x), (off + 1) % 4)
    tx = abi.make_tensor(X.ptr, x.shape, None, rt.FLOAT32, rt.GPU, True, D.t)
    out = abi.make_tensor(loss.ptr, (N,), None, rt.FLOAT32, rt.GPU, True, G.t)
    rt.backward("softmax_cross_entropy", [tx, Lb, st], out)
    check_ce_rows(x, lab, g, st.numpy(), loss.numpy(), D.numpy(), wst, wloss, wdx, 1e-2 * g)
