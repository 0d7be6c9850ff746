"""Max and min whose value the fast order may not decide in many rows or columns at once: dead
channels (every extreme a zero, of either sign), NaN in some columns, at their ends and at a chunk's
end, infinities; bit for bit against the oracle's fold, over rows shared by a wave and narrow
columns in one chunk and in several. Sums with a non-finite term in every row."""
from __future__ import annotations

import numpy as np
import pytest

from cases import assert_bits
from hostlib import HostTensor, oracle_forward

pytestmark = pytest.mark.gpu

SHAPES = [((1000, 100), 1), ((77, 5), 1), ((300, 33), 1), ((41, 129), 1), ((9, 512), 1), ((70, 513), 1),
          ((60000, 10), 0), ((60000, 3), 0), ((3000, 64), 0), ((200, 77), 0), ((5000, 7), 0), ((33000, 250), 0),
          ((300, 128, 9), 1), ((9, 2100, 30), 1)]


def _data(shape, dim, kind, sign):
    """Data whose extreme in the direction of `sign` is a zero along `dim`; kind adds NaN and infinities."""
    rng = np.random.RandomState(sum(shape) + len(kind))
    x = -sign * np.abs(rng.randn(*shape)).astype(np.float32)
    zero = rng.rand(*shape) < 0.3
    x[zero] = np.where(rng.rand(int(zero.sum())) < 0.5, np.float32(0.0), np.float32(-0.0))
    if kind == "nan":
        x[rng.rand(*shape) < 4.0 / shape[dim]] = np.nan
        x = np.moveaxis(x, dim, 0)
        x[-1].ravel()[::3] = np.nan                      # lines that end in a NaN
        x[:, ...].reshape(len(x), -1)[:, 1::4] = np.nan  # lines of nothing else
        x = np.ascontiguousarray(np.moveaxis(x, 0, dim))
    if kind == "inf":
        x[rng.rand(*shape) < 0.3] = -sign * np.inf
        np.moveaxis(x, dim, 0)[...].reshape(shape[dim], -1)[:, 2::5] = -sign * np.inf
    return x


@pytest.mark.parametrize("op", ["max", "min"])
@pytest.mark.parametrize("kind", ["dead", "nan", "inf"])
@pytest.mark.parametrize("shape, dim", SHAPES)
def test_extremes(shape, dim, kind, op):
    from plast_amd import runtime as rt
    from plast_amd.abi import KernelParams
    print(f"{op} {kind} {shape} dim {dim}", flush=True)
    x = _data(shape, dim, kind, 1 if op == "max" else -1)
    o = tuple(n for d, n in enumerate(shape) if d != dim)
    X, out = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor(o, zero=False)
    rt.forward(op, [X], out, KernelParams(dim, 0, 0.0))
    H, want = HostTensor(x), HostTensor(np.zeros(o, np.float32))
    oracle_forward(op, [H], want, KernelParams(dim, 0, 0.0))
    assert_bits(out.numpy(), want.numpy(), op)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("shape", [(300, 5), (200, 100), (50, 300)])
def test_sums_of_rows(shape, bad):
    from plast_amd import runtime as rt
    from plast_amd.abi import KernelParams
    x = np.random.RandomState(3).randn(*shape).astype(np.float32)
    x[:, 2] = bad
    X, out = rt.DeviceTensor.from_numpy(x), rt.DeviceTensor((shape[0],), zero=False)
    rt.forward("sum", [X], out, KernelParams(1, 0, 0.0))
    got = out.numpy()
    assert np.all(np.isnan(got)) if np.isnan(bad) else np.all(got == bad)
