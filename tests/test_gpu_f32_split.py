"""The fp32 expand class on the bf16 matrix cores (dq_gemm_f32.hip): every tile shape at its
edges, and inputs that the three-part split of the activations cannot hold."""
from __future__ import annotations

import numpy as np
import pytest

import dynalm_amd as dq
from dqtest import TYPES, activations, gguf_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def run(t, rows, x, k, bias=None):
    import dqtorch as T

    w = dq.Weight.upload(t, rows, k)
    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    y = torch.zeros((x.shape[0], w.n), device="cuda")
    b = None if bias is None else torch.from_numpy(bias).cuda()
    dq.matmul_plan(w, None, xd, x.shape[0], k, y, w.n, b, T.stream())
    torch.cuda.synchronize()
    return y.cpu().numpy()


def exact(t, rows, x, k):
    w = O.expand_x86(t, rows, k).astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        return x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T


# m, n, K in blocks: 64 x 64 tiles up to 256 of them; 128 x 64; 128 x 128 (N = 14336 at
# M = 130); 128 x 224 (189 tiles); one block of K (an empty second half), odd block counts
SHAPES = [(16, 1, 1), (17, 63, 3), (64, 65, 8), (65, 130, 5), (128, 2000, 8), (129, 6000, 8), (130, 14336, 8), (300, 13999, 8)]


@pytest.mark.parametrize("t", TYPES, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n,blocks", SHAPES)
def test_tiles(cuda, t, m, n, blocks):
    k = 256 * max(1, blocks // 4) if t in (O.Q4_K, O.Q6_K) else 32 * blocks
    rows = gguf_weights(t, n, k, 4100 + t + m)
    x = activations(m, k, 4200 + m)
    bias = O.normal(4300 + m, n)
    want, mag = exact(t, rows, x, k)
    # one rounding per block fold and inside its sums: far inside the class's 1e-5 of sum |terms|
    assert np.all(np.abs(run(t, rows, x, k, bias) - (want + bias)) <= 2e-6 * (mag + np.abs(bias)) + 1e-30)


@pytest.mark.parametrize("t", TYPES, ids=lambda t: O.TYPE_NAMES[t])
def test_non_finite_and_extreme_rows(cuda, t):
    """Rows with infinities or NaN come out as IEEE arithmetic gives them (the same in any
    order: an infinity, its sign, or NaN), rows near the type's limits come out right, and the
    other rows are untouched."""
    k, n, m = 512, 200, 40
    rows = gguf_weights(t, n, k, 4400 + t)
    x = activations(m, k, 4401)
    x[3, 7] = np.inf
    x[5, 300] = -np.inf
    x[6, [1, 400]] = np.inf
    x[8, 9] = np.nan
    x[11] = np.float32(1e-30) * x[11]
    x[13] = 0.0
    x[13, 100] = np.finfo(np.float32).max  # its bf16 rounding is infinite
    y = run(t, rows, x, k)
    want, mag = exact(t, rows, x, k)
    with np.errstate(over="ignore"):
        w32 = want.astype(np.float32)
    odd = [3, 5, 6, 8]
    assert np.array_equal(np.isnan(y[odd]), np.isnan(w32[odd])) and np.isinf(w32[odd]).any()
    assert np.array_equal(y[odd][np.isinf(w32[odd])], w32[odd][np.isinf(w32[odd])])
    rest = [r for r in range(m) if r not in odd]
    assert np.all(np.abs(y[rest] - want[rest]) <= 2e-6 * mag[rest])
    clean = activations(m, k, 4401)
    same = [r for r in range(m) if r not in odd + [11, 13]]
    assert np.array_equal(run(t, rows, clean, k)[same].view(np.uint32), y[same].view(np.uint32))


@pytest.mark.parametrize("t", TYPES, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n,blocks", SHAPES)
def test_many_odd_rows(cuda, t, m, n, blocks):
    """Batches whose rows hold infinities, NaN and values past the split's range, at the edges of every
    tile shape: IEEE's result in each, with a bias, beside rows that keep their bits."""
    k = 256 * max(1, blocks // 4) if t in (O.Q4_K, O.Q6_K) else 32 * blocks
    rows = gguf_weights(t, min(n, 300), k, 4600 + t + m)
    rows = np.tile(rows, (-(-n // rows.shape[0]), 1))[:n].copy()
    x = activations(m, k, 4700 + m)
    bias = O.normal(4800 + m, n)
    clean = run(t, rows, x, k, bias)
    x[::4, k - 1] = np.inf
    x[1::4, k // 2] = np.nan
    x[2::4, 0] = np.float32(-2e35)
    y = run(t, rows, x, k, bias)
    want, mag = exact(t, rows, x, k)
    want += bias
    fin = np.isfinite(want)
    with np.errstate(invalid="ignore"):
        diff = np.abs(y - want)
    assert np.array_equal(np.isfinite(y), fin) and np.array_equal(y[~fin], want[~fin].astype(np.float32), equal_nan=True)
    assert np.all(diff[fin] <= (2e-6 * (mag + np.abs(bias)))[fin])
    assert np.array_equal(y[3::4].view(np.uint32), clean[3::4].view(np.uint32))


@pytest.mark.parametrize("t", TYPES, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n", [(20, 100), (130, 700)])
def test_rows_of_every_magnitude(cuda, t, m, n):
    """Rows from subnormal values up keep fp32's relative error: the split holds every fp32 value."""
    k = 1024
    rows = gguf_weights(t, n, k, 4500 + t)
    x = activations(m, k, 4501).astype(np.float64)
    x = (x * 10.0 ** np.linspace(-42, 34, m)[:, None]).astype(np.float32)
    x[3, ::2] = 0.0
    want, mag = exact(t, rows, x, k)
    # the class's rounding, and half of the subnormal step where the output falls below the normal range
    assert np.all(np.abs(run(t, rows, x, k) - want) <= 2e-6 * mag + 2.0**-150)
