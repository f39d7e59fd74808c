"""The per-32 GEMM's offsets (dq_gemm_p32.hip): c_j = d * (code sum) runs as four bf16 parts.
Activation rows whose codes are all of one sign make the offsets as large as the dot itself,
and the rows' magnitudes run from 1e-37 to near the type's largest, infinities and NaN; the tile
counts cover one, two and four activation tiles, a partial one and a split K."""
from __future__ import annotations

import numpy as np
import pytest

import dynalm_amd as dq
from dqtest import gguf_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("m,n,k", [(5, 64, 512), (33, 300, 1024), (65, 200, 4096), (130, 4096, 256)])
def test_large_offsets(cuda, m, n, k):
    import dqtorch as T

    rows = gguf_weights(O.Q4_K, n, k, 5100 + m)
    rng = np.random.default_rng(5200 + m)
    x = np.abs(rng.standard_normal((m, k))).astype(np.float32) + np.float32(0.5)
    x *= (10.0 ** rng.permutation(np.linspace(-37, 35, m))[:, None]).astype(np.float32)
    x[m // 2] *= -1
    w = dq.Weight.upload(O.Q4_K, rows, k)
    y = torch.zeros((m, n), device="cuda")
    dq.matmul_act(w, dq.ACT_PER32, torch.from_numpy(x).cuda(), m, k, y, n, None, T.stream())
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    acts = O.quantize_act(O.ACT_PER32, x)
    want = O.matmul(O.Q4_K, O.ACT_PER32, rows, acts, k).astype(np.float64)
    # the contract's dot as two sums that cancel: fp32 rounding of each of K / 32 terms of both
    mag = np.abs(x.astype(np.float64)) @ np.abs(O.expand_x86(O.Q4_K, rows, k).astype(np.float64)).T
    bound = (k / 32 + 16) * 2.0**-23 * 3 * mag
    # da sc P 2^-24 rounds at half the subnormal step in each of K / 32 sub-blocks, before d 2^24
    # comes to it; the offsets' sum 2^-9 at a step in each of eight terms, before -dmin 2^9
    h = rows.reshape(n, k // 256, 144)[:, :, :4].copy().view(np.float16).astype(np.float64)
    bound += k / 32 * (np.abs(h[:, :, 0]).max() * 2.0**-126 + np.abs(h[:, :, 1]).max() * 2.0**-137)
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("m,n,k", [(5, 64, 512), (33, 300, 1024), (70, 200, 256)])
def test_infinite_and_nan_rows(cuda, m, n, k):
    """An infinity or a NaN in a row makes its sub-block's scale and offset so: the outputs that the
    contract makes infinite or NaN are one of them (the GEMM applies the scales in another order,
    in which an infinity may meet its opposite), and no other row changes."""
    import dqtorch as T

    rows = gguf_weights(O.Q4_K, n, k, 5300 + m)
    x = np.random.default_rng(5400 + m).standard_normal((m, k)).astype(np.float32)
    w = dq.Weight.upload(O.Q4_K, rows, k)

    def run(a):
        y = torch.zeros((m, n), device="cuda")
        dq.matmul_act(w, dq.ACT_PER32, torch.from_numpy(a).cuda(), m, k, y, n, None, T.stream())
        torch.cuda.synchronize()
        return y.cpu().numpy()

    clean = run(x)
    x[1, 7], x[2, k - 1], x[4, 40] = np.inf, -np.inf, np.nan
    got = run(x)
    want = O.matmul(O.Q4_K, O.ACT_PER32, rows, O.quantize_act(O.ACT_PER32, x), k)
    odd = ~np.isfinite(want)
    assert odd.any() and np.array_equal(~np.isfinite(got), odd)
    same = [r for r in range(m) if r not in (1, 2, 4)]
    assert np.array_equal(got[same].view(np.uint32), clean[same].view(np.uint32))
