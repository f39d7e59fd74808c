"""The per-32 GEMM's offsets (dq_gemm_p32.hip): c_j = d * (code sum) runs as three bf16 parts.
Activation rows whose codes are all of one sign make the offsets as large as the dot itself,
and the rows' magnitudes run from subnormal to near the type's largest; the tile counts cover
one, two and four activation tiles, a partial one and a split K."""
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
    x *= (10.0 ** rng.uniform(-36, 35, (m, 1))).astype(np.float32)
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
    bound = (k / 32 + 16) * 2.0**-23 * 3 * mag + 1e-38 * k  # + products below the normal range
    assert np.all(np.abs(got - want) <= bound)
