"""dq_matmul_act(DQ_ACT_Q16) on a few K-quant rows quantizes inside the GEMV: the bits of
dq_act_quantize + dq_gemv, split rows, ragged sizes, a bias, strided rows, and rows with
infinities, NaN, zeros and saturating codes included."""
from __future__ import annotations

import numpy as np
import pytest

import dynalm_amd as dq
from dqtest import activations, gguf_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("t,ms", [(O.Q4_K, (1, 2, 3, 4)), (O.Q6_K, (1, 2))], ids=["q4_K", "q6_K"])
@pytest.mark.parametrize("n,k", [(64, 256), (1, 512), (130, 2304), (4096, 14336), (17000, 256), (300, 20480)])
def test_fused_equals_quantize_then_gemv(cuda, t, ms, n, k):
    import dqtorch as T

    st = T.stream()
    rows = gguf_weights(t, n, k, 8100 + n)
    w = dq.Weight.upload(t, rows, k)
    bias = torch.from_numpy(O.normal(8200, n)).cuda()
    for m in ms:
        x = np.zeros((m, k + 3), np.float32)
        x[:, :k] = activations(m, k, 8300 + m)
        x[0, 5] = np.inf
        x[m - 1, 40:72] = 0.0
        if m > 1:
            x[1, 100] = np.nan
            x[1, 130] = -3e38
        xd = torch.from_numpy(x).cuda()
        y, z = torch.zeros((m, n), device="cuda"), torch.zeros((m, n), device="cuda")
        dq.matmul_act(w, dq.ACT_Q16, xd, m, k + 3, y, n, bias, st)
        acts = torch.empty((m, dq.act_row_bytes(dq.ACT_Q16, k)), dtype=torch.uint8, device="cuda")
        dq.act_quantize(dq.ACT_Q16, xd, m, k, k + 3, acts, st)
        dq.gemv(w, dq.ACT_Q16, acts, m, 0, n, z, n, bias, st)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy().view(np.uint32), z.cpu().numpy().view(np.uint32)), (m, n, k)
