"""dq_matmul_many's one-row K-quant jobs in one launch (k_gemv_many): every job has dq_matmul's
bits, over mixed types, ragged row counts, long rows, a bias, more jobs than a launch takes,
several K in one call and jobs of other kinds between them."""
from __future__ import annotations

import numpy as np
import pytest

import dynalm_amd as dq
from dqtest import activations, gguf_weights
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("ks,count", [((1536,), 3), ((256,), 2), ((4096, 2048), 9), ((8192,), 8), ((14336, 256, 14336), 11),
                                      ((16640,), 2)])
def test_one_row_jobs(cuda, ks, count):
    import dqtorch as T

    st = T.stream()
    jobs, keep, want = [], [], []
    for i in range(count):
        k = ks[i % len(ks)]
        t = (O.Q4_K, O.Q6_K)[i % 2] if i != 4 else O.Q8_0
        n = (256, 1, 63, 65, 1536)[i % 5]
        m = 1 if i != 5 else 3
        rows = gguf_weights(t, n, k, 7100 + 31 * i + k)
        w = dq.Weight.upload(t, rows, k)
        x = torch.from_numpy(activations(m, k, 7200 + i)).cuda()
        b = torch.from_numpy(O.normal(7300 + i, n)).cuda() if i % 3 == 0 else None
        y, ref = torch.full((m, n + 2), 7.0, device="cuda"), torch.full((m, n + 2), 7.0, device="cuda")
        dq.matmul(w, x, m, k, ref, n + 2, b, st)
        jobs.append((w, x, m, k, y, n + 2, b))
        keep.append((w, x, b))
        want.append(ref)
    dq.matmul_many(jobs, st)
    torch.cuda.synchronize()
    for i, (j, ref) in enumerate(zip(jobs, want)):
        a, b = j[4].cpu().numpy(), ref.cpu().numpy()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f"job {i}"
