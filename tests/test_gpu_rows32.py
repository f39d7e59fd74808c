"""The MFMA GEMV of Q8_0 / Q4_0 weights x per-32 rows (dq_rows32.hip) and its route."""
from __future__ import annotations

import numpy as np
import pytest

import dynalm_amd as dq
from dqtest import activations, gguf_weights, weight_rows
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

TYPES32 = [O.Q8_0, O.Q4_0]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def check(t, rows, x, k, y, bias=None):
    acts = O.quantize_act(O.ACT_PER32, x)
    want = O.matmul(t, O.ACT_PER32, rows, acts, k).astype(np.float64)
    mag = np.abs(x.astype(np.float64)) @ np.abs(O.expand_x86(t, rows, k).astype(np.float64)).T
    b = 0.0 if bias is None else bias
    # K / 32 terms, each and each partial sum rounded once, in two orders; codes are up to half
    # a step above |x|
    bound = (k / 32 + 16) * 2.0**-23 * 1.1 * (mag + np.abs(b) + np.abs(want))
    assert np.all(np.abs(y - (want + b)) <= bound + 1e-30)


# m, n, K: 16-, 32- and 64-row workgroups (tiles of 16 rows against 1.5 and 3 per CU), one
# block to a partial last step of four, one to three passes with a short last one
@pytest.mark.parametrize("t", TYPES32, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("m,n,k", [(3, 1, 32), (4, 17, 64), (5, 130, 96), (16, 63, 1312), (17, 200, 2048), (12, 4100, 160),
                                   (8, 6200, 256), (5, 12300, 288), (11, 14336, 128), (48, 65, 8192), (33, 40, 8224)])
def test_against_oracle(cuda, t, m, n, k):
    import dqtorch as T

    rows = gguf_weights(t, n, k, 6100 + t + m)
    x = activations(m, k, 6200 + m)
    bias = O.normal(6300 + m, n)
    w = dq.Weight.upload(t, rows, k)
    xs = np.zeros((m, k + 5), np.float32)
    xs[:, :k] = x
    xd = dev(xs)
    y = torch.zeros((m, n + 3), device="cuda")
    dq.matmul(w, xd, m, k + 5, y, n + 3, dev(bias), T.stream())
    got = host(y)
    assert not got[:, n:].any()
    check(t, rows, x, k, got[:, :n], bias)
    # the same bits from separately quantized rows (the GEMM's own from 13), and for any range
    # of weight rows
    acts = T.quantize(O.ACT_PER32, xd[:, :k].contiguous())
    z = torch.zeros((m, n), device="cuda")
    dq.gemv(w, dq.ACT_PER32, acts, m, 0, n, z, n, dev(bias), T.stream())
    full = host(z).copy()
    check(t, rows, x, k, full, bias)
    if m < 13:
        assert np.array_equal(full.view(np.uint32), got[:, :n].copy().view(np.uint32))
    n0, n1 = n // 3, n - n // 4
    z.zero_()
    dq.gemv(w, dq.ACT_PER32, acts, m, n0, n1, z, n, dev(bias), T.stream())
    part = host(z)
    assert np.array_equal(part[:, n0:n1].copy().view(np.uint32), full[:, n0:n1].copy().view(np.uint32))
    assert not part[:, :n0].any() and not part[:, n1:].any()


@pytest.mark.parametrize("t", TYPES32, ids=lambda t: O.TYPE_NAMES[t])
def test_saturated_codes(cuda, t):
    """Edge weight blocks (extreme codes and scales) against rows of full-scale codes."""
    import dqtorch as T

    m, n, k = 9, 64, 1024
    rows = weight_rows(t, n, k, 6400 + t, edge=True)
    x = np.where(np.arange(m * k).reshape(m, k) % 3 == 0, -1.0, 1.0).astype(np.float32)
    x[4] = 0.0
    w = dq.Weight.upload(t, rows, k)
    got = host(T.matmul(w, dev(x)))
    want = O.matmul(t, O.ACT_PER32, rows, O.quantize_act(O.ACT_PER32, x), k).astype(np.float64)
    mag = np.abs(x.astype(np.float64)) @ np.abs(O.expand_x86(t, rows, k).astype(np.float64)).T
    fine = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fine)
    assert np.all(np.abs(got - want)[fine] <= ((k / 32 + 16) * 2.0**-23 * 2 * mag + 1e-30)[fine])


@pytest.mark.parametrize("t", TYPES32, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("k", [96, 128, 160, 224])
def test_infinite_last_block(cuda, t, k):
    """An infinity or a NaN in a row's last block, which the lanes of a short last step repeat:
    each output is the infinity or NaN that the contract's order and the one-row call give."""
    import dqtorch as T

    m, n = 12, 64
    rows = gguf_weights(t, n, k, 6700 + t)
    x = activations(m, k, 6701)
    x[1, k - 3], x[2, k - 5], x[3, k - 1], x[4, 0] = np.inf, -np.inf, np.nan, np.inf
    w = dq.Weight.upload(t, rows, k)
    want = O.matmul(t, O.ACT_PER32, rows, O.quantize_act(O.ACT_PER32, x), k)
    one = np.concatenate([host(T.matmul(w, dev(x[r : r + 1]))).copy() for r in range(m)])
    for rr in (3, 5, 8, m):
        got = host(T.matmul(w, dev(x[:rr])))
        for ref in (want[:rr], one[:rr]):
            odd = ~np.isfinite(ref)
            assert np.array_equal(~np.isfinite(got), odd)
            assert np.array_equal(got[odd], ref[odd], equal_nan=True)
    assert np.isinf(want).any()


# N, K: every split of K -- 16 slices in 16-, 32- and 64-row workgroups, 8 slices (more row groups
# than CUs), two to eight ranges of 8 -- with slices of no, a few and uneven blocks
@pytest.mark.parametrize("t", TYPES32, ids=lambda t: O.TYPE_NAMES[t])
@pytest.mark.parametrize("n,k", [(70, 32), (300, 1504), (6200, 416), (14336, 96), (16500, 160), (6000, 8192), (7000, 8224),
                                 (5000, 8192), (4096, 8288), (3100, 8192), (2600, 8224), (2304, 8192), (130, 14336),
                                 (200, 7360), (6200, 6144), (9000, 11008)])
def test_the_one_row_bits(cuda, t, n, k):
    """A row's outputs are the one-row call's bit for bit whatever the rows beside it, from fp32 rows
    and from quantized ones, and for rows whose scales and products fall below the normal range."""
    import dqtorch as T

    rows = gguf_weights(t, min(n, 128), k, 6800 + t)
    rows = np.tile(rows, (-(-n // rows.shape[0]), 1))[:n].copy()
    w = dq.Weight.upload(t, rows, k)
    x = activations(16, k, 6801)
    x[2] *= np.float32(1e-36)
    x[5] *= np.float32(1e-39)
    x[7] *= np.float32(1e34)
    xd = dev(x)
    acts = T.quantize(O.ACT_PER32, xd)
    one = np.concatenate([host(T.matmul(w, xd[r : r + 1].contiguous())).copy() for r in range(16)])
    for m in (3, 4, 5, 8, 12, 16):
        z = torch.zeros((m, n), device="cuda")
        dq.gemv(w, dq.ACT_PER32, acts, m, 0, n, z, n, None, T.stream())
        assert np.array_equal(host(z).view(np.uint32), one[:m].view(np.uint32))
        if m < 13:
            assert np.array_equal(host(T.matmul(w, xd[:m].contiguous())).view(np.uint32), one[:m].view(np.uint32))


def test_first_call_under_capture(cuda):
    """A stream whose workspace is not there yet and cannot be allocated (capture): the call
    still runs, on the GEMV that needs none; three replays beside eager work."""
    m, n, k = 8, 300, 512
    rows = gguf_weights(O.Q4_0, n, k, 6500)
    w = dq.Weight.upload(O.Q4_0, rows, k)
    x = activations(m, k, 6501)
    xd, y, e = dev(x), torch.zeros((m, n), device="cuda"), torch.zeros((m, n), device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        dq.matmul(w, xd, m, k, y, n, None, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        y.zero_()
        g.replay()
        check(O.Q4_0, rows, x, k, host(y))
        dq.matmul(w, xd, m, k, e, n, None, torch.cuda.current_stream().cuda_stream)
        check(O.Q4_0, rows, x, k, host(e))


def test_threads_on_the_per_thread_default_stream(cuda):
    """Threads that each pass hipStreamPerThread (handle 2) at once have their own rows' outputs."""
    import ctypes
    import threading

    m, n, k = 8, 2000, 1024
    rows = gguf_weights(O.Q4_0, n, k, 6950)
    w = dq.Weight.upload(O.Q4_0, rows, k)
    hip = ctypes.CDLL("libamdhip64.so")
    xs = [dev(activations(m, k, 6951 + i)) for i in range(4)]
    ys = [[torch.zeros((m, n), device="cuda") for _ in range(50)] for _ in xs]
    want = []
    for x in xs:
        y = torch.zeros((m, n), device="cuda")
        dq.matmul(w, x, m, k, y, n, None, torch.cuda.current_stream().cuda_stream)
        want.append(host(y).copy())
    rc = []

    def calls(i):
        for y in ys[i]:
            dq.matmul(w, xs[i], m, k, y, n, None, 2)
        rc.append(hip.hipStreamSynchronize(ctypes.c_void_p(2)))

    threads = [threading.Thread(target=calls, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert rc == [0] * len(xs)
    for i, y in enumerate(ys):
        for z in y:
            assert np.array_equal(host(z), want[i])


def test_beside_another_threads_capture(cuda):
    """The first call on a stream (which allocates its workspace) while another thread captures: the
    call runs and the capture stays valid."""
    import ctypes
    import threading

    m, n, k = 8, 300, 512
    rows = gguf_weights(O.Q4_0, n, k, 6900)
    w = dq.Weight.upload(O.Q4_0, rows, k)
    x = activations(m, k, 6901)
    xd, y, z = dev(x), torch.zeros((m, n), device="cuda"), torch.zeros(8, device="cuda")
    hip = ctypes.CDLL("libamdhip64.so")
    fresh = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(fresh)) == 0
    err = []

    def call():
        try:
            dq.matmul(w, xd, m, k, y, n, None, fresh.value)
        except Exception as e:  # noqa: BLE001
            err.append(e)

    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        z.fill_(1.0)
        t = threading.Thread(target=call)
        t.start()
        t.join()
    assert not err
    assert hip.hipStreamSynchronize(fresh) == 0
    check(O.Q4_0, rows, x, k, host(y))
    g.replay()
    assert host(z).all()
    assert hip.hipStreamDestroy(fresh) == 0


@pytest.mark.parametrize("t", TYPES32, ids=lambda t: O.TYPE_NAMES[t])
def test_capture_outlives_the_stream_workspace(cuda, t):
    """A call captured on a stream that has a workspace does not use it: the graph replays
    right after a larger call on the stream has replaced the workspace."""
    import dqtorch as T

    m, n, k, kb = 8, 300, 512, 14336
    rows, big = gguf_weights(t, n, k, 6600 + t), gguf_weights(O.Q4_K, 64, kb, 6610)
    w, wb = dq.Weight.upload(t, rows, k), dq.Weight.upload(O.Q4_K, big, kb)
    x = activations(m, k, 6601)
    xd, y, e = dev(x), torch.zeros((m, n), device="cuda"), torch.zeros((m, n), device="cuda")
    # dq_gemm's activation layouts: 2 B a value and more in the stream's workspace, 7 MB and up
    acts = [T.quantize(O.ACT_PER32, torch.ones((b, kb), device="cuda")) for b in (256, 512, 1024)]
    yb = torch.zeros((1024, 64), device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    dq.matmul(w, xd, m, k, e, n, None, s.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        dq.matmul(w, xd, m, k, y, n, None, s.cuda_stream)
    for a in acts:
        dq.gemm(wb, dq.ACT_PER32, a, a.shape[0], 0, 64, yb, 64, None, s.cuda_stream)
        torch.cuda.synchronize()
        y.zero_()
        g.replay()
        check(t, rows, x, k, host(y))
