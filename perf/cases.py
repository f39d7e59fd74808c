"""The matmul calls whose time is measured, each as a user's program makes it.

An inference program keeps its weights on the GPU (`Weight`), has fp32 activation rows in
device memory and calls the Python mirror of the C ABI: `matmul`, `matmul_many`,
`matmul_gated` (dynacore's Device::matmul and its neighbours) or `matmul_plan` under the
plan of the step. The listed cases are the decode and prefill calls of Q4_K_M, Q8_0 and
Q4_0 models with the shapes of the tests and the benchmark; `draw` spreads shapes, row
counts, weight types, plans, bias and row strides over the same ranges.
"""
from __future__ import annotations

import math

import torch

import dynalm_amd as dq

TYPES = {"q4_0": dq.Q4_0, "q8_0": dq.Q8_0, "q4_k": dq.Q4_K, "q6_k": dq.Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}
KQUANTS = ("q4_k", "q6_k")
UNBOUNDED = 1 << 30

# A case: entry "matmul" (plan: the plan's name, "" for dq.matmul), "many" (q, k and v on one
# input), "gated" (SiLU) or "layer" (q/k/v, o, gate/up and down of a transformer layer; the
# norms and attention between them are not this framework's, so each has an input of its own);
# type: of the weights ("layer": of all but down, which is Q6_K); m rows of k values; n output
# rows ("layer": k is the model's width, n the k and v rows, ffn the MLP's width); layers: how
# many layers' weights a pass goes through, so that weights come from HBM as in a decode step.
_DEFAULTS = {"plan": "", "layers": 1, "bias": False, "wide": False, "ffn": 0}


def _case(name: str, **kw) -> dict:
    return {"name": name, **_DEFAULTS, **kw}


def listed() -> list[dict]:
    return [
        # one sequence's attention projections of a small model: the smallest call, all latency
        _case("decode_qkv_m1", entry="many", type="q4_k", m=1, n=256, k=1536),
        # one sequence through the gate (or up) projections of an 8B model's layers
        _case("decode_gate_m1", entry="matmul", type="q4_k", m=1, n=14336, k=4096, layers=16),
        # the same model's FFN down under the engine's plan for it (int16 activations)
        _case("decode_down_int16_m1", entry="matmul", plan="down", type="q6_k", m=1, n=4096, k=14336, layers=6),
        # eight sequences on a Q4_0 model
        _case("decode_q4_0_m8", entry="matmul", type="q4_0", m=8, n=14336, k=4096, layers=8),
        # sixteen sequences through the layers of a 1.5B model
        _case("decode_layers_m16", entry="layer", type="q4_k", m=16, n=256, k=1536, ffn=8960, layers=8),
        # and its output head
        _case("decode_head_m16", entry="matmul", type="q6_k", m=16, n=151936, k=1536),
        # a short prompt's rows, ragged, with a bias and rows inside wider buffers, engine's plan
        _case("batch_ragged_m77", entry="matmul", plan="engine", type="q4_k", m=77, n=5003, k=2304, bias=True, wide=True),
        # prefill of an 8B model: gate with super-block activations, with the engine's per-32
        # ones, its down projection with int16 ones, and the fp32 activations of the default plan
        _case("prefill_gate_m512", entry="matmul", type="q4_k", m=512, n=14336, k=4096),
        _case("prefill_gate_per32_m512", entry="matmul", plan="engine", type="q4_k", m=512, n=14336, k=4096),
        _case("prefill_down_int16_m512", entry="matmul", plan="down", type="q6_k", m=512, n=4096, k=14336),
        _case("prefill_gate_f32_m512", entry="matmul", plan="default", type="q4_k", m=512, n=14336, k=4096),
        # prefill of a Q8_0 model's square projection
        _case("prefill_q8_0_m512", entry="matmul", type="q8_0", m=512, n=4096, k=4096),
    ]


MOST = 512 * 14336 * 4096  # m n k of the largest listed cases


def draw(rng) -> dict:
    entry = rng.choice(["matmul", "matmul", "matmul", "many", "gated"])
    plan = rng.choice(["", "engine", "down", "default", "subscaled"]) if entry == "matmul" else ""
    typ = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q4_0"])
    if plan == "subscaled" and typ not in KQUANTS:
        typ = "q4_k"
    most_m = 512
    if plan == "subscaled":
        most_m = 8  # the rows that plan runs with sub-scaled activations
    elif plan == "down" and typ not in KQUANTS:
        most_m = 16  # int16 rows of these types run in passes of four
    m = int(round(math.exp(rng.uniform(0.0, math.log(most_m)))))
    unit = BLOCK[typ][0]
    k = unit * max(1, int(math.exp(rng.uniform(math.log(512), math.log(14336))) / unit))
    n = int(math.exp(rng.uniform(math.log(200), math.log(16384))))
    if rng.random() < 0.5:
        n = max(64, n // 64 * 64)
    copies = {"matmul": 1, "many": 3, "gated": 2}[entry]
    while copies * m * n * k > MOST:
        n = n // 2 + 1
    return {**_DEFAULTS, "entry": entry, "plan": plan, "type": typ, "m": m, "n": n, "k": k,
            "bias": entry != "gated" and rng.random() < 0.3,
            "wide": plan != "default" and rng.random() < 0.3}


# ------------------------------------------------------------------ weights and inputs


def _u8(t: torch.Tensor) -> torch.Tensor:
    return t.to(torch.uint8)


def _half(t: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """fp16 bytes of t [..., 1] and its value."""
    h = t.to(torch.float16)
    return h.view(torch.uint8), h.to(torch.float32)


def _safe(t: torch.Tensor) -> torch.Tensor:
    return torch.where(t == 0, torch.ones_like(t), t)


def _encode(typ: str, w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """GGUF blocks [blocks, bytes] of the values w [blocks, values] (plain round-to-nearest
    encoders), and the values they hold in 64 bits."""
    if typ == "q8_0":
        db, d = _half(w.abs().amax(1, keepdim=True) / 127)
        q = (w / _safe(d)).round().clamp(-127, 127)
        return torch.cat([db, q.to(torch.int8).view(torch.uint8)], 1), d.double() * q
    if typ == "q4_0":
        top = w.gather(1, w.abs().argmax(1, keepdim=True))
        db, d = _half(top / -8)
        q = (w / _safe(d)).add(8).round().clamp(0, 15)
        return torch.cat([db, _u8(q[:, :16]) | _u8(q[:, 16:]) << 4], 1), d.double() * (q.double() - 8)
    nb = w.shape[0]
    if typ == "q4_k":
        s = w.view(nb, 8, 32)
        low = (-s.amin(2)).clamp_min(0)
        step = (s.amax(2) + low) / 15
        db, d = _half(step.amax(1, keepdim=True) / 63)
        mb, dmin = _half(low.amax(1, keepdim=True) / 63)
        sc = (step / _safe(d)).round().clamp(0, 63)
        mn = (low / _safe(dmin)).round().clamp(0, 63)
        ds, dm = (d * sc).unsqueeze(2), (dmin * mn).unsqueeze(2)
        q = ((s + dm) / _safe(ds)).round().clamp(0, 15)
        a, b = _u8(sc), _u8(mn)
        scales = torch.cat([a[:, :4] | (a[:, 4:] >> 4) << 6, b[:, :4] | (b[:, 4:] >> 4) << 6,
                            (a[:, 4:] & 15) | (b[:, 4:] & 15) << 4], 1)
        c = _u8(q).view(nb, 4, 2, 32)
        qs = (c[:, :, 0] | c[:, :, 1] << 4).reshape(nb, 128)
        val = (d.double() * sc).unsqueeze(2) * q - (dmin.double() * mn).unsqueeze(2)
        return torch.cat([db, mb, scales, qs], 1), val.view(nb, 256)
    s = w.view(nb, 16, 16)
    step = s.abs().amax(2) / 31
    db, d = _half(step.amax(1, keepdim=True) / 127)
    sc = (step / _safe(d)).round().clamp(-128, 127)
    q = (s / _safe(d * sc).unsqueeze(2)).round().clamp(-32, 31)
    c = _u8(q + 32).view(nb, 2, 4, 32)
    ql = torch.stack([(c[:, :, 0] & 15) | (c[:, :, 2] & 15) << 4, (c[:, :, 1] & 15) | (c[:, :, 3] & 15) << 4], 2)
    qh = c[:, :, 0] >> 4 | (c[:, :, 1] >> 4) << 2 | (c[:, :, 2] >> 4) << 4 | (c[:, :, 3] >> 4) << 6
    blocks = torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc.to(torch.int8).view(torch.uint8), db], 1)
    return blocks, ((d.double() * sc).unsqueeze(2) * q).view(nb, 256)


def _weight_rows(typ: str, n: int, k: int, gen: torch.Generator, exact: bool):
    """n rows of k values as GGUF rows on the GPU, in pieces: (bytes, values in 64 bits or None)."""
    be, bb = BLOCK[typ]
    rows = max(1, (1 << 25) // k)
    raw, val = [], []
    for r0 in range(0, n, rows):
        r = min(rows, n - r0)
        # trained weights: near normal, rows of different size
        w = torch.randn((r, k), generator=gen, device="cuda") * (0.02 * (1 + torch.rand((r, 1), generator=gen, device="cuda")))
        b, v = _encode(typ, w.view(-1, be))
        raw.append(b.view(r, k // be * bb))
        if exact:
            val.append(v.view(r, k))
    return torch.cat(raw), torch.cat(val) if exact else None


def _rows(m: int, k: int, gen: torch.Generator) -> torch.Tensor:
    """Activation rows: per-channel gains and a few outlier channels, as after a norm."""
    gain = torch.exp(0.5 * torch.randn((1, k), generator=gen, device="cuda"))
    gain = torch.where(torch.rand((1, k), generator=gen, device="cuda") < 0.003, gain * 20, gain)
    return torch.randn((m, k), generator=gen, device="cuda") * gain


def _products(case: dict) -> list[tuple]:
    """The calls of one layer: (entry, type, rows of each weight, k)."""
    n, k, t = case["n"], case["k"], case["type"]
    if case["entry"] == "many":
        return [("many", t, [k, n, n] if n < k else [n, n // 4 + 1, n // 4 + 1], k)]
    if case["entry"] == "gated":
        return [("gated", t, [n, n], k)]
    if case["entry"] == "layer":
        f = case["ffn"]
        return [("many", t, [k, n, n], k), ("matmul", t, [k], k), ("gated", t, [f, f], k), ("matmul", "q6_k", [k], f)]
    return [("matmul", t, [n], k)]


def _inputs(case: dict, seed: int, exact: bool = False):
    """Each call's (entry, type, k, x, [(rows, values)], [bias]), from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    for _ in range(case["layers"]):
        for entry, typ, ns, k in _products(case):
            x = _rows(case["m"], k, gen)
            ws = [_weight_rows(typ, n, k, gen, exact) for n in ns]
            bias = [torch.randn(n, generator=gen, device="cuda") if case["bias"] else None for n in ns]
            yield entry, typ, k, x, ns, ws, bias


def _plan(name: str):
    if name == "":
        return None
    p = dq.plan_defaults()
    if name in ("engine", "down"):  # a backend with accelerated qmm kernels: int8 rows at any size
        p.int8_decode_max_rows = UNBOUNDED
    if name == "subscaled":  # the x86 tiers' choice for decode rows
        p.qmm = 0
    return dq.plan_ffn_down(p) if name == "down" else p


def prepare(case: dict, seed: int) -> dict:
    m, pad = case["m"], case["wide"]
    calls = []
    for entry, typ, k, x, ns, ws, bias in _inputs(case, seed):
        weights = [dq.Weight.upload_device(TYPES[typ], raw, n, k, raw.shape[1]) for n, (raw, _) in zip(ns, ws)]
        xs = k + 256 if pad else k
        xb = torch.zeros((m, xs), device="cuda")
        xb[:, :k] = x
        ys = [n + 64 if pad else n for n in (ns[:1] if entry == "gated" else ns)]
        y = [torch.zeros((m, s), device="cuda") for s in ys]
        calls.append((entry, weights, xb, xs, y, ys, ns, bias))
    torch.cuda.synchronize()
    return {"m": m, "plan": _plan(case["plan"]), "calls": calls}


def run(state: dict):
    m, plan = state["m"], state["plan"]
    stream = torch.cuda.current_stream().cuda_stream
    out = []
    for entry, w, x, xs, y, ys, ns, bias in state["calls"]:
        if entry == "many":
            dq.matmul_many([(w[i], x, m, xs, y[i], ys[i], bias[i]) for i in range(len(w))], stream)
        elif entry == "gated":
            dq.matmul_gated(dq.SILU, x, m, xs, w[0], w[1], y[0], ys[0], stream=stream)
        elif plan is None:
            dq.matmul(w[0], x, m, xs, y[0], ys[0], bias[0], stream)
        else:
            dq.matmul_plan(w[0], plan, x, m, xs, y[0], ys[0], bias[0], stream)
        out += [t[:, :n] for t, n in zip(y, ns)]
    return out


def work(case: dict) -> dict:
    m, nbytes, flops = case["m"], 0, 0
    for entry, typ, ns, k in _products(case):
        be, bb = BLOCK[typ]
        outs = ns[:1] if entry == "gated" else ns
        nbytes += sum(ns) * (k // be * bb) + 4 * m * k + 4 * m * sum(outs) + (4 * sum(ns) if case["bias"] else 0)
        flops += 2 * m * k * sum(ns)
    return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}


def tolerance(case: dict) -> dict:
    # fp32 sums of up to 14336 terms in another order, the integers inside a block exact: four
    # times the fp32 class's distance from 64 bits (1.2e-6 at k = 4096, the others 3e-7 at most)
    return {"rel": 5e-6}


# ------------------------------------------------------------------ the same in 64 bits


def _contract(case: dict, typ: str) -> str:
    """The activations' form (dynacore's kernel selection under the case's plan)."""
    plan, m = case["plan"], case["m"]
    if plan == "engine":
        return "per32"
    if plan == "down":
        return "int16"
    if plan == "default":
        return "per32" if m <= 4 else "subscaled" if m <= 8 and typ in KQUANTS else "f32"
    if plan == "subscaled":
        return "subscaled"
    return "q8_k" if typ in KQUANTS else "per32"


def _codes(x: torch.Tensor, scale: torch.Tensor, most: float) -> torch.Tensor:
    """x at its scale, the scale's inverse and the product rounded to fp32 as the contracts say."""
    inv = torch.where(scale > 0, torch.ones_like(scale) / _safe(scale), torch.zeros_like(scale))
    return (x * inv).round().clamp(-most, most)


def _over(t: torch.Tensor, by: float) -> torch.Tensor:
    return t / torch.full_like(t, by)  # a tensor: dividing by a number may multiply by its inverse


def _quantized(x: torch.Tensor, contract: str) -> torch.Tensor:
    m, k = x.shape
    if contract == "f32":
        return x.double()
    if contract == "subscaled":
        b = x.view(m, k // 256, 8, 32)
        a32 = b.abs().amax(3, keepdim=True)
        u = _over(a32.amax(2, keepdim=True), 127.0 * 128.0)
        mul = torch.where(u > 0, (a32 / _safe(u * 127.0)).ceil().clamp(1, 128), torch.ones_like(a32))
        s = u * mul
        return (u.double() * mul * _codes(b, s, 127).double()).view(m, k)
    size, most = {"per32": (32, 127.0), "int16": (32, 32767.0), "q8_k": (256, 127.0)}[contract]
    b = x.view(m, k // size, size)
    d = _over(b.abs().amax(2, keepdim=True), most)
    return (d.double() * _codes(b, d, 32768 if most > 127 else most)).view(m, k)


def exact(case: dict, seed: int):
    out = []
    for entry, typ, k, x, ns, ws, bias in _inputs(case, seed, exact=True):
        xq = _quantized(x, _contract(case, typ))
        ys = [xq @ v.t() for _, v in ws]
        if entry == "gated":
            ys = [ys[0] * torch.sigmoid(ys[0]) * ys[1]]
        out += [y if b is None else y + b.double() for y, b in zip(ys, bias)]
    return out
