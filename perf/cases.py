"""The work a program has this library do, as timed cases: the decode and prefill
projections of a GGUF model's layers, the attention between them, the load path,
and a short chat turn through the device runner, all through the C ABI of
include/aether_hip.h.

Shapes are the ones the repository's benchmark and tests use: the LLaMA-8B layer
(hidden 4096, 32 query / 8 KV heads of 128, FFN 14336, vocabulary 128256) and the
2048 / 6144 / 9216 widths around it. Weights are seeded synthetic GGUF blocks as
the benchmark describes them (f16 block scales |N(0,1)|·0.01, quants and
sub-scales uniform), activations N(0,1).

A decode case walks `layers` weights one after the other, as a decode step does:
a weight is not in a cache when its turn comes.
"""
import ctypes
import math

import numpy as np
import torch

import aether_amd as A

F16, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K = 1, 8, 10, 11, 12, 13, 14
DTYPES = {"f16": F16, "q8_0": Q8_0, "q2_k": Q2_K, "q3_k": Q3_K, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
GGUF_ORDER = (F16, Q2_K, Q3_K)  # kept as the file's [k][n] tensor; the others are [n][k] rows of blocks
HEAD_DIM = 128


def geometry(name):
    return A.block_geometry(DTYPES[name])


def weight_bytes(name, n, k):
    be, bb = geometry(name)
    return n * k // be * bb


# ── the cases ─────────────────────────────────────────────────────────────


def listed():
    return [
        # the K or V projection of a Q8_0 model's decode step: the smallest call, launch-bound
        dict(name="decode_kv_q8_0", kind="matmul", dtype="q8_0", m=1, n=1024, k=4096, layers=24, flags=""),
        # gate or up projection of a Q4_K decode step, the bulk of a step's weight bytes
        dict(name="decode_ffn_q4_k", kind="matmul", dtype="q4_k", m=1, n=14336, k=4096, layers=4, flags=""),
        # the LM head, the largest matrix of a step
        dict(name="decode_head_q6_k", kind="matmul", dtype="q6_k", m=1, n=128256, k=4096, layers=1, flags=""),
        # the same gate / up projection of a Q3_K_M model: the file's [k][n] tensor as it is
        dict(name="decode_ffn_q3_k", kind="matmul", dtype="q3_k", m=1, n=14336, k=4096, layers=4, flags=""),
        # a few rows at once: a very short prompt, a drafted continuation, a handful of sequences
        dict(name="batch7_ffn_q4_k", kind="matmul", dtype="q4_k", m=7, n=14336, k=4096, layers=4, flags=""),
        # prefill of a 512-token prompt, gate or up projection
        dict(name="prefill_ffn_q4_k", kind="matmul", dtype="q4_k", m=512, n=14336, k=4096, layers=1, flags=""),
        # prefill of a 203-token prompt in a Q3_K_M model, q or o projection
        dict(name="prefill_q_q3_k", kind="matmul", dtype="q3_k", m=203, n=4096, k=4096, layers=1, flags=""),
        # prefill of a 333-token prompt in an unquantised F16 model, q or o projection
        dict(name="prefill_q_f16", kind="matmul", dtype="f16", m=333, n=4096, k=4096, layers=1, flags=""),
        # decode attention of an 8B-shape layer deep into its 4096-position cache
        dict(name="attn_decode_3000", kind="attn_decode", heads=32, kv_heads=8, seq=3000, max_seq=4096, layers=4),
        # causal attention of a long prompt
        dict(name="attn_prefill_2000", kind="attn_prefill", heads=32, kv_heads=8, n=2000, max_seq=4096),
        # model load: one FFN tensor of a file, transposed and re-quantised into row blocks
        dict(name="load_ffn_q4_k", kind="load", dtype="q4_k", k=4096, n=14336),
        # a chat turn through the runner, Q4_K_M mix: prompt, then a few tokens with their logits
        dict(name="chat_q4_k_m", kind="chat", layers=4, d_model=4096, heads=32, kv_heads=8, d_ff=14336, vocab=32000,
             max_seq=1024, prompt=200, steps=6),
    ]


def spread(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "prefill", "prefill", "attn_decode", "attn_prefill", "load", "chat"])
    if kind in ("decode", "batch", "prefill"):
        name = rng.choice(["f16", "q8_0", "q2_k", "q3_k", "q4_k", "q4_k", "q5_k", "q6_k"])
        gguf = DTYPES[name] in GGUF_ORDER
        k = spread(rng, 1024, 14336, 32 if name == "q8_0" else 256)
        n = spread(rng, 1024, min(28672, 14336 * 4096 // k), 256 if name in ("q2_k", "q3_k") else 4 if gguf else 1)
        m = 1 if kind == "decode" else spread(rng, 2, 16) if kind == "batch" else spread(rng, 17, 512)
        layers = 1 if kind == "prefill" else max(1, min(24, (128 << 20) // weight_bytes(name, n, k)))
        # the residual projections accumulate; the int8 dot-product mode exists for the row-block formats
        flags = rng.choice(["", "", "acc", "" if gguf else "q8"])
        return dict(kind="matmul", dtype=name, m=m, n=n, k=k, layers=layers, flags=flags)
    if kind == "attn_decode":
        heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 8), (32, 4), (24, 8), (32, 32)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, seq=spread(rng, 1, 4096), max_seq=4096, layers=4)
    if kind == "attn_prefill":
        heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 8), (32, 4), (24, 8)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, n=spread(rng, 16, 2000 if heads != 24 else 500),
                    max_seq=4096)
    if kind == "load":
        name = rng.choice(["q8_0", "q4_k", "q5_k", "q6_k"])
        k = spread(rng, 1024, 14336, 32 if name == "q8_0" else 256)
        n = spread(rng, 1024, 14336 * 4096 // k)
        return dict(kind=kind, dtype=name, k=k, n=n)
    return dict(kind=kind, layers=rng.choice([1, 2, 3, 4]), d_model=rng.choice([2048, 4096]), heads=32,
                kv_heads=rng.choice([8, 4]), d_ff=rng.choice([6144, 9216, 14336]), vocab=32000, max_seq=1024,
                prompt=spread(rng, 1, 200), steps=rng.randint(1, 6))


# ── inputs ────────────────────────────────────────────────────────────────


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(0xAE7E + int(seed))


def normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def blocks(g, name, count):
    """`count` raw blocks of a format as the benchmark describes them: uint8 [count][block bytes]."""
    if name == "f16":
        return (normal(g, count) * 0.05).half().view(torch.uint8).reshape(count, 2)
    be, bb = geometry(name)
    raw = torch.randint(0, 256, (count, bb), generator=g, device="cuda", dtype=torch.uint8)

    def scale():
        return (normal(g, count).abs() * 0.01).half().view(torch.uint8).reshape(count, 2)

    if name == "q8_0":
        raw[:, 2:] = torch.randint(-127, 128, (count, 32), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        raw[:, 0:2] = scale()
    elif name in ("q4_k", "q5_k", "q2_k"):
        raw[:, 0:2] = scale()
        raw[:, 2:4] = scale()
    elif name == "q3_k":
        raw[:, 108:110] = scale()
    else:
        raw[:, 192:208] = torch.randint(-64, 64, (count, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        raw[:, 208:210] = scale()
    return raw


class Weight:
    """A registered weight, freed with its owner."""

    def __init__(self, name, n, k, raw):
        h = ctypes.c_void_p()
        A.check(A.lib().aeth_weight_create(DTYPES[name], n, k, raw.data_ptr(), 1, None, ctypes.byref(h)), "weight")
        self.handle = h

    def __del__(self):
        A.lib().aeth_weight_free(self.handle)


class Runner:
    def __init__(self, handle):
        self.handle = handle

    def __del__(self):
        A.lib().aeth_runner_free(self.handle)


def host(t):
    return t.cpu().numpy()


def matmul_inputs(case, g):
    """raw blocks of every layer's weight, the activations [layers][m][k] and the residual rows."""
    be = geometry(case["dtype"])[0]
    raws = [blocks(g, case["dtype"], case["n"] * case["k"] // be) for _ in range(case["layers"])]
    x = normal(g, case["layers"], case["m"], case["k"])
    res = normal(g, case["m"], case["n"]) if case["flags"] == "acc" else None
    return raws, x, res


def attn_inputs(case, g):
    nh, nkv, layers = case["heads"], case["kv_heads"], case.get("layers", 1)
    q = normal(g, layers, case.get("n", 1), nh * HEAD_DIM)
    kv = normal(g, layers, 2, nkv, case["max_seq"], HEAD_DIM)
    return q, kv


# a Q4_K_M file keeps attn_v and ffn_down in Q6_K
CHAT_DTYPES = ("q4_k", "q4_k", "q6_k", "q4_k", "q4_k", "q4_k", "q6_k")


def chat_shapes(case):
    d, qd, kvd, dff = case["d_model"], case["heads"] * HEAD_DIM, case["kv_heads"] * HEAD_DIM, case["d_ff"]
    return [(qd, d), (kvd, d), (kvd, d), (d, qd), (dff, d), (dff, d), (d, dff)]


def chat_weights(case, g):
    """Row-block weights whose products stay at activation scale (block scales shrunk by the row length)."""

    def weight(name, n, k):
        raw = blocks(g, name, n * k // 256)
        at, div = (208, 45.0) if name == "q6_k" else (0, 110.0)
        s = (normal(g, raw.shape[0]).abs() * (0.01 / div) * math.sqrt(4096 / k)).half()
        raw[:, at:at + 2] = s.view(torch.uint8).reshape(-1, 2)
        if name == "q4_k":  # a zero-mean weight: dmin·m balances d·sc·q
            raw[:, 2:4] = (s.float() * 7.5).half().view(torch.uint8).reshape(-1, 2)
            raw[:, 8:12] = raw[:, 4:8]
            raw[:, 12:16] = (raw[:, 12:16] & 15) * 17
        return raw

    d = case["d_model"]
    layers = []
    for _ in range(case["layers"]):
        ws = [weight(t, n, k) for t, (n, k) in zip(CHAT_DTYPES, chat_shapes(case))]
        layers.append((ws, 1 + normal(g, d, std=0.02), 1 + normal(g, d, std=0.02)))
    final = 1 + normal(g, d, std=0.02)
    head = weight("q6_k", case["vocab"], d)
    emb = normal(g, case["vocab"], d)
    tokens = torch.randint(0, case["vocab"], (case["prompt"] + case["steps"],), generator=g, device="cuda", dtype=torch.int32)
    return layers, final, head, emb, tokens


def prepare(case, seed):
    L = A.lib()
    A.check(L.aeth_init(0), "aeth_init")
    g = generator(seed)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    kind = case["kind"]
    if kind == "matmul":
        raws, x, res = matmul_inputs(case, g)
        m, n, k = case["m"], case["n"], case["k"]
        ws = [Weight(case["dtype"], n, k, r) for r in raws]
        flags = {"": 0, "acc": A.MM_ACCUMULATE, "q8": A.MM_Q8_ACTIVATIONS}[case["flags"]]
        # with accumulate every layer adds to the same residual rows, else each layer has its output
        y = torch.empty(*((m, n) if res is not None else (len(ws), m, n)), device="cuda")
        outs = [y if res is not None else y[i] for i in range(len(ws))]
        calls = [(w.handle, ctypes.c_void_p(x[i].data_ptr()), m, ctypes.c_void_p(outs[i].data_ptr()), flags, stream)
                 for i, w in enumerate(ws)]
        torch.cuda.synchronize()
        return dict(kind=kind, call=L.aeth_qmatmul, calls=calls, keep=(ws, x), res=res, y=y)
    if kind == "attn_decode":
        q, kv = attn_inputs(case, g)
        y = torch.empty(case["layers"], case["heads"] * HEAD_DIM, device="cuda")
        calls = [(q[i].data_ptr(), kv[i].data_ptr(), case["heads"], case["kv_heads"], HEAD_DIM, case["max_seq"],
                  case["seq"], y[i].data_ptr(), stream) for i in range(case["layers"])]
        return dict(kind=kind, call=L.aeth_attn_decode, calls=calls, keep=(q, kv), res=None, y=y)
    if kind == "attn_prefill":
        q, kv = attn_inputs(case, g)
        y = torch.empty(case["n"], case["heads"] * HEAD_DIM, device="cuda")
        calls = [(q.data_ptr(), case["heads"] * HEAD_DIM, kv.data_ptr(), case["n"], case["heads"], case["kv_heads"],
                  HEAD_DIM, case["max_seq"], y.data_ptr(), stream)]
        return dict(kind=kind, call=L.aeth_attn_prefill, calls=calls, keep=(q, kv), res=None, y=y)
    if kind == "load":
        be, bb = geometry(case["dtype"])
        k, n = case["k"], case["n"]
        src = blocks(g, case["dtype"], k * n // be)
        dst = torch.empty(n * (k // be) * bb, dtype=torch.uint8, device="cuda")
        ws = torch.empty(L.aeth_load_quant_ws_bytes(k, n), dtype=torch.uint8, device="cuda")
        calls = [(DTYPES[case["dtype"]], src.data_ptr(), k, n, dst.data_ptr(), ws.data_ptr(), stream)]
        return dict(kind=kind, call=L.aeth_load_quant, calls=calls, keep=(src, ws), res=None, y=dst)
    layers, final, head, emb, tokens = chat_weights(case, g)
    d, vocab = case["d_model"], case["vocab"]
    raw = [host(w) for ws, _, _ in layers for w in ws]
    norms = [host(t) for _, a, f in layers for t in (a, f)]
    final, head, emb = host(final), host(head), host(emb)
    cfg = A.LlamaConfig(vocab, d, case["layers"], case["heads"], case["kv_heads"], HEAD_DIM, case["d_ff"],
                        case["max_seq"], 500000.0, 1e-5, 0, 0)
    dts = (ctypes.c_int32 * len(raw))(*([DTYPES[t] for t in CHAT_DTYPES] * case["layers"]))
    pr = (ctypes.c_void_p * len(raw))(*[a.ctypes.data for a in raw])
    pn = (ctypes.c_void_p * len(norms))(*[a.ctypes.data for a in norms])
    h = ctypes.c_void_p()
    A.check(L.aeth_runner_create(ctypes.byref(cfg), pr, dts, pn, final.ctypes.data, head.ctypes.data, DTYPES["q6_k"],
                                 emb.ctypes.data, 0, ctypes.byref(h)), "runner")
    tokens = np.ascontiguousarray(host(tokens))
    logits = np.empty((case["steps"] + 1, vocab), np.float32)
    return dict(kind=kind, runner=Runner(h), prompt=case["prompt"], tokens=tokens, logits=logits)


def run(state):
    if state["kind"] == "chat":
        L, h, n = A.lib(), state["runner"].handle, state["prompt"]
        logits, tokens = state["logits"], state["tokens"]
        rc = L.aeth_runner_prefill(h, tokens.ctypes.data, n, logits[0].ctypes.data, None)
        for i in range(1, len(logits)):
            rc |= L.aeth_runner_decode(h, int(tokens[n + i - 1]), n + i - 1, logits[i].ctypes.data, None)
        A.check(rc, "chat")
        return logits
    if state["res"] is not None:
        state["y"].copy_(state["res"])
    call = state["call"]
    for args in state["calls"]:
        rc = call(*args)
        if rc:
            A.check(rc, "call")
    return state["y"]


# ── what a pass cannot do without ─────────────────────────────────────────


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, n, k, layers = case["m"], case["n"], case["k"], case["layers"]
        rows = 2 if case["flags"] == "acc" else layers  # the residual rows, once in and once out, or every output
        return dict(bytes=layers * (weight_bytes(case["dtype"], n, k) + 4 * m * k) + 4 * m * n * rows,
                    flops=2.0 * m * n * k * layers)
    if kind == "attn_decode":
        nh, nkv, seq, layers = case["heads"], case["kv_heads"], case["seq"], case["layers"]
        return dict(bytes=4 * HEAD_DIM * layers * (2 * nkv * seq + 2 * nh), flops=4.0 * nh * seq * HEAD_DIM * layers)
    if kind == "attn_prefill":
        nh, nkv, n = case["heads"], case["kv_heads"], case["n"]
        return dict(bytes=4 * HEAD_DIM * n * (2 * nkv + 2 * nh), flops=2.0 * nh * n * (n + 1) * HEAD_DIM)
    if kind == "load":
        return dict(bytes=2 * weight_bytes(case["dtype"], case["n"], case["k"]), flops=0)
    n, steps, layers = case["prompt"], case["steps"], case["layers"]
    shapes = chat_shapes(case)
    wb = layers * sum(weight_bytes(t, a, b) for t, (a, b) in zip(CHAT_DTYPES, shapes))
    wf = layers * sum(2.0 * a * b for a, b in shapes)
    head = weight_bytes("q6_k", case["vocab"], case["d_model"])
    kv_row = 2 * 4 * HEAD_DIM * case["kv_heads"] * layers
    seen = sum(n + i for i in range(1, steps + 1))
    return dict(bytes=(1 + steps) * (wb + head + 4 * case["vocab"]) + kv_row * (n + seen),
                flops=(n + steps) * wf + (1 + steps) * 2.0 * case["vocab"] * case["d_model"] +
                4.0 * HEAD_DIM * case["heads"] * layers * (n * (n + 1) / 2 + seen))


def tolerance(case):
    """Products and sums are f32 or better: against float64 the products come to 1e-7 .. 4e-7 of a result
    (the longest f32 chains, an F16 product, most), attention to 2e-7, and a chat turn, which carries the
    rounding of every layer before it, to 2e-6. About four times that. Loaded blocks are bytes."""
    kind = case["kind"]
    if kind == "load":
        return "exact"
    return {"rel": {"matmul": 4e-6, "attn_decode": 2e-6, "attn_prefill": 2e-6, "chat": 1e-5}[kind]}


# ── the same in float64 ───────────────────────────────────────────────────


def f16_at(raw, at):
    return raw[:, at:at + 2].contiguous().view(torch.float16).double()  # [blocks][1]


def bits(t, shift, mask):
    return ((t >> shift) & mask).double()


def k4_scales(raw):
    """The eight 6-bit scales and mins of the 12 bytes a Q4_K / Q5_K block keeps at byte 4."""
    a, b, c = raw[:, 4:8], raw[:, 8:12], raw[:, 12:16]
    sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], 1).double()
    mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], 1).double()
    return sc, mn


def dequantise(name, raw):
    """Raw blocks → float64 values, block after block."""
    if name == "f16":
        return raw.contiguous().view(torch.float16).double().reshape(-1)
    nb = raw.shape[0]
    if name == "q8_0":
        return (f16_at(raw, 0) * raw[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if name in ("q4_k", "q5_k"):
        sc, mn = k4_scales(raw)
        qs = raw[:, 16:] if name == "q4_k" else raw[:, 48:]
        q = torch.stack([bits(qs, 0, 15).reshape(nb, 4, 32), bits(qs, 4, 15).reshape(nb, 4, 32)], 2).reshape(nb, 8, 32)
        if name == "q5_k":
            shift = torch.arange(8, device=raw.device, dtype=torch.uint8)
            q += 16 * ((raw[:, 16:48, None] >> shift) & 1).double().reshape(nb, 8, 32)
        d, dmin = f16_at(raw, 0), f16_at(raw, 2)
        return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).reshape(-1)
    if name == "q6_k":
        ql, qh = raw[:, :128].reshape(nb, 2, 2, 32), raw[:, 128:192].reshape(nb, 2, 32)
        low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        high = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).double().reshape(nb, 16, 16) - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double()
        return ((f16_at(raw, 208) * sc)[:, :, None] * q).reshape(-1)
    qs = raw[:, 20:84] if name == "q2_k" else raw[:, 32:96]
    q = torch.stack([(qs.reshape(nb, 2, 32) >> s) & 3 for s in (0, 2, 4, 6)], 2).double()  # [blocks][2][4][32]
    if name == "q2_k":
        sc = raw[:, 4:20]
        d, dmin = f16_at(raw, 0), f16_at(raw, 2)
        w = (d * bits(sc, 0, 15))[:, :, None] * q.reshape(nb, 16, 16) - (dmin * bits(sc, 4, 15))[:, :, None]
        return w.reshape(-1)
    hm = raw[:, :32]
    hb = torch.stack([(hm >> t) & 1 for t in range(8)], 1).double().reshape(nb, 2, 4, 32)
    s = raw[:, 96:108]
    lo = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
    hi = torch.cat([(s[:, 8:12] >> t) & 3 for t in (0, 2, 4, 6)], 1)
    sc = (lo | (hi << 4)).double() - 32
    return ((f16_at(raw, 108) * sc)[:, :, None] * (q - 4 * (1 - hb)).reshape(nb, 16, 16)).reshape(-1)


def matrix(name, n, k, raw):
    """The weight as float64 [n][k]."""
    w = dequantise(name, raw)
    return w.reshape(k, n).t() if DTYPES[name] in GGUF_ORDER else w.reshape(n, k)


def q8_activations(x):
    """The values of the Q8_0 activation blocks of f32 rows (the int8 dot-product mode's A)."""
    m, k = x.shape
    b = torch.nn.functional.pad(x, (0, -k % 32)).reshape(m, -1, 32)
    d = b.abs().amax(2, keepdim=True) / 127
    q = torch.where(d > 0, torch.round(b * (1 / d)), torch.zeros_like(b)).clamp(-128, 127)
    return (q.double() * d.half().double()).reshape(m, -1)[:, :k]


def attention64(q, kv, heads, kv_heads, first):
    """Causal softmax attention, query i at position first + i; q [n][heads·128], kv [2][kv_heads][seq][128]."""
    n, seq = q.shape[0], kv.shape[2]
    hidden = torch.arange(seq, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    q = q.double().reshape(n, heads, HEAD_DIM)
    y = torch.empty(n, heads, HEAD_DIM, device=q.device, dtype=torch.float64)
    for h in range(heads):
        kk, vv = (kv[j, h // (heads // kv_heads)].double().contiguous() for j in (0, 1))
        s = (q[:, h].contiguous() @ kk.t().contiguous()) / math.sqrt(HEAD_DIM)
        y[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), 1) @ vv
    return y.reshape(n, heads * HEAD_DIM)


def exact(case, seed):
    g = generator(seed)
    kind = case["kind"]
    if kind == "load":
        return None  # bytes
    if kind == "matmul":
        raws, x, res = matmul_inputs(case, g)
        ys = []
        for i, raw in enumerate(raws):
            a = q8_activations(x[i]) if case["flags"] == "q8" else x[i].double()
            ys.append(a @ matrix(case["dtype"], case["n"], case["k"], raw).t().contiguous())
            raws[i] = None
        return torch.stack(ys) if res is None else res.double() + sum(ys)
    if kind == "attn_decode":
        q, kv = attn_inputs(case, g)
        return torch.cat([attention64(q[i], kv[i, :, :, :case["seq"]], case["heads"], case["kv_heads"], case["seq"] - 1)
                          for i in range(case["layers"])])
    if kind == "attn_prefill":
        q, kv = attn_inputs(case, g)
        return attention64(q[0], kv[0, :, :, :case["n"]], case["heads"], case["kv_heads"], 0)
    layers, final, head, emb, tokens = chat_weights(case, g)
    n, nh, nkv = len(tokens), case["heads"], case["kv_heads"]
    half = HEAD_DIM // 2
    freq = np.float32(500000.0) ** (np.float32(-2) * np.arange(half, dtype=np.float32) / np.float32(HEAD_DIM))
    theta = np.arange(n, dtype=np.float32)[:, None] * freq[None, :]  # f32 angles, as the model defines them
    cos, sin = (torch.from_numpy(f(theta)).cuda().double()[:, None, :] for f in (np.cos, np.sin))

    def rms(v, w):
        return v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-5) * w.double()

    def rope(v, count):
        v = v.reshape(n, count, HEAD_DIM)
        a, b = v[..., :half], v[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], 2)

    def times(v, name, shape, raw):
        return v @ matrix(name, *shape, raw).t().contiguous()

    x = emb[tokens.long()].double()
    for ws, attn_norm, ffn_norm in layers:
        t, s = CHAT_DTYPES, chat_shapes(case)
        h = rms(x, attn_norm)
        q = rope(times(h, t[0], s[0], ws[0]), nh)
        k = rope(times(h, t[1], s[1], ws[1]), nkv)
        v = times(h, t[2], s[2], ws[2]).reshape(n, nkv, HEAD_DIM)
        kv = torch.stack([k.transpose(0, 1), v.transpose(0, 1)])
        x = x + times(attention64(q.reshape(n, -1), kv, nh, nkv, 0), t[3], s[3], ws[3])
        h = rms(x, ffn_norm)
        gate, up = times(h, t[4], s[4], ws[4]), times(h, t[5], s[5], ws[5])
        x = x + times(torch.nn.functional.silu(gate) * up, t[6], s[6], ws[6])
    return times(rms(x[case["prompt"] - 1:n], final), "q6_k", (case["vocab"], case["d_model"]), head)
