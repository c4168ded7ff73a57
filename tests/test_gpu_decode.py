"""GPU parity of the decode-step kernels and the device LlamaRunner against
the CPU oracle's restatement of runner.rs (rmsnorm, RoPE, attention, SiLU,
argmax, one full decode step)."""
import ctypes
import threading

import numpy as np
import pytest

import aether_amd as A
from oracle import oracle as O
from tests._model64 import logits64
from tests._models import TINY, build_tiny, oracle_cfg
from tests._util import (F16, F32, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0, assert_close, assert_close_logits,
                         assert_close_rows, weight)

pytestmark = pytest.mark.gpu


def dev(torch, arr):
    return torch.from_numpy(np.ascontiguousarray(arr)).cuda()


@pytest.mark.parametrize("n", [4096, 1024, 8192, 4000, 100])
def test_rmsnorm(gpu, n):
    """Row lengths of the one-pass register kernel (multiples of 1024) and of
    the general loop."""
    torch = gpu
    rng = np.random.default_rng(1)
    x = rng.standard_normal((3, n)).astype(np.float32) * 3
    w = (1 + 0.02 * rng.standard_normal(n)).astype(np.float32)
    xd, wd = dev(torch, x), dev(torch, w)
    od = torch.empty_like(xd)
    A.check(A.lib().aeth_rmsnorm(xd.data_ptr(), wd.data_ptr(), 3, n, 1e-5, od.data_ptr(), None))
    torch.cuda.synchronize()
    ref = np.stack([O.rmsnorm(x[i], w, 1e-5) for i in range(3)])
    assert_close(od.cpu().numpy(), ref, tol=1e-5)


@pytest.mark.parametrize("pos", [0, 1, 2047, 5000])
def test_rope(gpu, pos):
    torch = gpu
    nh, hd, ms = 40, 128, 4096
    s, c = O.precompute_rope(ms, hd, 500000.0)
    x = np.random.default_rng(pos).standard_normal(nh * hd).astype(np.float32)
    xd, sd, cd = dev(torch, x), dev(torch, s), dev(torch, c)  # keep the device tensors alive across the call
    A.check(A.lib().aeth_rope(xd.data_ptr(), nh, hd, pos, sd.data_ptr(), cd.data_ptr(), ms, None))
    torch.cuda.synchronize()
    ref = O.apply_rope(x, nh, hd, pos, s, c, ms)
    assert_close(xd.cpu().numpy(), ref, tol=1e-5)
    if pos == 0:
        assert np.array_equal(xd.cpu().numpy(), x)  # θ = 0: identity


@pytest.mark.parametrize("seq", [1, 63, 64, 65, 127, 128, 129, 2049])
def test_attention_and_kv_append(gpu, seq):
    torch = gpu
    L = A.lib()
    nh, nkv, hd, ms = 32, 8, 128, 2304
    rng = np.random.default_rng(seq)
    kv = rng.standard_normal((2, nkv, ms, hd)).astype(np.float32)
    q = rng.standard_normal(nh * hd).astype(np.float32)
    k_new = rng.standard_normal(nkv * hd).astype(np.float32)
    v_new = rng.standard_normal(nkv * hd).astype(np.float32)
    kvd, kd, vd, qd = dev(torch, kv), dev(torch, k_new), dev(torch, v_new), dev(torch, q)
    slot = seq - 1
    A.check(L.aeth_kv_append(kvd.data_ptr(), kd.data_ptr(), vd.data_ptr(), nkv, hd, ms, slot, None))
    od = torch.empty(nh * hd, dtype=torch.float32, device="cuda")
    A.check(L.aeth_attn_decode(qd.data_ptr(), kvd.data_ptr(), nh, nkv, hd, ms, seq, od.data_ptr(), None))
    torch.cuda.synchronize()
    kv[0, :, slot, :] = k_new.reshape(nkv, hd)
    kv[1, :, slot, :] = v_new.reshape(nkv, hd)
    assert np.array_equal(kvd.cpu().numpy(), kv)
    ref = np.concatenate([O.attn_direct(q[h * hd:(h + 1) * hd], kv[0, h // (nh // nkv)], kv[1, h // (nh // nkv)], seq,
                                        hd) for h in range(nh)])
    assert_close(od.cpu().numpy(), ref, tol=1e-4)


@pytest.mark.parametrize("seq", [1, 65, 700])
def test_attention_ignores_stale_chunk_partials(gpu, seq):
    """The merge loads every chunk slot of its scratch before it reads the
    sequence length; slots past the live chunks hold what an earlier call left.
    An earlier call over 2049 positions with a NaN query leaves NaN partials in
    every slot: a shorter call after it on the same stream must match the
    oracle with no NaN."""
    torch = gpu
    L = A.lib()
    nh, nkv, hd, ms = 32, 8, 128, 2304
    rng = np.random.default_rng(100 + seq)
    kv = rng.standard_normal((2, nkv, ms, hd)).astype(np.float32)
    kvd = dev(torch, kv)
    od = torch.empty(nh * hd, dtype=torch.float32, device="cuda")
    qnan = dev(torch, np.full(nh * hd, np.nan, dtype=np.float32))
    A.check(L.aeth_attn_decode(qnan.data_ptr(), kvd.data_ptr(), nh, nkv, hd, ms, 2049, od.data_ptr(), None))
    torch.cuda.synchronize()
    assert np.isnan(od.cpu().numpy()).all()
    q = rng.standard_normal(nh * hd).astype(np.float32)
    qd = dev(torch, q)
    A.check(L.aeth_attn_decode(qd.data_ptr(), kvd.data_ptr(), nh, nkv, hd, ms, seq, od.data_ptr(), None))
    torch.cuda.synchronize()
    got = od.cpu().numpy()
    ref = np.concatenate([O.attn_direct(q[h * hd:(h + 1) * hd], kv[0, h // (nh // nkv)], kv[1, h // (nh // nkv)], seq,
                                        hd) for h in range(nh)])
    assert np.isfinite(got).all()
    assert_close(got, ref, tol=1e-4)


def test_attention_one_hot(gpu):
    """A query aligned with one cached key far above the rest attends only to
    that position: out = v_t."""
    torch = gpu
    nh, nkv, hd, ms, seq = 4, 1, 128, 256, 200
    kv = np.zeros((2, nkv, ms, hd), dtype=np.float32)
    rng = np.random.default_rng(3)
    kv[1] = rng.standard_normal((nkv, ms, hd))
    kv[0, 0, 77, :] = 1.0
    q = np.full(nh * hd, 10.0, dtype=np.float32)
    od = torch.empty(nh * hd, dtype=torch.float32, device="cuda")
    qd, kvd = dev(torch, q), dev(torch, kv)
    A.check(A.lib().aeth_attn_decode(qd.data_ptr(), kvd.data_ptr(), nh, nkv, hd, ms, seq, od.data_ptr(), None))
    torch.cuda.synchronize()
    got = od.cpu().numpy().reshape(nh, hd)
    for h in range(nh):
        np.testing.assert_allclose(got[h], kv[1, 0, 77], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("nh,nkv,ms,seq", [(64, 8, 4096, 3000), (8, 8, 512, 300), (16, 2, 8192, 8192),
                                           (32, 8, 2688, 2600), (4, 1, 256, 1)])
def test_attention_shapes(gpu, nh, nkv, ms, seq):
    """Query-head groups of 1, 4 and 8; the longest cache (8192 positions: 64
    chunks of 128, past the 32 the merge loads in one batch); back-to-back calls
    of different shapes share one workspace."""
    torch = gpu
    hd = 128
    rng = np.random.default_rng(seq + nh)
    kv = rng.standard_normal((2, nkv, ms, hd)).astype(np.float32)
    g = nh // nkv
    for rep in range(2):
        q = rng.standard_normal(nh * hd).astype(np.float32)
        s = seq if rep == 0 else max(1, seq // 3)
        od = torch.empty(nh * hd, dtype=torch.float32, device="cuda")
        qd, kvd = dev(torch, q), dev(torch, kv)
        A.check(A.lib().aeth_attn_decode(qd.data_ptr(), kvd.data_ptr(), nh, nkv, hd, ms, s, od.data_ptr(), None))
        torch.cuda.synchronize()
        ref = np.concatenate([O.attn_direct(q[h * hd:(h + 1) * hd], kv[0, h // g], kv[1, h // g], s, hd)
                              for h in range(nh)])
        assert_close(od.cpu().numpy(), ref, tol=1e-4, what="attn nh=%d nkv=%d seq=%d" % (nh, nkv, s))


def test_silu_mul_and_add(gpu):
    torch = gpu
    rng = np.random.default_rng(4)
    n = 14336
    g = (rng.standard_normal(n) * 4).astype(np.float32)
    u = rng.standard_normal(n).astype(np.float32)
    gd, ud = dev(torch, g), dev(torch, u)
    A.check(A.lib().aeth_silu_mul(gd.data_ptr(), ud.data_ptr(), n, None))
    A.check(A.lib().aeth_add(gd.data_ptr(), ud.data_ptr(), n, None))
    torch.cuda.synchronize()
    ref = (g * (1.0 / (1.0 + np.exp(-g))) * u + u).astype(np.float32)
    assert_close(gd.cpu().numpy(), ref, tol=1e-5)


def test_argmax_last_max_wins(gpu):
    torch = gpu
    n = 128256
    x = np.random.default_rng(5).standard_normal(n).astype(np.float32)
    x[[10, 50000, 128000]] = 9.0  # ties: the last index wins (Iterator::max_by)
    od = torch.empty(1, dtype=torch.int32, device="cuda")
    xd = dev(torch, x)
    A.check(A.lib().aeth_argmax(xd.data_ptr(), n, od.data_ptr(), None))
    torch.cuda.synchronize()
    assert int(od.cpu()[0]) == 128000 == O.argmax(x)


# Prefill attention (attention_batch, runner.rs:1809-1883) against an f64
# restatement of its formula: s_t = (q·k_t)/√hd for t ≤ i, max-subtracted
# softmax, Σ p_t v_t. Group sizes 1, 2, 4, 8 take the f32-MFMA kernel, 3 the
# f32 VALU one; ragged n against the 16-key and query blocks, n = max_seq with
# a partial last key block (the MFMA kernel's range-checked loads read its rows
# past n as zeros), the 8B shape, and sharp softmaxes (scaled q: the running
# max grows by more than the kernel's rescale threshold).
@pytest.mark.parametrize("n,nh,nkv,max_seq,qs", [(1, 4, 4, 8, 1.0), (70, 8, 2, 96, 1.0), (150, 4, 2, 192, 3.0),
                                                 (33, 8, 1, 40, 1.0), (64, 6, 2, 64, 1.0), (512, 32, 8, 512, 1.0),
                                                 (97, 16, 4, 128, 4.0), (37, 16, 2, 37, 2.0), (45, 4, 4, 45, 1.0),
                                                 (130, 8, 2, 160, 12.0)])
def test_attn_prefill_matches_f64(gpu, n, nh, nkv, max_seq, qs):
    torch = gpu
    hd = 128
    rng = np.random.default_rng(n * 13 + nh)
    stride = (nh + 2 * nkv) * hd
    q = (rng.standard_normal((n, stride)) * qs).astype(np.float32)
    kv = np.zeros((2, nkv, max_seq, hd), dtype=np.float32)
    kv[:, :, :n] = rng.standard_normal((2, nkv, n, hd)).astype(np.float32)
    out = torch.empty(n * nh * hd, dtype=torch.float32, device="cuda")
    qd, kvd = torch.from_numpy(q).cuda(), torch.from_numpy(kv).cuda()  # kept alive across the launch
    A.check(A.lib().aeth_attn_prefill(qd.data_ptr(), stride, kvd.data_ptr(), n, nh, nkv, hd, max_seq,
                                      out.data_ptr(), None), "attn_prefill")
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(n, nh, hd)
    G = nh // nkv
    ref = np.empty((n, nh, hd))
    K = kv[0].astype(np.float64)
    V = kv[1].astype(np.float64)
    for h in range(nh):
        qh = q[:, h * hd:(h + 1) * hd].astype(np.float64)
        sc = qh @ K[h // G, :n].T / np.sqrt(hd)
        sc[np.triu_indices(n, 1)] = -np.inf
        p = np.exp(sc - sc.max(axis=1, keepdims=True))
        ref[:, h] = (p / p.sum(axis=1, keepdims=True)) @ V[h // G, :n]
    assert_close(got.reshape(n, -1), ref.reshape(n, -1), what="attn_prefill n=%d nh=%d nkv=%d" % (n, nh, nkv))
    assert np.abs(got - ref).max() < 1e-5


def attn_prefill64(q, kv, n, nh, nkv, hd):
    """Causal attention in float64, and per output the sum of |p·v| (the scale of its rounding) and per row the largest
    Σ|q·k|/√hd of a visible key (the scale of its scores' rounding)."""
    G, ref, mag, smax = nh // nkv, np.empty((n, nh, hd)), np.empty((n, nh, hd)), np.empty((n, nh, 1))
    K, V = kv[0].astype(np.float64), kv[1].astype(np.float64)
    with np.errstate(invalid="ignore"):
        for h in range(nh):
            sc = q[:, h * hd:(h + 1) * hd].astype(np.float64) @ K[h // G, :n].T / np.sqrt(hd)
            sc[np.triu_indices(n, 1)] = -np.inf
            p = np.exp(sc - sc.max(axis=1, keepdims=True))
            p /= p.sum(axis=1, keepdims=True)
            p[np.triu_indices(n, 1)] = 0.0
            for i in range(n) if not np.isfinite(V[h // G, :n]).all() else ():
                ref[i, h] = p[i, :i + 1] @ V[h // G, :i + 1]
            if np.isfinite(V[h // G, :n]).all():
                ref[:, h] = p @ V[h // G, :n]
            mag[:, h] = p @ np.abs(V[h // G, :n])
            a = np.abs(q[:, h * hd:(h + 1) * hd]).astype(np.float64) @ np.abs(K[h // G, :n]).T / np.sqrt(hd)
            a[np.triu_indices(n, 1)] = 0.0
            smax[:, h, 0] = a.max(axis=1)
    return ref, mag, smax


# enough rows that the fp16-split kernel takes them (the f32 kernel's workgroups past two a CU; 513 the first so): every group size,
# odd and even block counts, a last key tile of 1 .. 32 keys; key tiles scaled 2^-2 .. 2^2 and value tiles 2^-12 ..
# 2^12 against each other, so that the tiles' exponents differ
@pytest.mark.parametrize("n,nh,nkv,max_seq", [(513, 32, 8, 520), (640, 32, 8, 640), (1025, 32, 8, 1100), (700, 64, 8, 704), (1300, 16, 8, 1300),
                                              (650, 32, 32, 1000)])
def test_attn_prefill_split_matches_f64(gpu, n, nh, nkv, max_seq):
    """Error: a score is the f32 sum of 24 matrix-core steps over parts that leave 2^-22 of a product, at most 2^-19 of
    its Σ|q·k|/√hd = A, which its probability takes on; probabilities and values carry 2^-22 of their own, the sums of
    at most n/64 + 10 steps less than 2^-19: 2^-19·(2 + A) of Σ|p·v| bounds it."""
    torch = gpu
    hd = 128
    rng = np.random.default_rng(n + nh)
    stride = (nh + 2 * nkv) * hd
    q = rng.standard_normal((n, stride)).astype(np.float32)
    kv = rng.standard_normal((2, nkv, max_seq, hd)).astype(np.float32)
    for t in range(0, n, 32):
        kv[0, :, t:t + 32] *= np.float32(2.0) ** rng.integers(-2, 3, (nkv, 1, 1))
        kv[1, :, t:t + 32] *= np.float32(2.0) ** rng.integers(-12, 13, (nkv, 1, 1))
    kv[:, :, n:] = np.nan  # slots past the prompt are never read
    q[5] = 0.0
    out = torch.empty(n * nh * hd, dtype=torch.float32, device="cuda")
    qd, kvd = torch.from_numpy(q).cuda(), torch.from_numpy(kv).cuda()

    def run():
        A.check(A.lib().aeth_attn_prefill(qd.data_ptr(), stride, kvd.data_ptr(), n, nh, nkv, hd, max_seq, out.data_ptr(),
                                          None), "attn_prefill")
        torch.cuda.synchronize()
        return out.cpu().numpy().reshape(n, nh, hd).copy()

    ref, mag, smax = attn_prefill64(q, kv, n, nh, nkv, hd)
    got = run()
    assert (np.abs(got - ref) <= 2.0 ** -19 * (2 + smax) * mag).all()
    assert np.array_equal(run(), got)
    # one KV head with an infinite key element and an infinite value: its rows as the f32 formula gives them
    kv[0, 1, n // 2, 3], kv[1, 1, n - 2, 7] = np.inf, -np.inf
    kvd.copy_(torch.from_numpy(kv))
    bad, G = run(), nh // nkv
    mine = np.arange(nh) // G == 1
    assert np.array_equal(bad[:, ~mine], got[:, ~mine])
    s = q.reshape(n, -1, hd)[:, :nh][:, mine][n // 2:, :, 3]  # the sign of that key's scores
    rows = bad[n // 2:, mine]
    assert np.isnan(rows[s > 0]).all()  # exp(inf - inf)
    below = np.abs(bad[:n // 2, mine] - ref[:n // 2, mine]) <= 2.0 ** -19 * (2 + smax[:n // 2, mine]) * mag[:n // 2, mine]
    assert below.all()
    assert np.isfinite(rows[:n - 2 - n // 2][s[:n - 2 - n // 2] < 0]).all()
    assert (rows[-2:, :, 7][s[-2:] < 0] == -np.inf).all()


def test_attn_prefill_two_threads_one_stream(gpu):
    """Two host threads with prompts of their own, and of growing lengths, on the null stream: every call gives the bytes it
    gives alone."""
    torch = gpu
    nh, nkv, sizes = 32, 8, (650, 700, 900, 1200)
    jobs = []
    for t in range(2):
        rng = np.random.default_rng(t)
        q = torch.from_numpy(rng.standard_normal((sizes[-1], nh * 128)).astype(np.float32)).cuda()
        kv = torch.from_numpy(rng.standard_normal((2, nkv, sizes[-1], 128)).astype(np.float32)).cuda()
        jobs.append((q, kv, [torch.empty(n, nh, 128, device="cuda") for n in sizes for _ in range(8)]))

    def call(q, kv, n, out):
        A.check(A.lib().aeth_attn_prefill(q.data_ptr(), nh * 128, kv.data_ptr(), n, nh, nkv, 128, sizes[-1], out.data_ptr(),
                                          None), "attn_prefill")

    torch.cuda.synchronize()
    start, errors = threading.Barrier(2), []

    def work(q, kv, outs):
        try:
            start.wait()
            for out in outs:
                call(q, kv, out.shape[0], out)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for q, kv, outs in jobs:
        for out in outs:
            alone = torch.empty_like(out)
            call(q, kv, out.shape[0], alone)
            torch.cuda.synchronize()
            assert torch.equal(out, alone)


def attn_prefill(torch, qd, stride, kvd, n, nh, nkv, max_seq, stream=None):
    out = torch.full((n, nh, 128), float("nan"), device="cuda")
    A.check(A.lib().aeth_attn_prefill(qd.data_ptr(), stride, kvd.data_ptr(), n, nh, nkv, 128, max_seq, out.data_ptr(),
                                      stream), "attn_prefill")
    return out


# what the two fp16 parts of the split kernel cannot hold beside what shares their power of two: a key or a dimension of the
# keys or values far above the others of its tile, one far below them, a dimension of some queries, and numbers whose
# scales' product overflows
WIDE = {"value": lambda q, k, v: v.__setitem__((0, 100), v[0, 100] * 1e9),
        "value dim": lambda q, k, v: v.__setitem__((1, slice(640, 672), 5), v[1, 640:672, 5] * 1e8),
        "small dim": lambda q, k, v: v.__setitem__((1, slice(0, None), 77), v[1, :, 77] * 1e-9),
        "key": lambda q, k, v: (k.__setitem__((0, 300), k[0, 300] * 1e8), q.__setitem__((slice(0, None), slice(0, 128)), 0.0)),
        "key dim": lambda q, k, v: (k.__setitem__((0, slice(0, None), 3), k[0, :, 3] * 1e9), q[:, 3:512:128].fill(0.0)),
        "query dim": lambda q, k, v: (q[200:300, 9::128].__imul__(1e10), k.__setitem__((slice(0, None), slice(0, None), 9), 0.0)),
        "scales": lambda q, k, v: (q[:, 9::128].__imul__(1e22), k.__setitem__((slice(0, None), 31, 9), 1e22),
                                   k.__setitem__((slice(0, None), slice(0, 31), 9), 0.0))}


@pytest.mark.parametrize("n,nh,nkv", [(700, 32, 8), (650, 64, 8)])
@pytest.mark.parametrize("what", list(WIDE))
def test_attn_prefill_wide_ranges(gpu, what, n, nh, nkv):
    """Numbers that the fp16 parts would not hold take the f32 arithmetic: per output 2^-19·(2 + A)·Σ|p·v| (the bound of
    the split kernel's test, here with nothing that grows with a number elsewhere in its tile)."""
    torch = gpu
    rng = np.random.default_rng(n)
    stride = (nh + 2 * nkv) * 128
    q = rng.standard_normal((n, stride)).astype(np.float32)
    kv = rng.standard_normal((2, nkv, n, 128)).astype(np.float32)
    WIDE[what](q, kv[0], kv[1])
    ref, mag, smax = attn_prefill64(q, kv, n, nh, nkv, 128)
    got = attn_prefill(torch, torch.from_numpy(q).cuda(), stride, torch.from_numpy(kv).cuda(), n, nh, nkv, n).cpu().numpy()
    ok = np.isfinite(smax[..., 0]) & (smax[..., 0] < 1e30)
    assert ok[:31].all()
    assert (np.abs(got - ref)[ok] <= (2.0 ** -19 * (2 + smax) * mag)[ok] + 1e-44).all()


def test_attn_prefill_under_capture(gpu):
    """Under graph capture a long prompt runs the f32 kernel (its scratch could not grow): the same attention as outside it
    to the bound of either, at every replay, with other eager work between the replays."""
    torch = gpu
    n, nh, nkv = 700, 32, 8
    rng = np.random.default_rng(1)
    stride = nh * 128
    q, kv = torch.empty(n, stride, device="cuda"), torch.empty(2, nkv, n, 128, device="cuda")
    out = torch.empty(n, nh, 128, device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        A.check(A.lib().aeth_attn_prefill(q.data_ptr(), stride, kv.data_ptr(), n, nh, nkv, 128, n, out.data_ptr(),
                                          s.cuda_stream), "attn_prefill")
    for _ in range(3):
        qh = rng.standard_normal((n, stride)).astype(np.float32)
        kvh = rng.standard_normal((2, nkv, n, 128)).astype(np.float32)
        q.copy_(torch.from_numpy(qh))
        kv.copy_(torch.from_numpy(kvh))
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        eager = attn_prefill(torch, q, stride, kv, n, nh, nkv, n).cpu().numpy()
        ref, mag, smax = attn_prefill64(qh, kvh, n, nh, nkv, 128)
        for got in (out.cpu().numpy(), eager):
            assert (np.abs(got - ref) <= 2.0 ** -19 * (2 + smax) * mag).all()


# ── device LlamaRunner vs the oracle's decode step ───────────────────────

def make_runner(m, c=TINY):
    cfg = A.LlamaConfig(**c)
    nl = c["num_layers"]
    wp = (ctypes.c_void_p * (nl * 7))(*[m["layers"][l][j].ctypes.data for l in range(nl) for j in range(7)])
    dt = (ctypes.c_int32 * (nl * 7))(*(m["layer_dtype"] * nl))
    npp = (ctypes.c_void_p * (nl * 2))(*[m["norms"][l][j].ctypes.data for l in range(nl) for j in range(2)])
    r = ctypes.c_void_p()
    A.check(A.lib().aeth_runner_create(ctypes.byref(cfg), wp, dt, npp, m["final"].ctypes.data, m["lm"].ctypes.data,
                                       m["lm_dtype"], m["emb"].ctypes.data, 0, ctypes.byref(r)), "runner_create")
    return r


@pytest.mark.parametrize("layer_dtype", [Q4_K, Q8_0, Q6_K, Q5_K])
def test_runner_decode_matches_oracle(gpu, layer_dtype):
    m = build_tiny(seed=2, layer_dtype=layer_dtype)
    r = make_runner(m)
    L = A.lib()
    c = TINY
    ocfg = oracle_cfg()
    s, co = O.precompute_rope(c["max_seq_len"], c["head_dim"], c["rope_base"])
    kv = np.zeros((c["num_layers"], 2, c["num_kv_heads"], c["max_seq_len"], c["head_dim"]), dtype=np.float32)
    fill = 0
    tok = 1
    try:
        for step in range(6):
            logits = np.empty(c["vocab_size"], dtype=np.float32)
            nxt = ctypes.c_int32()
            A.check(L.aeth_runner_decode(r, tok, step, logits.ctypes.data, ctypes.byref(nxt)), "decode")
            ref, fill = O.decode_step(ocfg, m["emb"][tok], step, m["layers"], [layer_dtype] * 7, m["norms"], m["final"],
                                      m["lm"], m["lm_dtype"], s, co, kv, fill)
            assert_close_logits(logits, ref, what="step %d" % step)
            assert nxt.value == O.argmax(logits)
            tok = O.argmax(ref)  # teacher forcing on the CPU's token
        assert L.aeth_runner_seq_len(r) == 6
        kv_dev = np.empty_like(kv)
        fl = ctypes.c_int32()
        A.check(L.aeth_runner_kv_to_host(r, kv_dev.ctypes.data, ctypes.byref(fl)))
        assert fl.value == 6
        assert_close_rows(kv_dev.reshape(-1, c["head_dim"]), kv.reshape(-1, c["head_dim"]), what="kv")
    finally:
        L.aeth_runner_free(r)


# Batched prefill (forward_batch) against the oracle's restatement: one query /
# key block (37), a full cache (64), a single token, and several ragged blocks
# with the GEMM path (150 of 192); GEMM for Q4_K, Q5_K and Q8_0 from 16 tokens (the fused
# RMSNorm prep and SwiGLU output included), the row-batched GEMV and standalone RMSNorm /
# SwiGLU below that (5, 12) and for the other formats.
@pytest.mark.parametrize("layer_dtype,n,max_seq", [(Q4_K, 37, 64), (Q8_0, 64, 64), (Q6_K, 1, 64), (Q4_K, 150, 192),
                                                   (Q5_K, 40, 64), (Q4_K, 5, 64), (Q4_K, 12, 64), (Q8_0, 150, 192),
                                                   (Q5_K, 150, 192)])
def test_runner_prefill_matches_oracle(gpu, layer_dtype, n, max_seq):
    c = dict(TINY, max_seq_len=max_seq)
    m = build_tiny(seed=7, layer_dtype=layer_dtype)
    r = make_runner(m, c)
    L = A.lib()
    ocfg = oracle_cfg(c)
    s, co = O.precompute_rope(c["max_seq_len"], c["head_dim"], c["rope_base"])
    kv = np.zeros((c["num_layers"], 2, c["num_kv_heads"], c["max_seq_len"], c["head_dim"]), dtype=np.float32)
    toks = np.random.default_rng(n).integers(0, c["vocab_size"], n).astype(np.int32)
    try:
        logits = np.empty(c["vocab_size"], dtype=np.float32)
        nxt = ctypes.c_int32()
        A.check(L.aeth_runner_prefill(r, toks.ctypes.data, n, logits.ctypes.data, ctypes.byref(nxt)), "prefill")
        ref = O.forward_batch(ocfg, m["emb"][toks], m["layers"], [layer_dtype] * 7, m["norms"], m["final"], m["lm"],
                              m["lm_dtype"], s, co, kv)
        assert_close_logits(logits, ref, what="prefill n=%d" % n)
        assert nxt.value == O.argmax(logits)
        assert L.aeth_runner_seq_len(r) == n
        kv_dev = np.empty_like(kv)
        fl = ctypes.c_int32()
        A.check(L.aeth_runner_kv_to_host(r, kv_dev.ctypes.data, ctypes.byref(fl)))
        assert fl.value == n
        assert_close_rows(kv_dev[:, :, :, :n].reshape(-1, c["head_dim"]), kv[:, :, :, :n].reshape(-1, c["head_dim"]),
                          what="kv after prefill")
        assert not kv_dev[:, :, :, n:].any()
        if n < max_seq:  # decoding continues from the prefilled cache
            tok = O.argmax(ref)
            A.check(L.aeth_runner_decode(r, tok, n, logits.ctypes.data, None), "decode after prefill")
            ref2, fill = O.decode_step(ocfg, m["emb"][tok], n, m["layers"], [layer_dtype] * 7, m["norms"], m["final"],
                                       m["lm"], m["lm_dtype"], s, co, kv, n)
            assert fill == n + 1 and L.aeth_runner_seq_len(r) == n + 1
            assert_close_logits(logits, ref2, what="decode after prefill")
    finally:
        L.aeth_runner_free(r)


# GQA group sizes G = query heads per KV head: the MFMA attention packs 16/G
# queries × G heads into its 16 score columns (G = 2 is TINY above); n = 70 is
# ragged against every query block, the 16-key blocks and the block pairs.
@pytest.mark.parametrize("heads,kv_heads", [(4, 4), (8, 2), (8, 1)])
def test_runner_prefill_gqa_groups(gpu, heads, kv_heads):
    c = dict(TINY, num_heads=heads, num_kv_heads=kv_heads, max_seq_len=96)
    n = 70
    m = build_tiny(seed=heads * 10 + kv_heads, c=c)
    r = make_runner(m, c)
    L = A.lib()
    s, co = O.precompute_rope(c["max_seq_len"], c["head_dim"], c["rope_base"])
    kv = np.zeros((c["num_layers"], 2, c["num_kv_heads"], c["max_seq_len"], c["head_dim"]), dtype=np.float32)
    toks = np.random.default_rng(heads).integers(0, c["vocab_size"], n).astype(np.int32)
    try:
        logits = np.empty(c["vocab_size"], dtype=np.float32)
        A.check(L.aeth_runner_prefill(r, toks.ctypes.data, n, logits.ctypes.data, None), "prefill")
        ref = O.forward_batch(oracle_cfg(c), m["emb"][toks], m["layers"], [Q4_K] * 7, m["norms"], m["final"], m["lm"],
                              m["lm_dtype"], s, co, kv)
        assert_close_logits(logits, ref, what="prefill heads=%d kv_heads=%d" % (heads, kv_heads))
    finally:
        L.aeth_runner_free(r)


# Files that mix formats inside a layer (llama.cpp's Q4_K_M keeps attn_v and
# ffn_down in Q6_K): q/k/v and gate/up of different formats are run as separate
# weights (three GEMVs into q|k|v, gate and up GEMVs then SiLU·up; strided GEMM
# columns in prefill). n = 150 takes the Q4_K GEMM with the output row stride.
MIXED = [[Q4_K, Q4_K, Q6_K, Q4_K, Q4_K, Q4_K, Q6_K],     # Q4_K_M
         [Q8_0, Q4_K, Q6_K, Q6_K, Q4_K, Q8_0, Q4_K]]     # every split, GEMV and GEMM columns


@pytest.mark.parametrize("mix", [0, 1])
@pytest.mark.parametrize("n", [1, 23, 150])
def test_runner_mixed_formats(gpu, mix, n):
    c = dict(TINY, max_seq_len=192)
    m = build_tiny(seed=11 + mix, layer_dtype=MIXED[mix], c=c)
    r = make_runner(m, c)
    L = A.lib()
    ocfg = oracle_cfg(c)
    s, co = O.precompute_rope(c["max_seq_len"], c["head_dim"], c["rope_base"])
    kv = np.zeros((c["num_layers"], 2, c["num_kv_heads"], c["max_seq_len"], c["head_dim"]), dtype=np.float32)
    toks = np.random.default_rng(n).integers(0, c["vocab_size"], n).astype(np.int32)
    try:
        logits = np.empty(c["vocab_size"], dtype=np.float32)
        A.check(L.aeth_runner_prefill(r, toks.ctypes.data, n, logits.ctypes.data, None), "prefill")
        ref = O.forward_batch(ocfg, m["emb"][toks], m["layers"], MIXED[mix], m["norms"], m["final"], m["lm"],
                              m["lm_dtype"], s, co, kv)
        # anchored on the float64 evaluation: at n = 150 the reference's own f32 logits
        # drift from it by 1.8e-5·max|row| (9.5e-4 on logits below 1)
        seq = list(toks)
        ex = lambda: logits64(c, m["emb"], m["layers"], MIXED[mix], m["norms"], m["final"], m["lm"], m["lm_dtype"], seq)
        assert_close_logits(logits, ref, what="mixed prefill n=%d" % n, exact=ex())
        fill = n
        tok = O.argmax(ref)
        for step in range(2):
            A.check(L.aeth_runner_decode(r, tok, fill, logits.ctypes.data, None), "mixed decode")
            ref, fill = O.decode_step(ocfg, m["emb"][tok], fill, m["layers"], MIXED[mix], m["norms"], m["final"],
                                      m["lm"], m["lm_dtype"], s, co, kv, fill)
            seq.append(tok)
            assert_close_logits(logits, ref, what="mixed decode step %d" % step, exact=ex())
            tok = O.argmax(ref)
        # separately stored weights export as they were given
        for j in range(7):
            blob = np.empty(m["layers"][1][j].nbytes, dtype=np.uint8)
            A.check(L.aeth_runner_export(r, j, 1, blob.ctypes.data, blob.nbytes), "export %d" % j)
            assert np.array_equal(blob, m["layers"][1][j].view(np.uint8).ravel()), "export %d" % j
    finally:
        L.aeth_runner_free(r)


# Layers and LM heads in the formats the reference keeps in GGUF order (F32 /
# F16 / Q2_K / Q3_K: dequantize + matmul_f32_gguf, dispatch.rs:126-133), mixed
# with fused ones: decode steps (eager and replayed as a HIP graph, whose
# GGUF-order GEMVs use the runner's own scratch) and prefill against the oracle.
GGUF_MIX = [[F16, Q2_K, Q3_K, F32, Q5_K, Q2_K, Q3_K], [Q3_K, Q3_K, Q3_K, Q2_K, Q2_K, Q2_K, F16]]


@pytest.mark.parametrize("mix,lm_dtype", [(0, F16), (1, Q6_K)])
def test_runner_gguf_order_formats(gpu, mix, lm_dtype):
    c = dict(TINY, max_seq_len=64)
    m = build_tiny(seed=21 + mix, layer_dtype=GGUF_MIX[mix], lm_dtype=lm_dtype, c=c)
    L = A.lib()
    ocfg = oracle_cfg(c)
    s, co = O.precompute_rope(c["max_seq_len"], c["head_dim"], c["rope_base"])
    n = 19
    toks = np.random.default_rng(mix).integers(0, c["vocab_size"], n).astype(np.int32)
    r = make_runner(m, c)
    try:
        kv = np.zeros((c["num_layers"], 2, c["num_kv_heads"], c["max_seq_len"], c["head_dim"]), dtype=np.float32)
        logits = np.empty(c["vocab_size"], dtype=np.float32)
        A.check(L.aeth_runner_prefill(r, toks.ctypes.data, n, logits.ctypes.data, None), "prefill")
        ref = O.forward_batch(ocfg, m["emb"][toks], m["layers"], GGUF_MIX[mix], m["norms"], m["final"], m["lm"],
                              lm_dtype, s, co, kv)
        seq = list(toks)
        ex = lambda: logits64(c, m["emb"], m["layers"], GGUF_MIX[mix], m["norms"], m["final"], m["lm"], lm_dtype, seq)
        assert_close_logits(logits, ref, what="gguf-order prefill", exact=ex())
        tok, fill = O.argmax(ref), n
        for step in range(2):
            nxt = ctypes.c_int32()
            A.check(L.aeth_runner_decode(r, tok, fill, logits.ctypes.data, ctypes.byref(nxt)), "decode")
            ref, fill = O.decode_step(ocfg, m["emb"][tok], fill, m["layers"], GGUF_MIX[mix], m["norms"], m["final"],
                                      m["lm"], lm_dtype, s, co, kv, fill)
            seq.append(tok)
            assert_close_logits(logits, ref, what="gguf-order decode %d" % step, exact=ex())
            assert nxt.value == O.argmax(logits)
            tok = O.argmax(ref)
    finally:
        L.aeth_runner_free(r)
    outs = []
    for use_graph in (0, 1):
        r = make_runner(m, c)
        t = (ctypes.c_int32 * 8)()
        A.check(L.aeth_runner_generate(r, 1, 0, 8, t, use_graph), "generate")
        outs.append(list(t))
        L.aeth_runner_free(r)
    assert outs[0] == outs[1]


def test_prefill_prep_is_not_another_weights(gpu):
    """q, k and v of three formats at 64 tokens: q's and v's GEMMs take the RMSNorm in their activation prep, formed once
    for both, k's (F16) forms its own between them in the same scratch. The values rows do not depend on k's format."""
    c = dict(TINY, vocab_size=64, d_model=4096, num_layers=1, num_heads=32, num_kv_heads=8, d_ff=256, max_seq_len=64)
    L, n, v = A.lib(), 64, []
    toks = (np.arange(n) % c["vocab_size"]).astype(np.int32)
    for kd in (Q4_K, F16):
        r = make_runner(build_tiny(seed=31, layer_dtype=[Q4_K, kd, Q6_K, Q4_K, Q4_K, Q4_K, Q4_K], c=c), c)
        try:
            A.check(L.aeth_runner_prefill(r, toks.ctypes.data, n, None, None), "prefill")
            kv, fl = np.empty((2, c["num_kv_heads"], n, c["head_dim"]), np.float32), ctypes.c_int32()
            A.check(L.aeth_runner_kv_to_host(r, kv.ctypes.data, ctypes.byref(fl)), "kv_to_host")
        finally:
            L.aeth_runner_free(r)
        v.append(kv[1])
    assert np.isfinite(v[0]).all() and np.array_equal(v[0], v[1])


# The step's results reach pageable memory through the runner's pinned buffer and pinned memory directly;
# either output may be NULL. The same prompt and step give the same bytes each way.
@pytest.mark.parametrize("vocab", [3, 512, 1283])
def test_runner_results_by_destination(gpu, vocab):
    c = dict(TINY, vocab_size=vocab)
    m = build_tiny(seed=23, c=c)
    r = make_runner(m, c)
    L = A.lib()
    toks = (np.arange(9) % vocab).astype(np.int32)
    pinned = gpu.empty(vocab, pin_memory=True)
    pageable = np.empty(vocab + 1, dtype=np.float32)
    nxt = ctypes.c_int32()
    try:
        def turn(dst, token):
            got = []
            for call in (lambda p, t: L.aeth_runner_prefill(r, toks.ctypes.data, len(toks), p, t),
                         lambda p, t: L.aeth_runner_decode(r, vocab - 1, len(toks), p, t)):
                pinned.fill_(-7.0)
                pageable.fill(-7.0)
                nxt.value = -1
                A.check(call(None if dst is None else dst.ctypes.data if dst is pageable else dst.data_ptr(),
                             ctypes.byref(nxt) if token else None), "step")
                assert pageable[vocab] == -7.0
                got.append((np.asarray(dst[:vocab]).copy() if dst is not None else None, nxt.value if token else None))
            return got

        want = turn(pinned, True)
        for dst, token in ((pageable, True), (pageable, False), (pinned, False), (None, True), (None, False)):
            for (a, t), (b, u) in zip(want, turn(dst, token)):
                assert b is None or np.array_equal(a, b)
                assert u is None or u == t == O.argmax(a)
    finally:
        L.aeth_runner_free(r)


def test_runner_prefill_bad_arguments(gpu):
    m = build_tiny(seed=8)
    r = make_runner(m)
    L = A.lib()
    try:
        toks = np.zeros(TINY["max_seq_len"] + 1, dtype=np.int32)
        assert L.aeth_runner_prefill(r, toks.ctypes.data, 0, None, None) == -1
        assert L.aeth_runner_prefill(r, toks.ctypes.data, TINY["max_seq_len"] + 1, None, None) == -1
        toks[3] = TINY["vocab_size"]
        assert L.aeth_runner_prefill(r, toks.ctypes.data, 5, None, None) == -1
    finally:
        L.aeth_runner_free(r)


def test_runner_generate_graph_matches_eager(gpu):
    m = build_tiny(seed=3)
    L = A.lib()
    outs = []
    for use_graph in (0, 1, 1):
        r = make_runner(m)
        toks = (ctypes.c_int32 * 10)()
        A.check(L.aeth_runner_generate(r, 1, 0, 10, toks, use_graph), "generate")
        if use_graph:  # a second replay batch continues the sequence
            more = (ctypes.c_int32 * 5)()
            A.check(L.aeth_runner_generate(r, toks[9], 10, 5, more, use_graph), "generate 2")
            outs.append(list(toks) + list(more))
        else:
            more = (ctypes.c_int32 * 5)()
            A.check(L.aeth_runner_generate(r, toks[9], 10, 5, more, 0), "generate 2")
            outs.append(list(toks) + list(more))
        L.aeth_runner_free(r)
    assert outs[0] == outs[1] == outs[2]


def test_c_api_surface(gpu):
    """aether_* over a device runner: queries, decode, argmax, budget."""
    L = A.lib()
    m = build_tiny(seed=4)
    r = make_runner(m)
    model = L.aether_model_from_runner(r)
    assert model
    try:
        assert L.aether_vocab_size(model) == TINY["vocab_size"]
        assert L.aether_num_layers(model) == TINY["num_layers"]
        assert L.aether_d_model(model) == TINY["d_model"]
        assert L.aether_context_len(model) == TINY["max_seq_len"]
        logits = np.empty(TINY["vocab_size"], dtype=np.float32)
        toks = (ctypes.c_int * 3)(1, 5, 9)
        assert L.aether_prefill(model, toks, 3, logits.ctypes.data) == 0
        assert L.aeth_runner_seq_len(r) == 3
        t = L.aether_argmax(model, logits.ctypes.data)
        assert t == O.argmax(logits)
        assert L.aether_sample(model, logits.ctypes.data, 0.0, 1.0) == t
        assert L.aether_decode(model, t, 3, logits.ctypes.data) == 0
        # a generous budget completes like aether_decode
        L.aether_set_frame_budget(model, 10000.0)
        assert abs(L.aether_frame_budget(model) - 10000.0) < 1e-3
        assert L.aether_decode_budgeted(model, 2, 4, logits.ctypes.data) == 0
        assert L.aeth_runner_seq_len(r) == 5
        assert L.aether_load(b"/nonexistent.gguf") is None
    finally:
        L.aether_free(model)


def test_decode_budgeted_timeout_and_resume(gpu):
    """aether_decode_budgeted (c_api.rs:324-355 → decode_step_budgeted,
    runner.rs:1201-1282) forced from the host: a budget of 1e-9 ms has expired
    at the first layer check, so the call returns AETHER_TIMEOUT (-2) without
    logits and records completed_layer = 0 (the reference's
    layer_idx.saturating_sub(1) at layer 0); a retry with the same (token, pos)
    resumes at layer 1 with the saved residual stream — i.e. layer 0 is skipped,
    exactly as the reference does — and, given time, completes. The oracle enters
    its decode step at layer 1 with x = the embedding (orc_decode_step_from). A
    retry with another (token, pos) drops the partial state and runs every layer."""
    L = A.lib()
    m = build_tiny(seed=6)
    r = make_runner(m)
    model = L.aether_model_from_runner(r)
    c = TINY
    ocfg = oracle_cfg()
    s, co = O.precompute_rope(c["max_seq_len"], c["head_dim"], c["rope_base"])
    kv = np.zeros((c["num_layers"], 2, c["num_kv_heads"], c["max_seq_len"], c["head_dim"]), dtype=np.float32)
    try:
        toks = np.array([3, 17, 29], np.int32)
        logits = np.full(c["vocab_size"], np.nan, np.float32)
        assert L.aether_prefill(model, toks.ctypes.data, 3, logits.ctypes.data) == 0
        O.forward_batch(ocfg, m["emb"][toks], m["layers"], [Q4_K] * 7, m["norms"], m["final"], m["lm"],
                        m["lm_dtype"], s, co, kv)
        tok = 41
        L.aether_set_frame_budget(model, 1e-9)
        sentinel = np.full(c["vocab_size"], 7.0, np.float32)
        for _ in range(2):  # expires before layer 0, then again right at the resume layer
            assert L.aether_decode_budgeted(model, tok, 3, sentinel.ctypes.data) == -2
            assert (sentinel == 7.0).all()  # no logits written on a timeout
            assert L.aeth_runner_seq_len(r) == 3
        L.aether_set_frame_budget(model, 1e6)
        assert L.aether_decode_budgeted(model, tok, 3, logits.ctypes.data) == 0
        assert L.aeth_runner_seq_len(r) == 4
        ref, fill = O.decode_step(ocfg, m["emb"][tok], 3, m["layers"], [Q4_K] * 7, m["norms"], m["final"], m["lm"],
                                  m["lm_dtype"], s, co, kv, 3, start_layer=1)
        assert fill == 4
        assert_close_logits(logits, ref, what="resumed at layer 1")
        # a timed-out attempt for (tok2, 4), then a different token at pos 4: fresh step
        L.aether_set_frame_budget(model, 1e-9)
        assert L.aether_decode_budgeted(model, 55, 4, sentinel.ctypes.data) == -2
        L.aether_set_frame_budget(model, 1e6)
        assert L.aether_decode_budgeted(model, 56, 4, logits.ctypes.data) == 0
        ref, fill = O.decode_step(ocfg, m["emb"][56], 4, m["layers"], [Q4_K] * 7, m["norms"], m["final"], m["lm"],
                                  m["lm_dtype"], s, co, kv, 4)
        assert_close_logits(logits, ref, what="fresh step after a dropped partial")
        kv_dev = np.empty_like(kv)
        fl = ctypes.c_int32()
        A.check(L.aeth_runner_kv_to_host(r, kv_dev.ctypes.data, ctypes.byref(fl)))
        assert fl.value == 5
        assert_close_rows(kv_dev[:, :, :, :5].reshape(-1, c["head_dim"]), kv[:, :, :, :5].reshape(-1, c["head_dim"]),
                          what="kv after budgeted steps")
        # budget <= 0: the plain decode
        L.aether_set_frame_budget(model, 0.0)
        assert L.aether_decode_budgeted(model, 57, 5, logits.ctypes.data) == 0
        ref, fill = O.decode_step(ocfg, m["emb"][57], 5, m["layers"], [Q4_K] * 7, m["norms"], m["final"], m["lm"],
                                  m["lm_dtype"], s, co, kv, 5)
        assert_close_logits(logits, ref, what="unbudgeted")
    finally:
        L.aether_free(model)


def test_runners_prefill_concurrently(gpu):
    """Two runners prefilling from two host threads at once (each on its own
    stream, with the GEMM's scratch per stream) give exactly their serial
    results; the Q4_K GEMM runs for n = 150."""
    import threading

    L = A.lib()
    c = dict(TINY, max_seq_len=192)
    models = [build_tiny(seed=40 + i, c=c) for i in range(2)]
    toks = [np.random.default_rng(60 + i).integers(0, c["vocab_size"], 150).astype(np.int32) for i in range(2)]

    def prefill(r, t, out):
        A.check(L.aeth_runner_prefill(r, t.ctypes.data, t.size, out.ctypes.data, None), "prefill")

    serial = []
    for i in range(2):
        r = make_runner(models[i], c)
        out = np.empty(c["vocab_size"], np.float32)
        prefill(r, toks[i], out)
        serial.append(out)
        L.aeth_runner_free(r)
    runners = [make_runner(models[i], c) for i in range(2)]
    try:
        for rep in range(3):
            outs = [np.empty(c["vocab_size"], np.float32) for _ in range(2)]
            th = [threading.Thread(target=prefill, args=(runners[i], toks[i], outs[i])) for i in range(2)]
            for t in th:
                t.start()
            for t in th:
                t.join()
            for i in range(2):
                assert np.array_equal(outs[i], serial[i]), "runner %d rep %d" % (i, rep)
    finally:
        for r in runners:
            L.aeth_runner_free(r)
