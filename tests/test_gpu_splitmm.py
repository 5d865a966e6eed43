"""The matrix-core products of fp32 / int8 rows with block-quantized weights
(csrc/splitmm.hpp) behind gemm_q, gemm_q_i8, gemm_w4a16, gemm_fp8,
moe_expert_ffn_q and moe_expert_ffn_q_i8, at the edges of their tiles, chunks
and launch rules, against 64-bit products of the oracle's dequantized weights.

Tolerance. Every output is a sum of K / 32 pieces (each a product of 32 terms
added in fp32 by the matrix core), added in two levels of at most 16 and 24
terms: in the 2-norm about sqrt(16 / 2 + 24 / 2 + 4) * 2^-24 / sqrt(3) = 1.7e-7
of the result at most; 2.5e-7 is the bound (fp32 vector sums: the same order).
Values with an offset per block (Q4_K, Q5_K: ds * q - dm) subtract two sums
several times the result: four times that.
"""
import numpy as np
import pytest
import torch

from glmserve_amd import ops
from moe_cases import GGUF_TYPES, random_gguf_rows

pytestmark = pytest.mark.gpu
TYPES = [8, 11, 12, 13, 14, 18, 23]
TOL = {t: 1e-6 if t in (12, 13) else 2.5e-7 for t in TYPES}


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _rows(t, rows, k, rng):
    """GGUF rows with row_bytes rounded up to a multiple of 4, and as packed. The matrix
    cores take whole dwords: an odd number of 98-, 110- or 210-byte blocks only in rows
    padded like this; packed, they stay on the vector kernels (test_gpu_gguf.py)."""
    w = random_gguf_rows(t, rows, k, rng)
    pad = -w.shape[1] % 4
    return np.concatenate([w, np.zeros((rows, pad), np.uint8)], 1), w


def _err(got, ref):
    assert np.isfinite(got).all()
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


def _quant(x):
    xq = torch.empty(x.shape, dtype=torch.int8, device="cuda")
    xs = torch.empty(x.shape[0], x.shape[1] // 32, device="cuda")
    ops.ref_quantize_act_q8(_dev(x), xq, xs)
    q, s = xq.cpu().numpy(), xs.cpu().numpy()
    return xq, xs, (q.reshape(len(x), -1, 32) * s.astype(np.float64)[:, :, None]).reshape(x.shape)


# Tokens: the tiles of 4, 16 and 32 and their remainders; K: one chunk, an odd
# number of chunks (the last one in the middle of a dword for the 2-byte aligned
# types) and more chunks than the 8 K shares; outputs: one block, a remainder.
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("n,in_,out", [(1, 256, 32), (4, 1280, 96), (5, 768, 64), (16, 2304, 32),
                                       (17, 1280, 160), (33, 256, 64)])
def test_gemm(oracle, qtype, n, in_, out):
    rng = np.random.default_rng(qtype * 100 + n)
    wp, w = _rows(qtype, out, in_, rng)
    W = oracle.gguf_dequant_rows(qtype, w, out, in_).astype(np.float64)
    x = rng.standard_normal((n, in_)).astype(np.float32)
    b = rng.standard_normal(out).astype(np.float32)
    y = torch.full((n, out), float("nan"), device="cuda")
    ops.ref_gemm_q(qtype, _dev(x), _dev(wp), _dev(b), y, wp.shape[1])
    assert _err(y.cpu().numpy(), x.astype(np.float64) @ W.T + b) < TOL[qtype]
    xq, xs, xd = _quant(x)
    ops.ref_gemm_q_i8(qtype, xq, xs, _dev(wp), None, y, wp.shape[1])
    assert _err(y.cpu().numpy(), xd @ W.T) < TOL[qtype]


# 64-token x 256-row tiles: 7 x 28 workgroups, the last tile one token.
@pytest.mark.parametrize("qtype", [8, 12, 18, 23])
def test_gemm_large_tiles(oracle, qtype):
    rng = np.random.default_rng(qtype)
    n, in_, out = 385, 256, 7168 - 32
    w = random_gguf_rows(qtype, out, in_, rng)
    W = oracle.gguf_dequant_rows(qtype, w, out, in_).astype(np.float64)
    x = rng.standard_normal((n, in_)).astype(np.float32)
    y = torch.full((n, out), float("nan"), device="cuda")
    wp = np.concatenate([w, np.zeros((out, -w.shape[1] % 4), np.uint8)], 1)
    ops.ref_gemm_q(qtype, _dev(x), _dev(wp), None, y, wp.shape[1])
    assert _err(y.cpu().numpy(), x.astype(np.float64) @ W.T) < TOL[qtype]
    xq, xs, xd = _quant(x)
    ops.ref_gemm_q_i8(qtype, xq, xs, _dev(wp), None, y, wp.shape[1])
    assert _err(y.cpu().numpy(), xd @ W.T) < TOL[qtype]


@pytest.mark.parametrize("n,in_,out,g", [(1, 256, 32, 32), (7, 768, 96, 96), (19, 512, 64, 512)])
def test_gemm_w4_fp8(oracle, n, in_, out, g):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, in_)).astype(np.float32)
    y = torch.full((n, out), float("nan"), device="cuda")
    q = rng.integers(0, 256, (out, in_ // 2), dtype=np.uint8)
    s = rng.uniform(0.001, 0.02, (out, in_ // g)).astype(np.float32)
    W = oracle.dequant_int4_rows(q, s, in_, g).astype(np.float64)
    ops.ref_gemm_w4a16(_dev(x), _dev(q), _dev(s), None, y, g)
    assert _err(y.cpu().numpy(), x.astype(np.float64) @ W.T) < 2.5e-7
    c = rng.integers(0, 256, (out, in_), dtype=np.uint8)
    c[(c & 0x7F) == 0x7F] = 0x3C
    sc = rng.uniform(0.5, 1.5, out).astype(np.float32)
    W = np.array([oracle.e4m3_to_f32(v) for v in range(256)], np.float64)[c] * sc[:, None].astype(np.float64)
    ops.ref_gemm_fp8(_dev(x), _dev(c), _dev(sc), None, y)
    assert _err(y.cpu().numpy(), x.astype(np.float64) @ W.T) < 2.5e-7


# E = 8, top-4: ungrouped (tiles of 4 with one row), then 12, 36, 280, 400, 2080 and 3840
# routed rows grouped (tiles of 8, 16, 16, 32, 32 or 64 and 64; int8 16 up to 2047 rows,
# then 32), ids outside [0, E) among them.
@pytest.mark.parametrize("types", [(18, 18, 23), (8, 8, 8), (12, 12, 13), (11, 11, 14), (23, 23, 18)])
@pytest.mark.parametrize("n,grouped", [(3, False), (3, True), (9, True), (70, True), (100, True),
                                       (520, True), (960, True)])
def test_moe(oracle, types, n, grouped):
    H, I, E, k = 1024, 512, 8, 4
    rng = np.random.default_rng(sum(types) + n)
    geo = [(types[0], I, H), (types[1], I, H), (types[2], H, I)]
    pk = [_rows(t, E * r, c, rng) for t, r, c in geo]
    W = [oracle.gguf_dequant_rows(t, p[1], E * r, c).reshape(E, r, c).astype(np.float64)
         for (t, r, c), p in zip(geo, pk)]
    dev = [_dev(p[0]) for p in pk]
    rb = tuple(p[0].shape[1] for p in pk)
    # block scales are about 1e-2: keep gate and up of order one
    x = (rng.standard_normal((n, H)) * 2e-2).astype(np.float32)
    ids = np.stack([rng.permutation(E)[:k] for _ in range(n)]).astype(np.int32)
    ids[rng.random((n, k)) < 0.1] = E
    ids[0] = [0, 1, 2, -1]
    w = rng.uniform(0.1, 1.0, (n, k)).astype(np.float32)
    flat, tok = ids.reshape(-1), np.arange(n * k) // k

    def ref_h(xd):
        h = np.zeros((n * k, I))
        for e in range(E):
            r = np.nonzero(flat == e)[0]
            g, u = xd[tok[r]] @ W[0][e].T, xd[tok[r]] @ W[1][e].T
            h[r] = g / (1 + np.exp(-g)) * u
        return h

    def ref_out(h):
        o = np.zeros((n, H))
        for e in range(E):
            r = np.nonzero(flat == e)[0]
            np.add.at(o, tok[r], w.reshape(-1)[r][:, None] * (h[r] @ W[2][e].T))
        return o

    live = (flat >= 0) & (flat < E)
    f = lambda *s: torch.zeros(*s, device="cuda")
    h_act, dpart, out = f(n * k, I), f(n * k, H), f(n, H)
    disp = torch.full((3 * E + 1 + n * k,), -7, dtype=torch.int32, device="cuda") if grouped else None
    tol = 4 * max(TOL[t] for t in types)   # products of products
    ops.ref_moe_expert_ffn_q(types, _dev(x), _dev(ids), _dev(w), *dev, I, E, rb, h_act, dpart, out, disp)
    h = ref_h(x.astype(np.float64))
    assert _err(h_act.cpu().numpy()[live], h[live]) < tol
    assert _err(out.cpu().numpy(), ref_out(h)) < tol
    # int8: gate/up from the quantized x, down from the quantized h it returns
    xq, xs, xd = _quant(x)
    hq, hs = torch.zeros(n * k, I, dtype=torch.int8, device="cuda"), f(n * k, I // 32)
    ops.ref_moe_expert_ffn_q_i8(types, xq, xs, _dev(ids), _dev(w), *dev, I, E, rb, h_act, hq, hs, dpart,
                                out, disp)
    assert _err(h_act.cpu().numpy()[live], ref_h(xd)[live]) < tol
    hd = hq.cpu().numpy().reshape(n * k, -1, 32) * hs.cpu().numpy().astype(np.float64)[:, :, None]
    assert _err(out.cpu().numpy(), ref_out(hd.reshape(n * k, I))) < tol


def _extreme_rows(in_, W, rng):
    """Rows of ordinary, very large and very small magnitudes, then one with an
    infinity and one with a NaN. The largest has outputs near the top of fp32 (its
    sums of codes alone overflow), the smallest subnormal low-order terms."""
    x = rng.standard_normal((8, in_)).astype(np.float32)
    x[1] *= np.float32(1e30 if np.abs(W).max() < 1e3 else 1e25)
    x[2] *= np.float32(1e-25)
    x[3, ::2] *= np.float32(1e-6)   # small terms beside large ones
    x[4] *= np.float32(1e37 / np.abs(x[4].astype(np.float64) @ W.T).max())
    x[5] *= np.float32(1e-36)
    x[6, 77] = -np.inf
    x[7, 200] = np.nan
    return x


def _check_extreme(got, x, W, tol):
    # Every row's relative accuracy; an infinity or NaN stays in its row and gives
    # what the product with the dequantized weights gives (NaN for a zero weight).
    ref = x.astype(np.float64) @ W.T
    for t in range(6):
        assert _err(got[t], ref[t]) < tol, t   # a norm over few outputs only: twice the bound
    with np.errstate(invalid="ignore"):
        inf = np.float32(-np.inf) * W[:, 77].astype(np.float32)
    assert np.array_equal(got[6], inf, equal_nan=True)
    assert np.isnan(got[7]).all()


# The tiles of 4 (a row at a time), 16 and 32 tokens.
@pytest.mark.parametrize("fmt", TYPES + ["w4", "fp8"])
def test_extreme_activations(oracle, fmt):
    in_, out = 512, 64
    rng = np.random.default_rng(TYPES.index(fmt) if fmt in TYPES else len(fmt))
    if fmt == "w4":
        q = rng.integers(0, 256, (out, in_ // 2), dtype=np.uint8)
        s = rng.uniform(0.001, 0.02, (out, in_ // 128)).astype(np.float32)
        W = oracle.dequant_int4_rows(q, s, in_, 128).astype(np.float64)
        run = lambda x, y: ops.ref_gemm_w4a16(x, _dev(q), _dev(s), None, y, 128)
    elif fmt == "fp8":
        c = rng.integers(0, 256, (out, in_), dtype=np.uint8)
        c[(c & 0x7F) == 0x7F] = 0x3C
        sc = rng.uniform(0.5e-3, 1.5e-3, out).astype(np.float32)
        W = np.array([oracle.e4m3_to_f32(v) for v in range(256)], np.float64)[c] * sc[:, None].astype(np.float64)
        run = lambda x, y: ops.ref_gemm_fp8(x, _dev(c), _dev(sc), None, y)
    else:
        w = random_gguf_rows(fmt, out, in_, rng)
        W = oracle.gguf_dequant_rows(fmt, w, out, in_).astype(np.float64)
        run = lambda x, y: ops.ref_gemm_q(fmt, x, _dev(w), None, y, w.shape[1])
    x = _extreme_rows(in_, W, rng)
    tol = 2 * TOL.get(fmt, 2.5e-7)
    for reps in (1, 3):
        y = torch.zeros(8 * reps, out, device="cuda")
        run(_dev(np.tile(x, (reps, 1))), y)
        for r in range(reps):
            _check_extreme(y.cpu().numpy()[8 * r:8 * r + 8], x, W, tol)
    y = torch.zeros(8, out, device="cuda")
    for t in range(8):
        run(_dev(x[t:t + 1]), y[t:t + 1])
    _check_extreme(y.cpu().numpy(), x, W, tol)


@pytest.mark.parametrize("qtype", [8, 12, 18])
def test_extreme_activations_large_tiles(oracle, qtype):
    rng = np.random.default_rng(qtype)
    n, in_, out = 385, 256, 7168 - 32
    w = random_gguf_rows(qtype, out, in_, rng)
    W = oracle.gguf_dequant_rows(qtype, w, out, in_).astype(np.float64)
    x = rng.standard_normal((n, in_)).astype(np.float32)
    ext = _extreme_rows(in_, W, rng)
    x[60:68] = ext
    x[384] = ext[4]
    y = torch.zeros(n, out, device="cuda")
    wp = np.concatenate([w, np.zeros((out, -w.shape[1] % 4), np.uint8)], 1)
    ops.ref_gemm_q(qtype, _dev(x), _dev(wp), None, y, wp.shape[1])
    got = y.cpu().numpy()
    _check_extreme(got[60:68], ext, W, 2 * TOL[qtype])
    ok = np.r_[0:60, 68:385]
    assert _err(got[ok], x[ok].astype(np.float64) @ W.T) < TOL[qtype]


# Tiles of 4 (ungrouped), 16 and 32 rows: gate and up of a token with an infinity,
# and of one whose sums of codes overflow.
@pytest.mark.parametrize("types", [(18, 18, 23), (12, 12, 14), (14, 14, 8)])
@pytest.mark.parametrize("n,grouped", [(3, False), (9, True), (100, True)])
def test_moe_extreme_activations(oracle, types, n, grouped):
    H, I, E, k = 1024, 512, 8, 4
    rng = np.random.default_rng(sum(types) + n)
    geo = [(types[0], I, H), (types[1], I, H), (types[2], H, I)]
    pk = [_rows(t, E * r, c, rng) for t, r, c in geo]
    W = [oracle.gguf_dequant_rows(t, p[1], E * r, c).reshape(E, r, c).astype(np.float64)
         for (t, r, c), p in zip(geo, pk)]
    x = (rng.standard_normal((n, H)) * 2e-2).astype(np.float32)
    x[1, 5] = np.inf
    ids = np.stack([rng.permutation(E)[:k] for _ in range(n)]).astype(np.int32)
    x[2] *= np.float32(1e18 / np.abs(np.einsum("k,erk->er", x[2].astype(np.float64), W[1])).max())
    w = rng.uniform(0.1, 1.0, (n, k)).astype(np.float32)
    f = lambda *s: torch.zeros(*s, device="cuda")
    h_act, dpart, out = f(n * k, I), f(n * k, H), f(n, H)
    disp = torch.zeros(3 * E + 1 + n * k, dtype=torch.int32, device="cuda") if grouped else None
    ops.ref_moe_expert_ffn_q(types, _dev(x), _dev(ids), _dev(w), *[_dev(p[0]) for p in pk], I, E,
                             tuple(p[0].shape[1] for p in pk), h_act, dpart, out, disp)
    h, d = h_act.cpu().numpy(), dpart.cpu().numpy()
    tol = 4 * max(TOL[t] for t in types)
    for r in range(n * k):
        t, e = r // k, ids[r // k, r % k]
        with np.errstate(invalid="ignore", over="ignore"):
            g, u = ((np.inf * W[m][e][:, 5] if t == 1 else W[m][e] @ x[t].astype(np.float64)) for m in (0, 1))
            ref = (g / (1 + np.exp(-g)) * u).astype(np.float32)
        if t == 1:
            assert np.array_equal(h[r], ref, equal_nan=True)
            continue
        assert _err(h[r].astype(np.float64), ref) < tol and np.isfinite(d[r]).all()
        assert _err(d[r].astype(np.float64), W[2][e] @ h[r].astype(np.float64)) < tol


# Q4_K / Q5_K weights centred on zero (as a checkpoint's are) with activations off zero: the
# offsets' sum must not take the product's accuracy with it.
@pytest.mark.parametrize("qtype", [12, 13])
@pytest.mark.parametrize("n", [3, 9, 40])
def test_offset_activations(oracle, qtype, n):
    rng = np.random.default_rng(qtype + n)
    in_, out = 6144, 512
    w = random_gguf_rows(qtype, out, in_, rng)
    b = w.reshape(out, in_ // 256, -1)
    d = np.ascontiguousarray(b[:, :, 0:2]).view(np.float16).astype(np.float32)
    b[:, :, 2:4] = (d * (7.5 if qtype == 12 else 15.5)).astype(np.float16).view(np.uint8)
    W = oracle.gguf_dequant_rows(qtype, w, out, in_).astype(np.float64)
    x = (rng.standard_normal((n, in_)) + 1).astype(np.float32)
    y = torch.zeros(n, out, device="cuda")
    ops.ref_gemm_q(qtype, _dev(x), _dev(w), None, y, w.shape[1])
    # the types without an offset have 9.5e-8 here at most; 10 % for the two roundings more per block
    assert _err(y.cpu().numpy(), x.astype(np.float64) @ W.T) < 1.045e-7


# int8 linears of at most 32-token tiles and gate/up of at most 16 rows add the exact
# integer dots in 64 bits: the result is the exact value rounded once, offsets included.
# (Scales and offsets are exact in fp32; the reference adds both parts in 64 bits, where
# dequantized fp32 weights would be rounded.) 1e-3: the 64-bit sums' own error beside a tie.
@pytest.mark.parametrize("qtype", [8, 12, 13, 14])
@pytest.mark.parametrize("n", [1, 16, 32])
def test_int8_linears_round_once(oracle, qtype, n):
    rng = np.random.default_rng(qtype + n)
    in_, out = 2304, 512
    w = random_gguf_rows(qtype, out, in_, rng)
    if qtype in (12, 13):
        parts = []
        for zero in (slice(2, 4), slice(0, 2)):   # ds * q, then -dm
            b = w.copy().reshape(out, in_ // 256, -1)
            b[:, :, zero] = 0
            parts.append(oracle.gguf_dequant_rows(qtype, b.reshape(w.shape), out, in_).astype(np.float64))
        W = parts[0] + parts[1]
    else:
        W = oracle.gguf_dequant_rows(qtype, w, out, in_).astype(np.float64)
    xq, xs, xd = _quant((rng.standard_normal((n, in_)) + 1).astype(np.float32))
    y = torch.full((n, out), float("nan"), device="cuda")
    wp = np.concatenate([w, np.zeros((out, -w.shape[1] % 4), np.uint8)], 1)
    ops.ref_gemm_q_i8(qtype, xq, xs, _dev(wp), None, y, wp.shape[1])
    assert (y.cpu().numpy() != (xd @ W.T).astype(np.float32)).mean() < 1e-3


# The matrix cores' fp32 addition rounds down: without the blocks of negated
# activations the mean error of these outputs is -5.9e-8 to -7.6e-8 of their rms
# (measured), with them 4e-9 at most. 8192 or more outputs of an rms error of 9e-8
# have a mean of 1e-9 by chance; a quarter of the smallest uncancelled one is the
# bound. (Q3_K, Q6_K and IQ4_XS hardly show it, Q4_K and Q5_K have the offset's error
# on top.) Rows off 16-byte alignment take the vector kernels: the sums of pieces are
# to be no further from 64 bits than theirs.
@pytest.mark.parametrize("fmt", [8, 18, "w4"])
@pytest.mark.parametrize("n", [16, 40])
def test_long_sums_have_no_bias(oracle, fmt, n):
    rng = np.random.default_rng(n)
    in_, out = 6144, 512
    if fmt == "w4":
        q = rng.integers(0, 256, (out, in_ // 2), dtype=np.uint8)
        s = rng.uniform(0.001, 0.02, (out, in_ // 128)).astype(np.float32)
        W = oracle.dequant_int4_rows(q, s, in_, 128).astype(np.float64)
        run = lambda x, y: ops.ref_gemm_w4a16(x, _dev(q), _dev(s), None, y, 128)
    else:
        w = random_gguf_rows(fmt, out, in_, rng)
        W = oracle.gguf_dequant_rows(fmt, w, out, in_).astype(np.float64)
        run = lambda x, y: ops.ref_gemm_q(fmt, x, _dev(w), None, y, w.shape[1])
    x = rng.standard_normal((n, in_)).astype(np.float32)
    ref = x.astype(np.float64) @ W.T
    err = []
    for off in (0, 1):
        xd = torch.zeros(n * in_ + 1, device="cuda")[off:off + n * in_].view(n, in_)
        xd.copy_(torch.from_numpy(x))
        y = torch.full((n, out), float("nan"), device="cuda")
        run(xd, y)
        err.append((y.cpu().numpy() - ref) / np.sqrt((ref ** 2).mean()))
    assert abs(err[0].mean()) < 1.5e-8
    assert np.sqrt((err[0] ** 2).mean()) < np.sqrt((err[1] ** 2).mean())


def test_unaligned_elementwise(oracle):
    # quantize_act_q8 and the combine on rows that are not 16-byte aligned.
    rng = np.random.default_rng(8)
    n, k, I, H, E, topk = 5, 96, 256, 512, 8, 4
    x = rng.standard_normal((n, k)).astype(np.float32)
    xf = torch.zeros(n * k + 1, device="cuda")
    xf[1:] = _dev(x.reshape(-1))
    xq, xs = torch.zeros(n * k + 1, dtype=torch.int8, device="cuda"), torch.zeros(n, k // 32, device="cuda")
    ops.ref_quantize_act_q8(xf[1:].view(n, k), xq[1:].view(n, k), xs)
    q, s = oracle.quant_act_q8(x)
    assert np.array_equal(xq[1:].cpu().numpy().reshape(n, k), q) and np.array_equal(xs.cpu().numpy(), s)
    g = _dev(random_gguf_rows(8, E * I, H, rng))
    d = _dev(random_gguf_rows(8, E * H, I, rng))
    x = _dev(rng.standard_normal((n, H)).astype(np.float32) * 0.02)
    ids = _dev(np.stack([rng.permutation(E)[:topk] for _ in range(n)]).astype(np.int32))
    w = _dev(rng.uniform(0.1, 1.0, (n, topk)).astype(np.float32))
    outs = []
    for off in (0, 1):
        dpart = torch.zeros(n * topk * H + off, device="cuda")[off:]
        out = torch.zeros(n, H, device="cuda")
        ops.ref_moe_expert_ffn_q((8, 8, 8), x, ids, w, g, g, d, I, E, (H // 32 * 34, H // 32 * 34, I // 32 * 34),
                                 torch.zeros(n * topk, I, device="cuda"), dpart, out, None)
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1]) and float(outs[0].abs().sum()) > 0
