"""The performance cases: the MoE branch of one transformer layer, as users of this package run it.

Every case is one pass over a whole MoE block (router, dispatch, routed experts, shared expert,
combine) at one batch, through the package's public entry points. Six ways to run it ("path"):

  w4         W4A16MoELayer.forward      bf16 activations: decode, speculative verify, prefill
  w4_f32     W4A16MoELayer.forward_f32  the caller's fp32 post-norm rows, rounded inside
  fp8        FP8MoELayer.forward        e4m3 block-scaled experts
  launchers  the reference-signature launchers one by one (fp32 rows, W4 experts registered with
             their packed copy, W4 shared expert through gemm_w4a16), the call sites a host keeps
  gguf_f32   the GGUF launchers with fp32 activations (expert types "gate,up,down", Q8_0 shared)
  gguf_i8    the same with int8 activations, the quantizer calls included

Geometries: the GLM-5-class layer (hidden 6144, 256 experts, top-8, expert width 2048), its share
under 8-way tensor parallelism (width 256), and small layers. Batches go from one token to a
prefill chunk, ragged counts among them.
"""
import math

import numpy as np
import torch

import glmserve_amd as G
from glmserve_amd import ops

# (hidden, expert width, routed experts, top-k)
GLM = (6144, 2048, 256, 8)
GLM_TP8 = (6144, 256, 256, 8)
MID = (2048, 512, 32, 4)
TINY = (256, 128, 16, 4)
SERVED = "18,18,23"          # IQ3_XXS gate / up, IQ4_XS down
Q8_0 = 8
BLOCK = {8: (32, 34), 12: (256, 144), 14: (256, 210), 18: (256, 98), 23: (256, 136)}
# fp16 block scales that give weights of about N(0, 0.02) with random codes
SCALE = {8: 2.7e-4, 12: 1.0e-4, 14: 1.5e-5, 18: 1.6e-4, 23: 1.6e-5}


def _case(path, shape, n, zipf=0.0, types=SERVED, name=None):
    c = {"path": path, "H": shape[0], "I": shape[1], "E": shape[2], "k": shape[3], "n": n,
         "zipf": zipf, "types": types}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One decoding sequence: launches and latency.
        _case("w4", GLM, 1, name="w4_decode_1"),
        # A few sequences, the host's fp32 rows, an odd batch.
        _case("w4_f32", GLM, 13, name="w4_f32_decode_13"),
        # A full decode batch (the headline workload).
        _case("w4", GLM, 64, name="w4_decode_64"),
        # Speculative verify, 8 sequences x 65 tokens, few experts take most rows.
        _case("w4", GLM, 520, zipf=1.1, name="w4_verify_520"),
        # A prefill chunk.
        _case("w4", GLM, 4096, name="w4_prefill_4096"),
        # FP8 experts: a decode batch and a long prefill chunk.
        _case("fp8", GLM, 24, name="fp8_decode_24"),
        _case("fp8", GLM, 8192, name="fp8_prefill_8192"),
        # A host that keeps the launchers' call sites, a short prompt of odd length.
        _case("launchers", GLM, 203, name="launchers_203"),
        # The GGUF checkpoint: one sequence, a decode batch, prompts.
        _case("gguf_f32", GLM, 1, name="gguf_f32_decode_1"),
        _case("gguf_i8", GLM, 64, name="gguf_i8_decode_64"),
        _case("gguf_f32", GLM, 1000, name="gguf_f32_prefill_1000"),
        _case("gguf_i8", GLM, 1024, name="gguf_i8_prefill_1024"),
    ]


# Largest batch of each path's range.
MAX_N = {"w4": 4096, "w4_f32": 4096, "fp8": 8192, "launchers": 1024, "gguf_f32": 1000,
         "gguf_i8": 1024}


def draw(rng):
    path = rng.choice(sorted(MAX_N))
    gguf = path.startswith("gguf")
    # The GGUF super-blocks need widths of whole 256s.
    shape = rng.choice([GLM, GLM, GLM, GLM_TP8, MID] + ([] if gguf else [TINY]))
    n = int(round(math.exp(rng.uniform(0.0, math.log(MAX_N[path])))))
    zipf = rng.choice([0.0, 0.0, 1.1])
    types = rng.choice([SERVED, SERVED, "8,8,8", "12,12,14"]) if gguf else SERVED
    return _case(path, shape, n, zipf, types)


# ---- inputs ------------------------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1009 + salt)
    return g


def _bytes(g, *shape):
    """Uniform random bytes (shape's last dimension a multiple of 8, or any total that is)."""
    total = int(np.prod(shape))
    w = torch.randint(-2**63, 2**63 - 1, ((total + 7) // 8,), generator=g, device="cuda",
                      dtype=torch.int64)
    return w.view(torch.uint8)[:total].view(*shape)


def _router(c, seed):
    """Router weights, correction bias (with a Zipf log-prior over the experts where asked for) and
    activations, all fp32 holding the values the path has them in."""
    g = _gen(seed, 1)
    H, E, n = c["H"], c["E"], c["n"]
    wr = 0.02 * torch.randn(E, H, generator=g, device="cuda")
    bias = torch.rand(E, generator=g, device="cuda") * 0.2 - 0.1
    if c["zipf"]:
        rank = torch.randperm(E, generator=g, device="cuda").float()
        bias = bias - c["zipf"] * torch.log(rank + 1.0)
    x = torch.randn(n, H, generator=g, device="cuda")
    if c["path"] in ("w4", "fp8"):
        x, wr = x.bfloat16().float(), wr.bfloat16().float()
    elif c["path"] == "w4_f32":
        wr = wr.bfloat16().float()
    return wr, bias, x


def _mats(c):
    H, I = c["H"], c["I"]
    return ((I, H), (I, H), (H, I))


def _w4_raw(c, seed, m, shared):
    """Matrix kind m (0 gate, 1 up, 2 down): int4 codes [*, rows, K/2], scales [*, rows, K/128]."""
    rows, K = _mats(c)[m]
    nm = 1 if shared else c["E"]
    g = _gen(seed, 10 + m + (5 if shared else 0))
    q = _bytes(g, nm, rows, K // 2)
    s = (0.01 * torch.randn(nm, rows, K // 128, generator=g, device="cuda")).abs()
    return q, s.bfloat16().float()


def _fp8_raw(c, seed, m, e0, e1):
    """Codes and 128 x 128 block scales of experts [e0, e1) (expert E: the shared one)."""
    rows, K = _mats(c)[m]
    g = _gen(seed, 100 + 1000 * m + e0)
    nm = e1 - e0
    v = torch.randn(nm, rows, K, generator=g, device="cuda").mul_(96.0).clamp_(-448.0, 448.0)
    s = (0.02 / 96.0) * (0.5 + torch.rand(nm, rows // 128, K // 128, generator=g, device="cuda"))
    return v.to(torch.float8_e4m3fn).view(torch.uint8), s


def _fp8_chunks(c):
    E = c["E"]
    return [(e, min(e + 16, E)) for e in range(0, E, 16)] + [(E, E + 1)]


def _row_bytes(t, K):
    return K // BLOCK[t][0] * BLOCK[t][1]


def _gguf_raw(t, nrows, K, g):
    """nrows rows of K elements of GGUF type t: random codes, finite block scales."""
    be, bb = BLOCK[t]
    nb = K // be
    q = _bytes(g, nrows, nb, bb)
    d = (0.5 + torch.rand(nrows, nb, 1, generator=g, device="cuda")) * SCALE[t]
    put = lambda off, v: q[:, :, off:off + 2].copy_(v.half().view(torch.uint8).view(nrows, nb, 2))
    put(208 if t == 14 else 0, d)
    if t == 12:
        put(2, 7.5 * d)
    return q.view(nrows, nb * bb)


def _gguf_weights(c, seed):
    types = [int(t) for t in c["types"].split(",")]
    H, I, E = c["H"], c["I"], c["E"]
    routed = [_gguf_raw(t, E * rows, K, _gen(seed, 20 + m))
              for m, (t, (rows, K)) in enumerate(zip(types, _mats(c)))]
    shared = [_gguf_raw(Q8_0, rows, K, _gen(seed, 30 + m)) for m, (rows, K) in enumerate(_mats(c))]
    return types, routed, shared


def prepare(case, seed):
    c = case
    path, H, I, E, k, n = c["path"], c["H"], c["I"], c["E"], c["k"], c["n"]
    wr, bias, x = _router(c, seed)
    f32 = lambda *shape: torch.empty(*shape, device="cuda")
    st = {"case": c, "x": x, "out": f32(n, H)}
    if path in ("w4", "w4_f32"):
        pk = []
        for shared in (False, True):
            for m, (rows, K) in enumerate(_mats(c)):
                q, s = _w4_raw(c, seed, m, shared)
                pk.append(G.pack_w4a16(q, s, q.shape[0], rows, K))
                del q, s
        layer = G.W4A16MoELayer(H, I, E, k, wr.bfloat16(), bias, pk[0], pk[1], pk[2],
                                (pk[3], pk[4], pk[5]))
        st["layer"] = layer
        if path == "w4":
            st["x"] = x.bfloat16()
            st["ws"] = layer.alloc_workspace(n)
        else:
            st["ws"] = layer.alloc_workspace_f32(n)
    elif path == "fp8":
        packed, scales = [], []
        for m, (rows, K) in enumerate(_mats(c)):
            pq = torch.empty((E + 1) * rows * K, dtype=torch.uint8, device="cuda")
            sc = f32(E + 1, rows // 128, K // 128)
            for e0, e1 in _fp8_chunks(c):
                q, s = _fp8_raw(c, seed, m, e0, e1)
                G.pack_fp8(q, e1 - e0, rows, K, out=pq[e0 * rows * K:e1 * rows * K])
                sc[e0:e1] = s
            packed.append(pq)
            scales.append(sc)
        cut = [E * rows * K for rows, K in _mats(c)]
        r = [(packed[m][:cut[m]], scales[m][:E]) for m in range(3)]
        sh = tuple((packed[m][cut[m]:], scales[m][E:]) for m in range(3))
        layer = G.FP8MoELayer(H, I, E, k, wr.bfloat16(), bias, r[0], r[1], r[2], sh)
        st.update(layer=layer, x=x.bfloat16(), ws=layer.alloc_workspace(n))
    else:
        st.update(wr=wr, bias=bias, logits=f32(n, E),
                  ids=torch.empty(n, k, dtype=torch.int32, device="cuda"), w=f32(n, k),
                  g=f32(n, I), u=f32(n, I), gu=f32(n, I), sh=f32(n, H))
        if path == "launchers":
            raw = [t for m in range(3) for t in _w4_raw(c, seed, m, False)]
            st["experts"] = ops.RefW4Experts(*raw, hidden=H, moe_inter=I)
            st["ws"] = torch.empty(st["experts"].workspace_bytes(n, k), dtype=torch.uint8,
                                   device="cuda")
            st["shared"] = [tuple(t[0] for t in _w4_raw(c, seed, m, True)) for m in range(3)]
        else:
            types, routed, shared = _gguf_weights(c, seed)
            st.update(types=types, routed=routed, shared=shared,
                      rb=[_row_bytes(t, K) for t, (_, K) in zip(types, _mats(c))],
                      srb=[_row_bytes(Q8_0, K) for _, K in _mats(c)],
                      h=f32(n * k, I), dpart=f32(n * k, H),
                      disp=torch.empty(3 * E + 1 + n * k, dtype=torch.int32, device="cuda"))
            if path == "gguf_i8":
                i8 = lambda r, w: torch.empty(r, w, dtype=torch.int8, device="cuda")
                st.update(xq=i8(n, H), xs=f32(n, H // 32), hq=i8(n * k, I), hs=f32(n * k, I // 32),
                          gq=i8(n, I), gs=f32(n, I // 32))
    torch.cuda.synchronize()
    return st


# ---- one pass ----------------------------------------------------------------------------------

def run(state):
    st = state
    c = st["case"]
    path, H, I, E, k, n = c["path"], c["H"], c["I"], c["E"], c["k"], c["n"]
    x, out = st["x"], st["out"]
    if path in ("w4", "fp8"):
        st["layer"].forward(x, out, st["ws"])
        return out
    if path == "w4_f32":
        st["layer"].forward_f32(x, out, st["ws"])
        return out
    ids, w, gu, sh = st["ids"], st["w"], st["gu"], st["sh"]
    G.router_logits_f32(x, st["wr"], None, st["logits"])
    G.moe_router(st["logits"], st["bias"], n, E, k, True, 2.5, ids, w)
    if path == "launchers":
        ops.RefW4Experts.set_workspace(st["ws"])
        st["experts"].ffn(x, ids, w, out)
        (gq, gs), (uq, us), (dq, ds) = st["shared"]
        ops.ref_gemm_w4a16(x, gq, gs, None, st["g"])
        ops.ref_gemm_w4a16(x, uq, us, None, st["u"])
        ops.ref_silu_mul(st["g"], st["u"], gu)
        ops.ref_gemm_w4a16(gu, dq, ds, None, sh)
    elif path == "gguf_f32":
        gq, uq, dq = st["routed"]
        ops.ref_moe_expert_ffn_q(st["types"], x, ids, w, gq, uq, dq, I, E, st["rb"], st["h"],
                                 st["dpart"], out, st["disp"])
        sg, su, sd = st["shared"]
        ops.ref_gemm_q(Q8_0, x, sg, None, st["g"], st["srb"][0])
        ops.ref_gemm_q(Q8_0, x, su, None, st["u"], st["srb"][1])
        ops.ref_silu_mul(st["g"], st["u"], gu)
        ops.ref_gemm_q(Q8_0, gu, sd, None, sh, st["srb"][2])
    else:
        gq, uq, dq = st["routed"]
        xq, xs = st["xq"], st["xs"]
        ops.ref_quantize_act_q8(x, xq, xs)
        ops.ref_moe_expert_ffn_q_i8(st["types"], xq, xs, ids, w, gq, uq, dq, I, E, st["rb"],
                                    st["h"], st["hq"], st["hs"], st["dpart"], out, st["disp"])
        sg, su, sd = st["shared"]
        ops.ref_gemm_q_i8(Q8_0, xq, xs, sg, None, st["g"], st["srb"][0])
        ops.ref_gemm_q_i8(Q8_0, xq, xs, su, None, st["u"], st["srb"][1])
        ops.ref_silu_mul(st["g"], st["u"], gu)
        ops.ref_quantize_act_q8(gu, st["gq"], st["gs"])
        ops.ref_gemm_q_i8(Q8_0, st["gq"], st["gs"], sd, None, sh, st["srb"][2])
    ops.ref_add_inplace(out, sh)
    return {"out": out, "logits": st["logits"], "ids": ids, "weights": w}


# ---- what a pass cannot do without --------------------------------------------------------------

def _distinct(c):
    """Distinct routed experts of a batch, from a host draw of the same distributions."""
    r = np.random.default_rng(5)
    E, n = c["E"], c["n"]
    bias = r.uniform(-0.1, 0.1, E)
    if c["zipf"]:
        bias -= c["zipf"] * np.log(r.permutation(E) + 1.0)
    logit = r.standard_normal((n, E)) * (0.02 * math.sqrt(c["H"]))
    choose = 1.0 / (1.0 + np.exp(-logit)) + bias
    return len(np.unique(np.argpartition(-choose, c["k"] - 1, axis=1)[:, :c["k"]]))


def work(case):
    c = case
    path, H, I, E, k, n = c["path"], c["H"], c["I"], c["E"], c["k"], c["n"]
    U = _distinct(c)
    w4 = 3 * (I * H // 2)
    xb, wb = (2, 2) if path in ("w4", "fp8") else (4, 2) if path == "w4_f32" else (4, 4)
    if path in ("w4", "w4_f32"):
        weights = (U + 1) * (w4 + 3 * I * H // 128 * 2)
    elif path == "fp8":
        weights = (U + 1) * 3 * (I * H + I * H // 128 // 128 * 4)
    elif path == "launchers":
        # packed experts (bf16 scales), shared expert in the launchers' own layout (fp32 scales)
        weights = U * (w4 + 3 * I * H // 128 * 2) + w4 + 3 * I * H // 128 * 4
    else:
        types = [int(t) for t in c["types"].split(",")]
        per = sum(rows * _row_bytes(t, K) for t, (rows, K) in zip(types, _mats(c)))
        weights = U * per + sum(rows * _row_bytes(Q8_0, K) for rows, K in _mats(c))
    nbytes = weights + E * H * wb + E * 4 + n * H * xb + n * H * 4
    if path not in ("w4", "w4_f32", "fp8"):
        nbytes += n * E * 4
    return {"bytes": nbytes, "flops": 2 * n * H * E + n * (k + 1) * 6 * H * I}


def tolerance(case):
    return TOLERANCE[case["path"]]


# About four times the relative error each path shows against exact() over the ranges above: 1.6e-3
# with bf16 / fp16 intermediates (w4), 1.0e-3 with the shared expert in fp32 (launchers), 1.9e-3 with
# e4m3 ones, whose codes flip near ties (fp8), 2.3e-7 with fp32 sums (gguf_f32), 1.2e-4 with int8 codes
# of the intermediate that flip near ties (gguf_i8).
TOLERANCE = {
    "w4": {"rel": 6e-3},
    "w4_f32": {"rel": 6e-3},
    "fp8": {"rel": 8e-3},
    "launchers": {"rel": 4e-3},
    "gguf_f32": {"rel": 1e-6},
    "gguf_i8": {"rel": 5e-4},
}


# ---- the same in 64 bits -------------------------------------------------------------------------

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _deq_gguf(t, q, K):
    """Rows of GGUF type t (uint8 [rows, row_bytes]) as float64 [rows, K]."""
    be, bb = BLOCK[t]
    rows, nb = q.shape[0], K // be
    b = q.view(rows, nb, bb)
    i = b.to(torch.int64)
    if t == 8:
        w = _f16(b[:, :, 0:2]) * b[:, :, 2:].contiguous().view(torch.int8).double()
    elif t == 12:
        s, qs = i[:, :, 4:16], i[:, :, 16:]
        lo_sc, lo_mn = s[:, :, 0:4] & 63, s[:, :, 4:8] & 63
        hi_sc = (s[:, :, 8:12] & 15) | ((s[:, :, 0:4] >> 6) << 4)
        hi_mn = (s[:, :, 8:12] >> 4) | ((s[:, :, 4:8] >> 6) << 4)
        sc, mn = torch.cat([lo_sc, hi_sc], 2).double(), torch.cat([lo_mn, hi_mn], 2).double()
        qs = qs.view(rows, nb, 4, 32)
        v = torch.stack([qs & 15, qs >> 4], 3).reshape(rows, nb, 8, 32).double()
        d, m = _f16(b[:, :, 0:2]).unsqueeze(3), _f16(b[:, :, 2:4]).unsqueeze(3)
        w = d * sc.unsqueeze(3) * v - m * mn.unsqueeze(3)
    elif t == 14:
        ql, qh = i[:, :, 0:128].view(rows, nb, 2, 2, 32), i[:, :, 128:192].view(rows, nb, 2, 32)
        sc = b[:, :, 192:208].contiguous().view(torch.int8).double()
        v = torch.stack([(ql[:, :, :, j % 2] >> (4 * (j // 2))) & 15 | (((qh >> (2 * j)) & 3) << 4)
                         for j in range(4)], 3)
        w = _f16(b[:, :, 208:210]).unsqueeze(3) * sc.unsqueeze(3) * \
            (v.reshape(rows, nb, 16, 16).double() - 32.0)
    elif t == 18:
        aux = i[:, :, 66:98].view(rows, nb, 8, 4)
        aux = aux[..., 0] | (aux[..., 1] << 8) | (aux[..., 2] << 16) | (aux[..., 3] << 24)
        i7 = torch.stack([(aux >> (7 * l)) & 127 for l in range(4)], 3)
        bits = torch.stack([(i7 >> e) & 1 for e in range(7)], 4)
        bits = torch.cat([bits, bits.sum(4, keepdim=True) & 1], 4)          # the parity sign
        grid = torch.tensor([int(v, 16) for v in IQ3_GRID.split()], device=q.device)
        g = grid[i[:, :, 2:66]].view(rows, nb, 8, 4, 2)
        mag = torch.stack([(g >> (8 * e)) & 255 for e in range(4)], 5).view(rows, nb, 8, 4, 8)
        db = _f16(b[:, :, 0:2]) * (0.5 + (aux >> 28).double()) * 0.5
        w = db.view(rows, nb, 8, 1, 1) * mag.double() * (1.0 - 2.0 * bits.double())
    else:                                                                    # IQ4_XS
        sh = i[:, :, 2] | (i[:, :, 3] << 8)
        sc = torch.stack([((i[:, :, 4 + j // 2] >> (4 * (j % 2))) & 15) | (((sh >> (2 * j)) & 3) << 4)
                          for j in range(8)], 2).double() - 32.0
        nl = torch.tensor(IQ4_NL, dtype=torch.float64, device=q.device)
        qs = i[:, :, 8:136].view(rows, nb, 8, 16)
        v = nl[torch.cat([qs & 15, qs >> 4], 3)]
        w = _f16(b[:, :, 0:2]).unsqueeze(3) * sc.unsqueeze(3) * v
    return w.reshape(rows, K)


def _deq_w4(q, s):
    rows, half = q.shape
    v = torch.stack([q & 15, q >> 4], 2).view(rows, half * 2).double() - 8.0
    return (v.view(rows, -1, 128) * s.double().unsqueeze(2)).view(rows, half * 2)


def _q_i8(v):
    """The int8 activation rule: per 32 values, scale absmax / 127, round half to even (fp32)."""
    v = v.float()
    b = v.reshape(v.shape[0], -1, 32)
    a = b.abs().amax(2, keepdim=True)
    s = a / torch.full_like(a, 127.0)      # a true division: by a number torch multiplies instead
    inv = torch.where(s > 0, 1.0 / s, torch.zeros_like(s))
    return (torch.round(b * inv).double() * s.double()).view(v.shape)


def _q_fp8(v):
    """The fp8 activation rule: per 128 values, scale amax / 448, e4m3 round to nearest even."""
    v = v.float()
    b = v.reshape(v.shape[0], -1, 128)
    a = b.abs().amax(2, keepdim=True)
    s = a / torch.full_like(a, 448.0)
    s = torch.where(s > 0, s, torch.ones_like(s))
    q = (b / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return (q.double() * s.double()).view(v.shape)


def exact(case, seed):
    c = case
    path, H, I, E, k, n = c["path"], c["H"], c["I"], c["E"], c["k"], c["n"]
    wr, bias, x = _router(c, seed)
    # The router of every path works on bf16 rows and weights.
    xb = x.bfloat16().double()
    logits = xb @ wr.bfloat16().double().t()
    score = torch.sigmoid(logits)
    ids = (score + bias.double()).topk(k, dim=1).indices
    w = score.gather(1, ids)
    w = 2.5 * w / w.sum(1, keepdim=True)

    act = {"fp8": _q_fp8, "gguf_i8": _q_i8}.get(path, lambda v: v)
    xe = act(x.double() if path.startswith("gguf") else xb)
    if path == "gguf_i8" or path == "gguf_f32":
        types, routed, shared = _gguf_weights(c, seed)
        mat = lambda m, e: (_deq_gguf(Q8_0, shared[m], _mats(c)[m][1]) if e == E else
                            _deq_gguf(types[m], routed[m].view(E, _mats(c)[m][0], -1)[e],
                                      _mats(c)[m][1]))
    elif path == "fp8":
        held = {}

        def mat(m, e):
            e0, e1 = (E, E + 1) if e == E else (e // 16 * 16, min(e // 16 * 16 + 16, E))
            if held.get(m, (None,))[0] != e0:
                held[m] = (e0,) + _fp8_raw(c, seed, m, e0, e1)
            _, q, s = held[m]
            v, s = q[e - e0].view(torch.float8_e4m3fn).double(), s[e - e0].double()
            return v * s.repeat_interleave(128, 0).repeat_interleave(128, 1)
    else:
        raw = [[_w4_raw(c, seed, m, sh) for m in range(3)] for sh in (False, True)]
        mat = lambda m, e: _deq_w4(raw[e == E][m][0][0 if e == E else e],
                                   raw[e == E][m][1][0 if e == E else e])

    def ffn(e, rows):
        g, u = rows @ mat(0, e).t(), rows @ mat(1, e).t()
        return act(g * torch.sigmoid(g) * u).double() @ mat(2, e).t()

    # The launchers' shared linears keep the caller's fp32 rows.
    out = ffn(E, x.double() if path == "launchers" else xe)
    for e in range(E):
        t, s = (ids == e).nonzero(as_tuple=True)
        if len(t):
            out.index_add_(0, t, w[t, s].unsqueeze(1) * ffn(e, xe[t]))
    if path in ("w4", "w4_f32", "fp8"):
        return out
    return {"out": out, "logits": logits, "ids": ids.int(), "weights": w}


# Format data of the GGUF types: the IQ4_NL values and the IQ3_XXS codebook (four magnitudes of one
# byte each per entry).
IQ4_NL = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
IQ3_GRID = """
    04040404 04040414 04040424 04040c0c 04040c1c 04040c3e 04041404 04041414 04041c0c 04042414 04043e1c 04043e2c
    040c040c 040c041c 040c0c04 040c0c14 040c140c 040c142c 040c1c04 040c1c14 040c240c 040c2c24 040c3e04 04140404
    04140414 04140424 04140c0c 04141404 04141414 04141c0c 04141c1c 04141c3e 04142c0c 04142c3e 04143e2c 041c040c
    041c043e 041c0c04 041c0c14 041c142c 041c3e04 04240c1c 04241c3e 04242424 04242c3e 04243e1c 04243e2c 042c040c
    042c043e 042c1c14 042c2c14 04341c2c 04343424 043e0c04 043e0c24 043e0c34 043e241c 043e340c 0c04040c 0c04041c
    0c040c04 0c040c14 0c04140c 0c04141c 0c041c04 0c041c14 0c041c24 0c04243e 0c042c04 0c0c0404 0c0c0414 0c0c0c0c
    0c0c1404 0c0c1414 0c14040c 0c14041c 0c140c04 0c140c14 0c14140c 0c141c04 0c143e14 0c1c0404 0c1c0414 0c1c1404
    0c1c1c0c 0c1c2434 0c1c3434 0c24040c 0c24042c 0c242c04 0c2c1404 0c2c1424 0c2c2434 0c2c3e0c 0c34042c 0c3e1414
    0c3e2404 14040404 14040414 14040c0c 14040c1c 14041404 14041414 14041434 14041c0c 14042414 140c040c 140c041c
    140c042c 140c0c04 140c0c14 140c140c 140c1c04 140c341c 140c343e 140c3e04 14140404 14140414 14140c0c 14140c3e
    14141404 14141414 14141c3e 14142404 14142c2c 141c040c 141c0c04 141c0c24 141c3e04 141c3e24 14241c2c 14242c1c
    142c041c 142c143e 142c240c 142c3e24 143e040c 143e041c 143e0c34 143e242c 1c04040c 1c040c04 1c040c14 1c04140c
    1c04141c 1c042c04 1c04342c 1c043e14 1c0c0404 1c0c0414 1c0c1404 1c0c1c0c 1c0c2424 1c0c2434 1c14040c 1c14041c
    1c140c04 1c14142c 1c142c14 1c143e14 1c1c0c0c 1c1c1c1c 1c241c04 1c24243e 1c243e14 1c2c0404 1c2c0434 1c2c1414
    1c2c2c2c 1c340c24 1c341c34 1c34341c 1c3e1c1c 1c3e3404 24040424 24040c3e 24041c2c 24041c3e 24042c1c 24042c3e
    240c3e24 24141404 24141c3e 24142404 24143404 24143434 241c043e 241c242c 24240424 24242c0c 24243424 242c142c
    242c241c 242c3e04 243e042c 243e0c04 243e0c14 243e1c04 2c040c14 2c04240c 2c043e04 2c0c0404 2c0c0434 2c0c1434
    2c0c2c2c 2c140c24 2c141c14 2c143e14 2c1c0414 2c1c2c1c 2c240c04 2c24141c 2c24143e 2c243e14 2c2c0414 2c2c1c0c
    2c342c04 2c3e1424 2c3e2414 34041424 34042424 34042434 34043424 340c140c 340c340c 34140c3e 34143424 341c1c04
    341c1c34 34242424 342c042c 342c2c14 34341c1c 343e041c 343e140c 3e04041c 3e04042c 3e04043e 3e040c04 3e041c14
    3e042c14 3e0c1434 3e0c2404 3e140c14 3e14242c 3e142c14 3e1c0404 3e1c0c2c 3e1c1c1c 3e1c3404 3e24140c 3e24240c
    3e2c0404 3e2c0414 3e2c1424 3e341c04
"""
