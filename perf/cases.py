"""Performance cases of the quantized matmul path: what an inference engine calls on one GPU, through arcinfer_amd.qmatmul.

Kinds of case (a dict of plain values):
  gemv    one decode product, T tokens (1..8) against one read of a weight, called as an engine without graphs calls it
  ffn     a dense FFN layer: RMS norm + quantize, gate and up products, SwiGLU + quantize, down product. Decode sizes
          (M <= 8 tokens: GEMVs) replay a captured graph, as a decode loop does; prompts (GEMMs, the up product fused
          with silu(gate) through accumulate = 2) are called eagerly
  gemm    one prompt product of M tokens whose int8 activations are in hand
  moe     a mixture-of-experts FFN: routing, expert products and the weighted sum into x
Weights are random GGUF blocks (quants and sub-scales uniform, super-scales |N(0, sigma)|), activations N(0, 1) with
1 % outlier channels, router logits Zipf-distributed. Sizes are the repository's benchmark shapes (27B-class FFN:
5120 / 17408; 256 experts of 512, hidden 2048), and others of the same ranges.
"""
import math
import os
import re

import numpy as np
import torch

from arcinfer_amd import formats as F
from arcinfer_amd import qmatmul as qm

TYPES = ("Q8_0", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "IQ3_S")
MOE_TYPES = ("Q8_0", "IQ4_XS", "IQ3_S", "Q6_K")


def listed():
    return [
        # the smallest call: one attention-sized projection of one token
        {"name": "gemv_q8_0_4096", "kind": "gemv", "type": "Q8_0", "N": 4096, "K": 4096, "T": 1},
        # batch-1 decode of one FFN layer
        {"name": "ffn_decode_iq4_xs", "kind": "ffn", "type": "IQ4_XS", "down": "IQ4_XS", "E": 5120, "F": 17408, "M": 1},
        # speculative verification of five draft tokens, the usual mixed file (down in Q6_K)
        {"name": "ffn_verify5_q4_k", "kind": "ffn", "type": "Q4_K", "down": "Q6_K", "E": 5120, "F": 17408, "M": 5},
        # a short chat turn, or a batch of 24 decoding sequences
        {"name": "ffn_short24_iq4_xs", "kind": "ffn", "type": "IQ4_XS", "down": "IQ4_XS", "E": 5120, "F": 17408, "M": 24},
        # a medium prompt of ragged length, a whole FFN layer
        {"name": "ffn_prompt777_q4_k", "kind": "ffn", "type": "Q4_K", "down": "Q6_K", "E": 5120, "F": 17408, "M": 777},
        # attention-sized projection of a 512-token prompt
        {"name": "gemm_iq3_s_512", "kind": "gemm", "type": "IQ3_S", "N": 5120, "K": 5120, "M": 512, "act32": True},
        # long rows, ragged token count
        {"name": "gemm_q5_k_333", "kind": "gemm", "type": "Q5_K", "N": 5120, "K": 17408, "M": 333, "act32": True},
        # the 2K-token prompt product, in the file types that are used most
        {"name": "gemm_q4_k_2048", "kind": "gemm", "type": "Q4_K", "N": 17408, "K": 5120, "M": 2048, "act32": True},
        {"name": "gemm_iq4_xs_2048", "kind": "gemm", "type": "IQ4_XS", "N": 17408, "K": 5120, "M": 2048, "act32": True},
        # MoE layer: four decoding tokens, a short prompt, a long prompt
        {"name": "moe_decode4", "kind": "moe", "type": "IQ4_XS", "down": "IQ4_XS", "NE": 256, "NU": 8, "E": 2048,
         "F": 512, "T": 4},
        {"name": "moe_short96", "kind": "moe", "type": "IQ4_XS", "down": "Q6_K", "NE": 256, "NU": 8, "E": 2048,
         "F": 512, "T": 96},
        {"name": "moe_prompt4096", "kind": "moe", "type": "IQ4_XS", "down": "IQ4_XS", "NE": 256, "NU": 8, "E": 2048,
         "F": 512, "T": 4096},
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(("gemv", "ffn", "ffn", "gemm", "gemm", "gemm", "moe", "moe"))
    t = rng.choice(TYPES)
    if kind == "gemv":
        return {"kind": kind, "type": t, "N": _log_int(rng, 512, 17408, 16), "K": _log_int(rng, 1024, 17408, 256),
                "T": rng.randint(1, 8)}
    if kind == "ffn":
        down = rng.choice((t, t, "Q6_K"))
        M = rng.choice((rng.randint(1, 8), _log_int(rng, 9, 777)))
        return {"kind": kind, "type": t, "down": down, "E": _log_int(rng, 1024, 5120, 256),
                "F": _log_int(rng, 2048, 17408, 256), "M": M}
    if kind == "gemm":
        return {"kind": kind, "type": t, "N": _log_int(rng, 1024, 17408, 16), "K": _log_int(rng, 1024, 5120, 256),
                "M": _log_int(rng, 9, 2048), "act32": rng.random() < 0.8}
    t = rng.choice(MOE_TYPES)
    return {"kind": kind, "type": t, "down": rng.choice((t, t, "Q6_K")), "NE": rng.choice((32, 64, 128, 256)),
            "NU": rng.choice((4, 6, 8)), "E": _log_int(rng, 1024, 2048, 256), "F": rng.choice((256, 512, 768)),
            "T": _log_int(rng, 1, 2048)}


# ---- inputs -----------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _half_bytes(n, sigma, g):
    d = torch.randn(n, generator=g, device="cuda").abs_().mul_(sigma).half()
    return d.view(torch.uint8).view(n, 2)


def _blocks(name, rows, K, seed):
    """Random GGUF bytes of a weight, uint8 [rows, row bytes], made on the GPU."""
    g = _gen(seed)
    if name == "Q8_0":
        n = rows * K // 32
        b = torch.empty((n, 34), dtype=torch.uint8, device="cuda")
        b[:, 2:] = torch.randint(-127, 128, (n, 32), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        b[:, :2] = _half_bytes(n, 0.02 / 127, g)
        return b.view(rows, -1)
    n = rows * K // 256
    t = F.TYPES_BY_NAME[name]
    b = torch.randint(0, 256, (n, F.SB_BYTES[t]), generator=g, device="cuda", dtype=torch.uint8)
    at = 208 if name == "Q6_K" else 0
    b[:, at:at + 2] = _half_bytes(n, 0.01, g)
    if name in ("Q4_K", "Q5_K"):
        b[:, 2:4] = _half_bytes(n, 0.01, g)
    return b.view(rows, -1)


def _rows(M, K, seed):
    """f32 activations, 1 % of the channels 20 times larger."""
    g = _gen(seed)
    x = torch.randn((M, K), generator=g, device="cuda")
    ch = torch.randperm(K, generator=g, device="cuda")[:max(1, K // 100)]
    x[:, ch] *= 20.0
    return x


def _logits(T, NE, seed):
    g = _gen(seed)
    rank = torch.randperm(NE, generator=g, device="cuda").float() + 1
    u = torch.rand((T, NE), generator=g, device="cuda").clamp_(1e-7, 1 - 1e-7)
    return -1.1 * torch.log(rank)[None, :] - torch.log(-torch.log(u))


def _weight(name, rows, K, seed):
    return qm.QWeight(F.TYPES_BY_NAME[name], _blocks(name, rows, K, seed), rows, K)


def _stride(M):
    return (M + 15) // 16 * 16


def prepare(case, seed):
    s = {"case": case}
    k = case["kind"]
    seed = seed * 16
    if k in ("gemv", "gemm"):
        M = case["T"] if k == "gemv" else case["M"]
        s["w"] = _weight(case["type"], case["N"], case["K"], seed)
        x = _rows(M, case["K"], seed + 1)
        s["acts"] = qm.quantize_act(x, M_stride=_stride(M), act32=case.get("act32", True))
        s["C"] = torch.empty((M, case["N"]), device="cuda")
    elif k == "ffn":
        E, Fw, M = case["E"], case["F"], case["M"]
        s["gate"] = _weight(case["type"], Fw, E, seed)
        s["up"] = _weight(case["type"], Fw, E, seed + 1)
        s["down"] = _weight(case["down"], E, Fw, seed + 2)
        s["x"] = _rows(M, E, seed + 3)
        s["norm"] = torch.rand(E, generator=_gen(seed + 4), device="cuda") + 0.5
        s["y"] = torch.empty((M, E), device="cuda")
        if M <= 8:
            s["gu"] = torch.empty((M, 2 * Fw), device="cuda")
            _ffn(s)  # (first-launch work stays out of the capture)
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                _ffn(s)
        else:
            s["h"] = torch.empty((M, Fw), device="cuda")
    else:
        E, Fw, NE, T = case["E"], case["F"], case["NE"], case["T"]
        s["gate"] = _weight(case["type"], NE * Fw, E, seed)
        s["up"] = _weight(case["type"], NE * Fw, E, seed + 1)
        s["down"] = _weight(case["down"], NE * E, Fw, seed + 2)
        s["logits"] = _logits(T, NE, seed + 3)
        s["acts"] = qm.quantize_act(_rows(T, E, seed + 4), M_stride=_stride(T))
        s["x"] = torch.empty((T, E), device="cuda")
        s["ws"] = qm.moe_workspace(T, NE, case["NU"], E, Fw)
    return s


EPS = 1e-6


def _ffn(s):
    case = s["case"]
    Fw, M = case["F"], case["M"]
    aq, asc, absum, _ = qm.rmsnorm_quant(s["x"], s["norm"], EPS, M_stride=_stride(M))
    if M <= 8:
        gu = s["gu"]
        qm.gemv(s["gate"], aq, asc, absum, T=M, C=gu, ldc=2 * Fw)
        qm.gemv(s["up"], aq, asc, absum, T=M, C=gu, ldc=2 * Fw, c_off=Fw)
        hq = qm.swiglu_quant(gu, Fw, M_stride=_stride(M))
        return qm.gemv(s["down"], *hq, T=M, C=s["y"])
    qm.gemm(s["gate"], aq, asc, absum, M=M, C=s["h"])
    qm.gemm(s["up"], aq, asc, absum, M=M, C=s["h"], accumulate=2)
    hq = qm.swiglu_quant(s["h"], Fw, fused=True, M_stride=_stride(M))
    return qm.gemm(s["down"], *hq, M=M, C=s["y"])


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "gemv":
        return qm.gemv(state["w"], *state["acts"], T=case["T"], C=state["C"])
    if k == "gemm":
        return qm.gemm(state["w"], *state["acts"], M=case["M"], C=state["C"], act32=case["act32"])
    if k == "ffn":
        if "graph" in state:
            state["graph"].replay()
            return [state["gu"], state["y"]]
        y = _ffn(state)
        return [state["h"], y]
    aq, asc, _ = state["acts"]
    return qm.moe_grouped(state["gate"], state["up"], state["down"], case["NE"], state["logits"], case["NU"], aq, asc,
                          state["x"], state["ws"])


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def _wb(name, rows, K):
    return F.weight_bytes(F.TYPES_BY_NAME[name], rows, K)


def work(case):
    k = case["kind"]
    if k in ("gemv", "gemm"):
        M, N, K = case["T"] if k == "gemv" else case["M"], case["N"], case["K"]
        return {"bytes": _wb(case["type"], N, K) + M * K + M * K // 8 + 4 * M * N, "flops": 2.0 * M * N * K}
    E, Fw = case["E"], case["F"]
    if k == "ffn":
        M = case["M"]
        b = 2 * _wb(case["type"], Fw, E) + _wb(case["down"], E, Fw) + 4 * M * E + 4 * M * E + 4 * E
        return {"bytes": b + (8 if M <= 8 else 4) * M * Fw, "flops": 6.0 * M * E * Fw}
    T, NE, NU = case["T"], case["NE"], case["NU"]
    # (experts a batch reaches: T * NU picks, uniform; the router's skew makes it somewhat fewer)
    n = int(NE * (1.0 - (1.0 - 1.0 / NE) ** (T * NU)))
    b = n * (2 * _wb(case["type"], Fw, E) + _wb(case["down"], E, Fw)) + 4 * T * NE + T * E + T * E // 8 + 4 * T * E
    return {"bytes": b, "flops": 6.0 * T * NU * E * Fw}


def tolerance(case):
    # one product: exact integer block sums, f32 scales and f32 sums over up to 544 blocks (measured against 64 bits:
    # 1e-7 to 4e-7)
    if case["kind"] in ("gemv", "gemm"):
        return {"rel": 2e-6, "max": 2e-5}
    # chained products: an f32 difference in the last place moves a value across a rounding tie of the int8
    # quantization between them now and then, by a whole step (measured against 64 bits: 4e-5 to 6e-4)
    return {"rel": 1e-3, "max": 5e-2}


# ---- the same in 64 bits, in plain torch ------------------------------------------------------------------------------
_KV = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def _iq3s_grid():
    """The IQ3_S codebook (data: 512 words of four bytes) from the repository's table file, as float64 [512, 4]."""
    path = os.path.join(os.path.dirname(os.path.abspath(F.__file__)), "csrc", "iq_tables.inc")
    with open(path) as f:
        body = re.search(r"#define QM_IQ3S_GRID_INIT \{(.*?)\}", f.read(), re.S).group(1)
    words = np.array([int(w, 16) for w in re.findall(r"0x([0-9a-fA-F]+)u", body)], dtype=np.uint32)
    return torch.from_numpy(words.view(np.uint8).reshape(-1, 4).astype(np.float64)).cuda()


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _k_scales(b):
    """The eight 6-bit scales and mins of Q4_K / Q5_K superblocks: b uint8 [n, 12]."""
    b = b.int()
    lo_s, lo_m, hi = b[:, 0:4], b[:, 4:8], b[:, 8:12]
    sc = torch.cat([lo_s & 63, (hi & 15) | ((lo_s >> 6) << 4)], 1)
    mn = torch.cat([lo_m & 63, (hi >> 4) | ((lo_m >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _dequant(name, raw, K):
    """GGUF rows (uint8 [rows, bytes], on the GPU) -> float64 [rows, K]."""
    rows = raw.shape[0]
    if name == "Q8_0":
        b = raw.reshape(-1, 34)
        return (b[:, 2:].contiguous().view(torch.int8).double() * _f16(b[:, :2])).view(rows, K)
    b = raw.reshape(rows * K // 256, -1)
    n = b.shape[0]
    if name in ("Q4_K", "Q5_K"):
        d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        sc, mn = _k_scales(b[:, 4:16])
        qs = b[:, -128:].reshape(n, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32).double()
        if name == "Q5_K":
            qh = b[:, 16:48].reshape(n, 1, 32).int() >> torch.arange(8, device="cuda").view(1, 8, 1)
            q += 16.0 * (qh & 1).double()
        return (d[:, :, None] * sc[:, :, None] * q - dmin[:, :, None] * mn[:, :, None]).view(rows, K)
    if name == "Q6_K":
        ql, qh = b[:, :128].reshape(n, 2, 64).int(), b[:, 128:192].reshape(n, 2, 32).int()
        lo = torch.cat([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32)  # (per half: l, l + 32, then their high nibbles)
        hi = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (lo | (hi << 4)).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return (q.view(n, 16, 16) * sc[:, :, None] * _f16(b[:, 208:210])[:, :, None]).view(rows, K)
    if name == "IQ4_XS":
        kv = torch.tensor(_KV, dtype=torch.float64, device="cuda")
        sh = b[:, 2:4].contiguous().view(torch.int16).int() & 0xFFFF
        i = torch.arange(8, device="cuda")
        sl = (b[:, 4:8].int()[:, i // 2] >> (4 * (i % 2))) & 15
        sc = (sl | (((sh >> (2 * i)) & 3) << 4)) - 32
        qs = b[:, 8:136].reshape(n, 8, 16)
        q = kv[torch.cat([qs & 15, qs >> 4], 2).long()]
        return (q * (sc.double() * _f16(b[:, 0:2]))[:, :, None]).view(rows, K)
    # IQ3_S: d | qs[64] | qh[8] | signs[32] | scales[4]
    grid = _iq3s_grid()
    i8 = torch.arange(8, device="cuda")
    idx = b[:, 2:66].reshape(n, 8, 8).int() | (((b[:, 66:74].int()[:, :, None] >> i8) & 1) << 8)
    v = grid[idx.long()].reshape(n, 8, 32)
    sg = (b[:, 74:106].reshape(n, 8, 4, 1).int() >> i8) & 1
    v = torch.where(sg.reshape(n, 8, 32) == 1, -v, v)
    sc = 1.0 + 2.0 * ((b[:, 106:110].int()[:, i8 // 2] >> (4 * (i8 % 2))) & 15).double()
    return (v * (sc * _f16(b[:, 0:2]))[:, :, None]).view(rows, K)


def _times(x, name, raw, K):
    """x [M, K] float64 times the weight's transpose, a slice of its rows at a time."""
    return torch.cat([x @ _dequant(name, raw[r:r + 2048], K).T for r in range(0, raw.shape[0], 2048)], 1)


def _int8(x, B=32):
    """Rows quantized to int8 per B values and back: f32 input as the quantizer rounds it, float64 input in 64 bits."""
    a = x.cpu().numpy()
    v = a.reshape(a.shape[0], -1, B)
    top = np.abs(v).max(axis=2, keepdims=True)
    one = v.dtype.type(127)
    inv = np.divide(one, top, out=np.zeros_like(top), where=top > 0)
    q = np.rint(v * inv).astype(np.float64) * (top / one).astype(np.float64)
    return torch.from_numpy(q.reshape(a.shape)).cuda()


def _silu(x):
    return x / (1.0 + torch.exp(-x))


def exact(case, seed):
    k = case["kind"]
    seed = seed * 16
    if k in ("gemv", "gemm"):
        N, K = case["N"], case["K"]
        M = case["T"] if k == "gemv" else case["M"]
        x = _int8(_rows(M, K, seed + 1), 32 if case.get("act32", True) else 256)
        return _times(x, case["type"], _blocks(case["type"], N, K, seed), K)
    E, Fw = case["E"], case["F"]
    if k == "ffn":
        M = case["M"]
        x = _rows(M, E, seed + 3).double()
        norm = (torch.rand(E, generator=_gen(seed + 4), device="cuda") + 0.5).double()
        a = _int8(x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * norm)
        g = _times(a, case["type"], _blocks(case["type"], Fw, E, seed), E)
        u = _times(a, case["type"], _blocks(case["type"], Fw, E, seed + 1), E)
        h = _silu(g) * u
        y = _times(_int8(h), case["down"], _blocks(case["down"], E, Fw, seed + 2), Fw)
        return [torch.cat([g, u], 1) if M <= 8 else h, y]
    T, NE, NU = case["T"], case["NE"], case["NU"]
    a = _int8(_rows(T, E, seed + 4))
    lg = _logits(T, NE, seed + 3).double()
    top, ids = lg.topk(NU, 1)
    wts = torch.softmax(top, 1)
    gate = _blocks(case["type"], NE * Fw, E, seed)
    up = _blocks(case["type"], NE * Fw, E, seed + 1)
    down = _blocks(case["down"], NE * E, Fw, seed + 2)
    y = torch.zeros((T, E), dtype=torch.float64, device="cuda")
    for e in range(NE):
        t, j = (ids == e).nonzero(as_tuple=True)
        if len(t) == 0:
            continue
        fr, er = slice(e * Fw, (e + 1) * Fw), slice(e * E, (e + 1) * E)
        h = _silu(a[t] @ _dequant(case["type"], gate[fr], E).T) * (a[t] @ _dequant(case["type"], up[fr], E).T)
        y[t] += wts[t, j][:, None] * (_int8(h) @ _dequant(case["down"], down[er], Fw).T)
    return y
