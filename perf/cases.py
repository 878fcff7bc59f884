"""The work this library is measured on: single layers and calls of a DeepSeek-V4-Flash
pipeline stage, through the package's public entry points.

Sizes are the V4-Flash shapes that bench.py and the tests use: hidden 4096, 256 routed
MXFP4 experts of 2048 (top-6) and one FP8 shared expert, q_lora 1024, 64 heads of 512,
the five FP8 projections of a block, a 128-row attention window with 512 selected rows.
Activations are bf16 N(0, 1) rows (a normed hidden state), FP4 weights the e2m1 codes of
a normal distribution with e8m0 scales around 2^-7, FP8 weights normal e4m3 codes with
128 x 128 block scales, so every product keeps an O(1) output.

Kinds of case:
  moe      HipMoE.forward: gate, top-6, the routed experts and the shared one, for T tokens
           (decode, speculative verification, prefill, a prompt longer than one chunk)
  stage    DecodeStage.replay: decoder blocks (norms, projections, residuals, MoE) as one graph
  proj     the attention side's prefill producers: residual + norm + quantisation, wq_a with
           wkv, q_norm, wq_b with the indexer's wq_b
  linear   one FP8 projection of a packed weight from bf16 rows (PackedFp8Linear)
  fp8      fp8_gemm on a row-major weight, as the reference's callers hold it
  fp4      fp4_gemm on a row-major MXFP4 expert weight (a layer the MoE path declines)
  grouped  grouped_fp4_gemm: one row per selected expert (the banked decode path)
  attn     sparse_attn: decode over a long cache, or the prefill of a prompt chunk
"""

import math

import torch

from wanferenz_amd import kernels, synth
from wanferenz_amd.moe import HipMoE, MoEConfig, MoEWeights
from wanferenz_amd.stage import DecodeStage, StageBlock

D, I, E, TOPK = 4096, 2048, 256, 6
ROUTE_SCALE, SWIGLU_LIMIT, EPS = 1.5, 10.0, 1e-6
VOCAB = 4096
Q_LORA, HEAD_DIM, Q_WIDTH, IDX_WIDTH = 1024, 512, 32768, 8192
WINDOW, SELECTED, RATIO = 128, 512, 4
# (N, K) of the FP8 projections of a block: wq_a, wkv, wq_b, the indexer's wq_b, wo_b, and
# the shared expert's w1 / w2
FP8_SHAPES = ((1024, 4096), (512, 4096), (32768, 1024), (8192, 1024), (4096, 8192), (2048, 4096), (4096, 2048))


def listed():
    return [
        # one decode step's MoE layer at one token: latency, 107 MB of weights
        {"name": "moe_t1", "kind": "moe", "T": 1, "route": "bias"},
        # a speculative verification / small batch: between the decode and the prefill widths
        {"name": "moe_t23", "kind": "moe", "T": 23, "route": "bias"},
        # the prefill of a 2048-token prompt with the skewed expert popularity of bench.py
        {"name": "moe_t2048", "kind": "moe", "T": 2048, "route": "zipf"},
        # a long prompt in one call, experts evenly loaded
        {"name": "moe_t6000", "kind": "moe", "T": 6000, "route": "bias"},
        # the graph-captured decode step of two blocks, four tokens
        {"name": "stage_t4", "kind": "stage", "T": 4, "blocks": 2},
        # the attention side's producers in the prefill of an odd prompt length
        {"name": "proj_m1999", "kind": "proj", "M": 1999},
        # the smallest call: the attention output projection of one decoded token
        {"name": "linear_m1", "kind": "linear", "M": 1, "N": 4096, "K": 8192, "ue8m0": True},
        # a short prompt through fp8_gemm on the reference's row-major weight and float scales
        {"name": "fp8_m100", "kind": "fp8", "M": 100, "N": 4096, "K": 4096, "ue8m0": False},
        # one popular expert's rows of a prefill through the row-major fp4_gemm
        {"name": "fp4_m333", "kind": "fp4", "M": 333, "N": 2048, "K": 4096},
        # the six selected experts' w1|w3 of one decoded token
        {"name": "grouped_g6", "kind": "grouped", "G": 6, "N": 4096, "K": 4096},
        # decode attention of four sequences, 64k of context behind each
        {"name": "attn_decode_b4", "kind": "attn", "B": 4, "S": 1, "start": 65535, "H": 64},
        # attention of a 2048-token prompt
        {"name": "attn_prefill_s2048", "kind": "attn", "B": 1, "S": 2048, "start": 0, "H": 64},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe", "stage", "proj", "linear", "linear", "fp8", "fp4", "grouped", "attn",
                       "attn"))
    if kind == "moe":
        return {"kind": kind, "T": _log_int(rng, 1, 6000), "route": rng.choice(("bias", "zipf", "hash"))}
    if kind == "stage":
        return {"kind": kind, "T": rng.randint(1, 8), "blocks": rng.randint(1, 2)}
    if kind == "proj":
        return {"kind": kind, "M": _log_int(rng, 5, 2048)}
    if kind in ("linear", "fp8"):
        n, k = rng.choice(FP8_SHAPES)
        return {"kind": kind, "M": _log_int(rng, 1, 2048 if kind == "linear" else 512), "N": n, "K": k,
                "ue8m0": rng.random() < 0.7}
    if kind == "fp4":
        n, k = rng.choice(((2048, 4096), (4096, 2048), (4096, 4096)))
        return {"kind": kind, "M": _log_int(rng, 1, 2048), "N": n, "K": k}
    if kind == "grouped":
        n, k = rng.choice(((4096, 4096), (4096, 2048)))
        return {"kind": kind, "G": rng.randint(1, 32), "N": n, "K": k}
    if rng.random() < 0.5:
        return {"kind": kind, "B": rng.randint(1, 8), "S": rng.choice((1, 1, 2, 5)), "start": _log_int(rng, 200, 65535),
                "H": rng.choice((16, 32, 64, 64))}
    return {"kind": kind, "B": 1, "S": _log_int(rng, 33, 2048), "start": rng.choice((0, _log_int(rng, 64, 8192))),
            "H": rng.choice((16, 32, 64, 64))}


# ---------------------------------------------------------------- inputs ------

def _gen(seed, tag):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1009 + tag * 7919) & 0x7FFFFFFF)


def _rows(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16)


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _fp4_code_table():
    """256 nibble codes whose uniform draw gives the e2m1 codes of N(0, 2)."""
    u = (torch.arange(256, dtype=torch.float64) + 0.5) / 256
    v = 2.0 * math.sqrt(2.0) * torch.erfinv(2 * u - 1)
    mag = torch.argmin((v.abs()[:, None] - torch.tensor(_E2M1, dtype=torch.float64)[None]).abs(), dim=1)
    return (mag + 8 * (v < 0).long()).to(torch.uint8).cuda()


def _fp4_codes(g, *shape):
    """Packed e2m1 bytes, filled in pieces so that the index temporaries stay small."""
    n = math.prod(shape)
    table = _fp4_code_table()
    out = torch.empty(n, dtype=torch.uint8, device="cuda")
    piece = 1 << 27
    for at in range(0, n, piece):
        m = min(piece, n - at)
        r = torch.randint(0, 65536, (m,), dtype=torch.int32, device="cuda", generator=g)
        out[at:at + m] = table[r & 255] | (table[r >> 8] << 4)
    return out.view(*shape)


def _fp4_scales(g, *shape):
    return torch.randint(119, 122, shape, dtype=torch.uint8, device="cuda", generator=g)


def _fp8_weight(g, n, k, e8m0=True):
    """(e4m3 [n, k], block scales [ceil(n/128), ceil(k/128)])."""
    w = (torch.randn(n, k, device="cuda", generator=g) * 64.0).clamp(-448, 448).to(torch.float8_e4m3fn)
    shape = ((n + 127) // 128, (k + 127) // 128)
    if e8m0:
        s = torch.randint(114, 117, shape, dtype=torch.uint8, device="cuda", generator=g).view(torch.float8_e8m0fnu)
    else:
        s = (0.7 + 0.7 * torch.rand(*shape, device="cuda", generator=g)) * 2.0 ** -12
    return w, s


def _moe_tensors(seed, tag, route):
    """One MoE layer's tensors in the reference's bank layout."""
    g = _gen(seed, tag)
    t = {"gate_w": (torch.randn(E, D, device="cuda", generator=g) * 0.02).to(torch.bfloat16), "gate_bias": None,
         "tid2eid": None}
    if route == "hash":
        t["tid2eid"] = torch.rand(VOCAB, E, device="cuda", generator=g).topk(TOPK, dim=1)[1].to(torch.int32)
    elif route == "zipf":
        t["gate_bias"] = torch.from_numpy(synth.zipf_bias(E, 1.1, synth.zipf_v4_beta())).cuda()
    else:
        t["gate_bias"] = torch.randn(E, device="cuda", generator=g) * 0.01
    t["w13"], t["w13_s"] = _fp4_codes(g, E, 2 * I, D // 2), _fp4_scales(g, E, 2 * I, D // 32)
    t["w2"], t["w2_s"] = _fp4_codes(g, E, D, I // 2), _fp4_scales(g, E, D, I // 32)
    for name, (n, k) in (("sh_w1", (I, D)), ("sh_w3", (I, D)), ("sh_w2", (D, I))):
        w, s = _fp8_weight(g, n, k)
        t[name], t[name + "_s"] = w.view(torch.uint8), s.view(torch.uint8)
    return t


def _moe_layer(t, max_tokens):
    cfg = MoEConfig(dim=D, inter=I, n_experts=E, topk=TOPK, route_scale=ROUTE_SCALE, swiglu_limit=SWIGLU_LIMIT)
    return HipMoE(cfg, MoEWeights(**t), max_tokens=max_tokens, keep_reference=False)


def _token_inputs(case, seed):
    g = _gen(seed, 1)
    ids = torch.randint(0, VOCAB, (case["T"],), device="cuda", generator=g) if case.get("route") == "hash" else None
    return _rows(g, case["T"], D), ids


def _norm_weight(g, n):
    return 0.5 + torch.rand(n, device="cuda", generator=g)


def _attn_side(seed, tag):
    """Norm weights and projections of a block's attention side: (attn_norm, q_norm, wq_a, wkv, wq_b, idx_wq_b)."""
    g = _gen(seed, tag)
    return {"attn_norm": _norm_weight(g, D), "q_norm": _norm_weight(g, Q_LORA), "wq_a": _fp8_weight(g, Q_LORA, D),
            "wkv": _fp8_weight(g, HEAD_DIM, D), "wq_b": _fp8_weight(g, Q_WIDTH, Q_LORA),
            "idx_wq_b": _fp8_weight(g, IDX_WIDTH, Q_LORA), "wo_b": _fp8_weight(g, D, IDX_WIDTH),
            "ffn_norm": _norm_weight(g, D)}


def _quant(x, ue8m0, e8m0_scales):
    """e4m3 codes and per-128 scales of bf16 rows, as act_quant defines them (plain torch)."""
    z = x.float().unflatten(-1, (-1, 128))
    amax = z.abs().amax(-1, keepdim=True).clamp_min(1e-4) * (1.0 / 448.0)
    if ue8m0:
        mant, exp = torch.frexp(amax)
        s = torch.ldexp(torch.ones_like(amax), torch.where(mant == 0.5, exp - 1, exp))
    else:
        s = amax
    q = (z / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).flatten(-2)
    s = s.squeeze(-1)
    if e8m0_scales:
        s = ((s.view(torch.int32) >> 23) & 255).to(torch.uint8).view(torch.float8_e8m0fnu)
    return q, s


def _gemm_inputs(case, seed):
    """a, its scales and the row-major weight of a linear / fp8 / fp4 / grouped case."""
    g = _gen(seed, 2)
    kind, n, k = case["kind"], case["N"], case["K"]
    if kind == "grouped":
        x = _rows(g, case["G"], k)
        w, s = _fp4_codes(g, case["G"], n, k // 2), _fp4_scales(g, case["G"], n, k // 32)
    else:
        x = _rows(g, case["M"], k)
        if kind == "fp4":
            w, s = _fp4_codes(g, n, k // 2), _fp4_scales(g, n, k // 32)
        else:
            w, s = _fp8_weight(g, n, k, e8m0=case["ue8m0"])
    if kind in ("fp4", "grouped"):
        w, s = w.view(torch.float4_e2m1fn_x2), s.view(torch.float8_e8m0fnu)
    return x, w, s


def _attn_inputs(case, seed):
    """q, kv, sink and the index rows: the causal window, then the selected compressed rows
    (one per four positions), best first, -1 where a position has fewer."""
    g = _gen(seed, 3)
    B, S, H, start = case["B"], case["S"], case["H"], case["start"]
    prev = min(WINDOW - 1, start)          # rows before the chunk that its windows reach
    comp = (start + S) // RATIO
    n = prev + S + comp
    q, kv = _rows(g, B, S, H, HEAD_DIM), _rows(g, B, n, HEAD_DIM)
    sink = torch.randn(H, device="cuda", generator=g)
    pos = torch.arange(S, device="cuda")[:, None]
    win = (pos + prev - WINDOW + 1).clamp(min=0) + torch.arange(min(prev + S, WINDOW), device="cuda")
    win = torch.where(win > pos + prev, torch.full_like(win, -1), win)
    have = (start + pos + 1) // RATIO
    m = min(SELECTED, comp)
    score = torch.rand(B, S, comp, device="cuda", generator=g)
    score = score.masked_fill(torch.arange(comp, device="cuda")[None, None] >= have[None], -1.0)
    val, sel = score.topk(m, dim=-1)
    sel = torch.where(val < 0, torch.full_like(sel, -1), sel + prev + S)
    idx = torch.cat([win[None].expand(B, -1, -1), sel], dim=-1).to(torch.int32).contiguous()
    return q, kv, sink, idx, HEAD_DIM ** -0.5


def prepare(case, seed):
    kind = case["kind"]
    if kind == "moe":
        x, ids = _token_inputs(case, seed)
        return kind, _moe_layer(_moe_tensors(seed, 10, case["route"]), case["T"]), x, ids
    if kind == "stage":
        blocks = []
        for b in range(case["blocks"]):
            p = _attn_side(seed, 20 + b)
            moe = _moe_layer(_moe_tensors(seed, 10 + b, "bias"), case["T"])
            blocks.append(StageBlock(p["attn_norm"], p["q_norm"], p["ffn_norm"],
                                     kernels.PackedFp8Pair(*p["wq_a"], *p["wkv"]),
                                     kernels.PackedFp8Pair(*p["wq_b"], *p["idx_wq_b"]),
                                     kernels.PackedFp8Linear(*p["wo_b"]), moe))
        stage = DecodeStage(blocks, case["T"], EPS)
        stage.capture()
        return kind, stage, _token_inputs(case, seed)[0]
    if kind == "proj":
        p, g = _attn_side(seed, 20), _gen(seed, 4)
        x, b = _rows(g, case["M"], D), _rows(g, case["M"], D)
        return (kind, x, b, p["attn_norm"], p["q_norm"], kernels.PackedFp8Pair(*p["wq_a"], *p["wkv"]),
                kernels.PackedFp8Pair(*p["wq_b"], *p["idx_wq_b"]))
    if kind == "attn":
        return (kind,) + _attn_inputs(case, seed)
    x, w, s = _gemm_inputs(case, seed)
    if kind == "linear":
        return kind, kernels.PackedFp8Linear(w, s, "ue8m0" if case["ue8m0"] else None), x
    a, a_s = _quant(x, case.get("ue8m0", True), case.get("ue8m0", True))
    return kind, a, a_s, w, s


def run(state):
    kind, args = state[0], state[1:]
    if kind == "moe":
        layer, x, ids = args
        return layer.forward(x, ids)
    if kind == "stage":
        stage, x = args
        return [stage.replay(x), stage.q, stage.kv]
    if kind == "proj":
        x, b, attn_norm, q_norm, qa_kv, q_idx = args
        h, q, s = kernels.add_rms_norm_quant(x, b, attn_norm, EPS)
        qa, kv = qa_kv.gemm(q, s)
        qq, qs = kernels.rms_norm_quant(qa, q_norm, EPS)
        return [h, kv, *q_idx.gemm(qq, qs)]
    if kind == "linear":
        return args[0](args[1])
    if kind == "fp8":
        return kernels.fp8_gemm(*args)
    if kind == "fp4":
        return kernels.fp4_gemm(*args)
    if kind == "grouped":
        return kernels.grouped_fp4_gemm(*args)
    return kernels.sparse_attn(*args)


# ------------------------------------------------------------------ work ------

def _distinct_experts(T, route):
    """Expected number of experts that T tokens select."""
    p = [TOPK / E] * E
    if route == "zipf":
        r = [(i + 1) ** -1.1 for i in range(E)]
        p = [min(1.0, TOPK * v / sum(r)) for v in r]
    return sum(1.0 - (1.0 - q) ** T for q in p)


def _moe_work(T, route):
    expert = 3 * I * D // 2 + 3 * I * D // 32
    bank = _distinct_experts(T, route) * expert + 3 * I * D + E * D * 2
    return bank + 4 * T * D, 2.0 * T * (3 * I * D * (TOPK + 1) + E * D)


def work(case):
    kind = case["kind"]
    if kind == "moe":
        b, f = _moe_work(case["T"], case["route"])
    elif kind in ("stage", "proj"):
        M = case["T"] if kind == "stage" else case["M"]
        w = (Q_LORA + HEAD_DIM) * D + (Q_WIDTH + IDX_WIDTH) * Q_LORA
        out = HEAD_DIM + Q_WIDTH + IDX_WIDTH
        if kind == "proj":
            b, f = w + 2 * M * (3 * D + out), 2.0 * M * w
        else:
            w += D * IDX_WIDTH
            mb, mf = _moe_work(M, "bias")
            b, f = case["blocks"] * (w + mb + 2 * M * (Q_WIDTH + HEAD_DIM)), case["blocks"] * (2.0 * M * w + mf)
    elif kind == "attn":
        B, S, H, start = case["B"], case["S"], case["H"], case["start"]
        rows = sum(min(WINDOW, start + s + 1) + min(SELECTED, (start + s + 1) // RATIO) for s in range(S))
        n = min(WINDOW - 1, start) + S + (start + S) // RATIO
        read = min(n, rows)  # a decoded position reads its own rows, a prompt every row
        idx = min(WINDOW, start + S) + min(SELECTED, (start + S) // RATIO)
        b = 2.0 * B * (2 * S * H * HEAD_DIM + read * HEAD_DIM) + 4.0 * B * S * idx
        f = 4.0 * B * rows * H * HEAD_DIM
    else:
        n, k = case["N"], case["K"]
        m = case["G"] if kind == "grouped" else case["M"]
        wb = n * k if kind in ("linear", "fp8") else n * k // 2 + n * k // 32
        b = wb * (m if kind == "grouped" else 1) + m * k * (2 if kind == "linear" else 1) + 2 * m * n
        f = 2.0 * m * n * k
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """Four times the distance from fp64 (exact) that the layers show: 1.7e-3 is the bf16
    rounding of an output, 2.1e-3 to 2.7e-3 with an intermediate quantised to e4m3, where
    the last bit of a bf16 value moves a code.  A stage chains four such quantisations a
    block, each of which turns a distance d of its input into about sqrt(0.09 d)."""
    kind = case["kind"]
    if kind == "stage":
        return {"rel": 0.03}
    return {"rel": {"moe": 0.009, "proj": 0.008, "attn": 0.008}.get(kind, 0.007)}


# ----------------------------------------------------------------- exact ------

def _deq(q, s):
    """fp64 rows of e4m3 codes with per-128 scales."""
    sd = s.view(torch.uint8).double() if s.dtype == torch.float8_e8m0fnu else None
    sd = torch.exp2(sd - 127.0) if sd is not None else s.double()
    return q.to(torch.float32).double() * sd.repeat_interleave(128, -1)


def _q64(x, ue8m0=True):
    """The fp64 values that act_quant of bf16 rows stands for."""
    return _deq(*_quant(x.to(torch.bfloat16), ue8m0, False))


def _w8(w, s):
    n, k = w.shape
    sd = torch.exp2(s.view(torch.uint8).double() - 127.0) if s.dtype != torch.float32 else s.double()
    return (w.view(torch.float8_e4m3fn).float().double()
            * sd.repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k])


def _w4(w, s):
    """fp64 [N, K] of packed e2m1 [N, K/2] and e8m0 [N, K/32] bytes."""
    t = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device="cuda")
    u = w.view(torch.uint8).int()
    v = torch.stack([t[u & 15], t[u >> 4]], dim=-1).flatten(-2)
    return v * torch.exp2(s.view(torch.uint8).double() - 127.0).repeat_interleave(32, -1)


def _expert64(x, w1, w3, w2, weight):
    """The three linears of an expert, each rounded to the bf16 that it hands on."""
    gate = _bf(x @ w1.t()).double().clamp(max=SWIGLU_LIMIT)
    up = _bf(x @ w3.t()).double().clamp(-SWIGLU_LIMIT, SWIGLU_LIMIT)
    h = torch.nn.functional.silu(gate) * up
    return _bf(_q64(h if weight is None else h * weight) @ w2.t()).double()


def _moe64(t, x, ids):
    """One MoE layer of bf16 rows x in fp64."""
    score = torch.sqrt(torch.nn.functional.softplus(x.double() @ t["gate_w"].double().t()))
    if t["tid2eid"] is not None:
        sel = t["tid2eid"][ids].long()
    else:
        sel = (score + t["gate_bias"].double()).topk(TOPK, dim=-1)[1]
    w = score.gather(1, sel)
    w = w / w.sum(-1, keepdim=True) * ROUTE_SCALE
    xq = _q64(x)
    y = _expert64(xq, _w8(t["sh_w1"], t["sh_w1_s"]), _w8(t["sh_w3"], t["sh_w3_s"]), _w8(t["sh_w2"], t["sh_w2_s"]), None)
    for e in range(E):
        tok, slot = torch.where(sel == e)
        if tok.numel():
            w13, w2 = _w4(t["w13"][e], t["w13_s"][e]), _w4(t["w2"][e], t["w2_s"][e])
            y.index_add_(0, tok, _expert64(xq[tok], w13[:I], w13[I:], w2, w[tok, slot, None]))
    return y


def _norm64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _bf(x):
    return x.to(torch.bfloat16)


def exact(case, seed):
    kind = case["kind"]
    if kind == "moe":
        x, ids = _token_inputs(case, seed)
        return _moe64(_moe_tensors(seed, 10, case["route"]), x, ids)
    if kind == "stage":
        h, e = _token_inputs(case, seed)[0], None
        for b in range(case["blocks"]):
            p = _attn_side(seed, 20 + b)
            h = h if e is None else _bf(h.double() + e.double())
            xq = _q64(_norm64(h, p["attn_norm"]))
            kv = xq @ _w8(*p["wkv"]).t()
            qq = _q64(_norm64(_bf(xq @ _w8(*p["wq_a"]).t()), p["q_norm"]))
            q = qq @ _w8(*p["wq_b"]).t()
            o = _q64(qq @ _w8(*p["idx_wq_b"]).t()) @ _w8(*p["wo_b"]).t()
            h = _bf(_bf(o).double() + h.double())
            e = _bf(_moe64(_moe_tensors(seed, 10 + b, "bias"), _bf(_norm64(h, p["ffn_norm"])), None))
        return [h.double() + e.double(), q, kv]
    if kind == "proj":
        p, g = _attn_side(seed, 20), _gen(seed, 4)
        x, b = _rows(g, case["M"], D), _rows(g, case["M"], D)
        h = _bf(x.double() + b.double())
        xq = _q64(_norm64(h, p["attn_norm"]))
        qq = _q64(_norm64(_bf(xq @ _w8(*p["wq_a"]).t()), p["q_norm"]))
        return [x.double() + b.double(), xq @ _w8(*p["wkv"]).t(), qq @ _w8(*p["wq_b"]).t(),
                qq @ _w8(*p["idx_wq_b"]).t()]
    if kind == "attn":
        q, kv, sink, idx, scale = _attn_inputs(case, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        kv = kv.double()
        for b in range(case["B"]):
            for at in range(0, case["S"], 128):
                ix = idx[b, at:at + 128].long()
                rows = kv[b][ix.clamp(min=0)]                                     # [s, topk, d]
                sc = torch.matmul(q[b, at:at + 128].double(), rows.transpose(1, 2).contiguous()) * scale
                sc = sc.masked_fill((ix < 0)[:, None], -math.inf)
                m = torch.maximum(sc.amax(-1, keepdim=True), sink.double()[None, :, None])
                pr = torch.exp(sc - m)
                den = pr.sum(-1, keepdim=True) + torch.exp(sink.double()[None, :, None] - m)
                out[b, at:at + 128] = torch.matmul(pr / den, rows)
        return out
    x, w, s = _gemm_inputs(case, seed)
    a = _q64(x, case.get("ue8m0", True))
    if kind in ("linear", "fp8"):
        return a @ _w8(w, s).t()
    if kind == "fp4":
        return a @ _w4(w, s).t()
    return torch.stack([a[g] @ _w4(w[g], s[g]).t() for g in range(case["G"])])
