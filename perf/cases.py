"""The calls a program on this framework makes, as cases to time and compare.

Five paths, each through its public entry points:

``moe``       ``MoEBlock.forward``: router, top-k, permutation, MXFP4 gate/up
              and down experts, combine.  Decode (one token, a batch), a
              prompt chunk, a long prefill.
``int4``      ``Context.int4_linear``: group-scaled INT4 weights against bf16
              activations (GPTQ and CT layouts, with and without zero points,
              bias or residual).
``int8_mlp``  a dense feed-forward on INT8-prequantized activations and GPTQ
              INT4 weights: RMSNorm + quantization, gate and up, SiLU product
              + quantization, down with the residual.
``head``      ``Context.fp8_output_projection``: FP8 vocabulary projection
              with the greedy token.
``int4_moe``  the routed block on INT4 (compressed-tensors) experts, node by
              node.

Weights are drawn on the GPU in the compiled package's layouts, with
magnitudes that keep activations of order one, as trained weights do.
"""
from __future__ import annotations

import math

import torch

from nerve_amd.hip import Context
from nerve_amd.moe import ExpertBank, Int4CtExpertBank, MoEBlock, int4_ct_spec, topk_spec

DEV = "cuda:0"
LIMIT = 7.0
EPS = 1e-5

# (experts, top_k, hidden, intermediate) of the MXFP4 blocks
MOE_SHAPES = [(32, 4, 2880, 2880), (128, 4, 2880, 2880), (64, 6, 2048, 1536)]
# (K, N) of the INT4 linears; the last ones are not multiples of the column tiles
INT4_SHAPES = [(4096, 14336), (14336, 4096), (4096, 4096), (2816, 5136), (4096, 11024)]
# (hidden, intermediate, group) of the INT8-activation feed-forwards
INT8_SHAPES = [(4096, 14336, 128), (4096, 11008, 128), (2880, 5760, 64), (2048, 6144, 32)]
# (K, N) of the listed heads, and the drawn ones' K; their N is any size from
# 32000 up to the listed head's weight bytes
HEAD = (2880, 201088)
HEAD_K = [2048, 2880, 4096]
# (experts, top_k, hidden, intermediate, group) of the INT4 experts
INT4_MOE_SHAPES = [(256, 10, 3072, 1024, 32), (64, 6, 2048, 1408, 32)]


def _moe(tokens, shape=0, skew=0.0):
    E, k, H, I = MOE_SHAPES[shape]
    return dict(path="moe", tokens=tokens, experts=E, top_k=k, hidden=H, inter=I, skew=skew)


def _int4(rows, K, N, layout="gptq", group=128, zeros=False, op="linear", scale="f16"):
    return dict(path="int4", rows=rows, K=K, N=N, layout=layout, group=group, zeros=zeros, op=op, scale=scale)


def _int8(rows, shape=0, scale="f16"):
    H, I, G = INT8_SHAPES[shape]
    return dict(path="int8_mlp", rows=rows, hidden=H, inter=I, group=G, scale=scale)


def _head(rows, logits="f32", block_rows=1, K=HEAD[0], N=HEAD[1]):
    return dict(path="head", rows=rows, K=K, N=N, logits=logits, block_rows=block_rows)


def _int4_moe(tokens, shape=0):
    E, k, H, I, G = INT4_MOE_SHAPES[shape]
    return dict(path="int4_moe", tokens=tokens, experts=E, top_k=k, hidden=H, inter=I, group=G)


def listed():
    return [
        # One user's next token through one MoE layer.
        dict(_moe(1), name="moe_decode_1"),
        # A decode batch: the benchmark's default layer.
        dict(_moe(16), name="moe_decode_16"),
        # A short prompt, or one chunk of a longer one, of odd length.
        dict(_moe(150), name="moe_chunk_150"),
        # A long prefill over many experts whose popularity is skewed.
        dict(_moe(2048, shape=1, skew=1.1), name="moe_prefill_2048"),
        # One token through an asymmetric GPTQ up projection.
        dict(_int4(1, 4096, 14336, zeros=True), name="int4_gptq_decode_1"),
        # A prompt of odd length through a CT down projection that adds the residual.
        dict(_int4(301, 14336, 4096, layout="ct", op="linear_residual", scale="bf16"), name="int4_ct_prefill_301"),
        # One token through a whole INT8-activation feed-forward.
        dict(_int8(1), name="int8_mlp_decode_1"),
        # A decode batch, or a speculative window, through the same.
        dict(_int8(48), name="int8_mlp_batch_48"),
        # The next token's logits and the greedy id.
        dict(_head(1), name="head_decode_1"),
        # The same for a decode batch.
        dict(_head(64), name="head_batch_64"),
        # Scoring a prompt: bf16 logits at every position.
        dict(_head(512, logits="bf16"), name="head_score_512"),
        # A decode batch through an INT4 expert layer.
        dict(_int4_moe(16), name="int4_moe_decode_16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo - 0.49 if lo > 1 else 0.6), math.log(hi + 0.49))))))


def draw(rng):
    path = rng.choice(["moe", "moe", "int4", "int4", "int8_mlp", "head", "int4_moe"])
    if path == "moe":
        return _moe(_log_int(rng, 1, 2048), rng.randrange(len(MOE_SHAPES)), rng.choice([0.0, 0.6, 1.1]))
    if path == "int4":
        K, N = rng.choice(INT4_SHAPES)
        layout = rng.choice(["gptq", "gptq", "ct"])
        group = 128 if layout == "ct" else rng.choice([32, 64, 128, 128])
        return _int4(_log_int(rng, 1, 512), K, N, layout, group, layout == "gptq" and rng.random() < 0.5,
                     rng.choice(["linear", "linear_bias", "linear_residual"]), rng.choice(["f16", "bf16"]))
    if path == "int8_mlp":
        return _int8(_log_int(rng, 1, 256), rng.randrange(len(INT8_SHAPES)), rng.choice(["f16", "bf16"]))
    if path == "head":
        K = rng.choice(HEAD_K)
        return _head(_log_int(rng, 1, 512), rng.choice(["f32", "bf16"]), rng.choice([1, 1, 128]), K,
                     rng.randint(32000, min(HEAD[1], HEAD[0] * HEAD[1] // K)))
    return _int4_moe(_log_int(rng, 1, 256), rng.randrange(len(INT4_MOE_SHAPES)))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

_context = None


def _ctx():
    """The program's one handle on the device."""
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _bytes(g, *shape, lo=0, hi=256):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.uint8)


def _words(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31, shape, generator=g, device=DEV, dtype=torch.int64).to(torch.int32)


def _normal(g, *shape, std=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _bits(t):
    return t.view(torch.int16)


def _group_scales(g, kind, contraction, *shape):
    """Scales that give a row of uniform 4-bit codes unit gain."""
    s = (torch.rand(shape, generator=g, device=DEV) + 0.5) / (4.6 * math.sqrt(contraction))
    return s.to(torch.bfloat16 if kind == "bf16" else torch.float16)


def _router(g, E, H, tokens, skew):
    """Router rows and tokens: channel 0 carries a constant, through which the
    router ranks its experts' popularity as rank^-skew."""
    w = torch.randn(E, H, generator=g, device=DEV) * 0.02
    x = torch.randn(tokens, H, generator=g, device=DEV)
    if skew:
        rank = torch.randperm(E, generator=g, device=DEV).float() + 1
        x[:, 0] = 4.0
        w[:, 0] = -skew * rank.log() / 4.0
    return w.to(torch.bfloat16), x.to(torch.bfloat16)


def _moe_inputs(case, seed):
    g = _gen(seed)
    E, H, I = case["experts"], case["hidden"], case["inter"]
    router, x = _router(g, E, H, case["tokens"], case["skew"])
    bank = dict(gate_w=_bytes(g, E, I, H // 2), gate_s=_bytes(g, E, I, H // 32, lo=118, hi=122),
                up_w=_bytes(g, E, I, H // 2), up_s=_bytes(g, E, I, H // 32, lo=118, hi=122),
                down_w=_bytes(g, E, H, I // 2), down_s=_bytes(g, E, H, I // 32, lo=118, hi=122))
    return dict(router=router, x=x, bank=bank)


def _int4_weights(g, K, N, layout, group, scale, zeros):
    if layout == "gptq":
        return dict(w=_words(g, K // 8, N), s=_group_scales(g, scale, K, K // group, N),
                    z=_words(g, K // group, N // 8) if zeros else None)
    return dict(w=_words(g, N, K // 8), s=_group_scales(g, scale, K, N, K // group), z=None)


def _int4_inputs(case, seed):
    g = _gen(seed)
    M, K, N = case["rows"], case["K"], case["N"]
    d = _int4_weights(g, K, N, case["layout"], case["group"], case["scale"], case["zeros"])
    d["x"] = _normal(g, M, K)
    d["aux"] = {"linear": None, "linear_bias": _normal(g, N), "linear_residual": _normal(g, M, N)}[case["op"]]
    return d


def _int8_inputs(case, seed):
    g = _gen(seed)
    M, H, I, G, sc = case["rows"], case["hidden"], case["inter"], case["group"], case["scale"]
    return dict(x=_normal(g, M, H), norm=(1 + 0.1 * torch.randn(H, generator=g, device=DEV)).to(torch.bfloat16),
                gate=_int4_weights(g, H, I, "gptq", G, sc, False), up=_int4_weights(g, H, I, "gptq", G, sc, False),
                down=_int4_weights(g, I, H, "gptq", G, sc, False))


def _head_inputs(case, seed):
    g = _gen(seed)
    M, K, N, br = case["rows"], case["K"], case["N"], case["block_rows"]
    nblk = (K + 127) // 128
    W = torch.empty(N, K, dtype=torch.uint8, device=DEV)
    rows = (N + br - 1) // br
    scale = torch.empty(rows, nblk, dtype=torch.bfloat16, device=DEV)
    step = 16384
    for r in range(0, N, step):
        wf = torch.randn(min(step, N - r), K, generator=g, device=DEV) * 0.02
        n = wf.shape[0]
        if br == 1:
            s = (wf.abs().amax(1, keepdim=True) / 448.0).to(torch.bfloat16)
            scale[r:r + n] = s
            per = s.float()
        else:
            pad = torch.nn.functional.pad(wf.abs(), (0, nblk * 128 - K, 0, -n % br))
            s = (pad.view(-1, br, nblk, 128).amax((1, 3)) / 448.0).to(torch.bfloat16)
            scale[r // br:r // br + s.shape[0]] = s
            per = s.float().repeat_interleave(br, 0)[:n].repeat_interleave(128, 1)[:, :K]
        W[r:r + n] = (wf / per).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    return dict(W=W, scale=scale, x=_normal(g, M, K))


def _int4_moe_inputs(case, seed):
    g = _gen(seed)
    E, H, I, G = case["experts"], case["hidden"], case["inter"], case["group"]
    router, x = _router(g, E, H, case["tokens"], 0.0)
    return dict(router=router, x=x, gate_up_w=_words(g, E, 2 * I, H // 8),
                gate_up_s=_group_scales(g, "bf16", H, E, 2 * I, H // G), down_w=_words(g, E, H, I // 8),
                down_s=_group_scales(g, "bf16", I, E, H, I // G))


# ---------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------

def _zeros(*shape, dtype=torch.int16):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def prepare(case, seed):
    c, path = _ctx(), case["path"]
    if path == "moe":
        d = _moe_inputs(case, seed)
        block = MoEBlock(c, _bits(d["router"]), ExpertBank(**d["bank"]), case["top_k"], limit=LIMIT)
        return dict(path=path, block=block, x=_bits(d["x"]))
    if path == "int4":
        d = _int4_inputs(case, seed)
        M, K, N = case["rows"], case["K"], case["N"]
        spec = (f"{case['op']}_batch16_int4_{case['layout']}_s{case['scale']}_g{case['group']}_{K}x{N}.comp")
        return dict(path=path, ctx=c, spec=spec, x=_bits(d["x"]), w=d["w"], s=_bits(d["s"]), z=d["z"],
                    aux=None if d["aux"] is None else _bits(d["aux"]), rows=M, y=_zeros(M, N))
    if path == "int8_mlp":
        d = _int8_inputs(case, seed)
        M, H, I, G, sc = case["rows"], case["hidden"], case["inter"], case["group"], case["scale"]
        lin = "linear{}_prequant_pairpacked_batch16_int4_gptq_s{}_g{}_{}x{}.comp".format
        s = dict(path=path, ctx=c, rows=M, x=_bits(d["x"]), norm=_bits(d["norm"]),
                 norm_spec=f"rms_norm_quantize_batch16_int8_pairpacked_b32_h{H}_eps{EPS:.9g}_offset0.comp",
                 up_spec=lin("", sc, G, H, I), down_spec=lin("_residual", sc, G, I, H),
                 act_spec=f"silu_multiply_quantize_batch16_int8_pairpacked_b32_h{I}.comp")
        for n in ("gate", "up", "down"):
            s[n] = (d[n]["w"], _bits(d[n]["s"]))
        s.update(normed=_zeros(M, H), hq=_zeros(M, H, dtype=torch.int8), hs=_zeros(M, H // 32, dtype=torch.float32),
                 hsum=_zeros(M, H // 32, dtype=torch.int32), g=_zeros(M, I), u=_zeros(M, I), act=_zeros(M, I),
                 iq=_zeros(M, I, dtype=torch.int8), isc=_zeros(M, I // 32, dtype=torch.float32),
                 isum=_zeros(M, I // 32, dtype=torch.int32), y=_zeros(M, H))
        return s
    if path == "head":
        d = _head_inputs(case, seed)
        M, K, N = case["rows"], case["K"], case["N"]
        spec = f"tied_output_projection_batch16_fp8_e4m3_b{case['block_rows']}x128_{N}x{K}_scale1_to_f32.comp"
        bf = case["logits"] == "bf16"
        return dict(path=path, ctx=c, spec=spec, x=_bits(d["x"]), W=d["W"], scale=_bits(d["scale"]), rows=M,
                    f32=None if bf else _zeros(M, N, dtype=torch.float32), bf16=_zeros(M, N) if bf else None,
                    token=_zeros(M, dtype=torch.int32))
    d = _int4_moe_inputs(case, seed)
    B, E, k, H, I, G = (case[n] for n in ("tokens", "experts", "top_k", "hidden", "inter", "group"))
    bank = Int4CtExpertBank(d["gate_up_w"], _bits(d["gate_up_s"]), d["down_w"], _bits(d["down_s"]))
    control = torch.tensor([B, 0, 0, 0, 0, 0, 0, 0], dtype=torch.int32, device=DEV)
    return dict(path=path, ctx=c, B=B, E=E, H=H, k=k, x=_bits(d["x"]), router=_bits(d["router"]), bank=bank,
                topk=topk_spec(E, k), gate_up=int4_ct_spec("gate_up", H, I, E, k, G),
                down=int4_ct_spec("down", H, I, E, k, G), logits=_zeros(B, E), routes=_zeros(B, k, dtype=torch.int32),
                frames=_zeros(B * (k * I // 2 + k), dtype=torch.int32), control=control, outputs=_zeros(B, k, H),
                y=_zeros(B, H))


def run(state):
    s = state
    path = s["path"]
    if path == "moe":
        return s["block"].forward(s["x"]).view(torch.bfloat16)
    c = s["ctx"]
    if path == "int4":
        c.int4_linear(s["spec"], s["x"], s["w"], s["s"], s["z"], s["aux"], s["y"], s["rows"])
        return s["y"].view(torch.bfloat16)
    if path == "int8_mlp":
        M = s["rows"]
        c.rms_norm_quantize_int8_pairpacked(s["norm_spec"], s["x"], s["norm"], s["normed"], s["hq"], s["hs"],
                                            s["hsum"], M)
        c.int4_linear_pairpacked(s["up_spec"], s["hq"], s["hs"], s["hsum"], *s["gate"], None, s["g"], M)
        c.int4_linear_pairpacked(s["up_spec"], s["hq"], s["hs"], s["hsum"], *s["up"], None, s["u"], M)
        c.silu_multiply_quantize_int8_pairpacked(s["act_spec"], s["g"], s["u"], s["act"], s["iq"], s["isc"],
                                                 s["isum"], M)
        c.int4_linear_pairpacked(s["down_spec"], s["iq"], s["isc"], s["isum"], *s["down"], s["x"], s["y"], M)
        return s["act"].view(torch.bfloat16), s["y"].view(torch.bfloat16)
    if path == "head":
        c.fp8_output_projection(s["spec"], s["x"], s["W"], s["scale"], s["f32"], s["bf16"], s["token"], s["rows"])
        return (s["bf16"].view(torch.bfloat16) if s["f32"] is None else s["f32"]), s["token"]
    B, bank = s["B"], s["bank"]
    c.router_linear_bf16(s["x"], s["router"], s["logits"], B, s["H"], s["E"])
    c.moe_router_topk(s["topk"], s["logits"], None, s["routes"], None, B)
    c.moe_route_compact(s["gate_up"], s["routes"], s["frames"], s["control"], B)
    c.int4_moe_gate_up(s["gate_up"], s["x"], s["routes"], s["frames"], bank.addresses, bank.gate_slots, s["control"], B)
    c.moe_route_compact(s["down"], s["routes"], None, s["control"], B)
    c.int4_moe_down(s["down"], s["frames"], s["routes"], s["outputs"], bank.addresses, bank.down_slots, s["control"], B)
    c.moe_reduce(s["outputs"], s["y"], B, s["H"], s["k"])
    return s["y"].view(torch.bfloat16)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _distinct(E, k, tokens, skew):
    """Experts that a batch is expected to reach: k of E per token, with
    popularity rank^-skew times a log-normal of the router's random part."""
    if not skew:
        return E * (1 - (1 - k / E) ** tokens)
    p = [(r + 1.0) ** -skew for r in range(E)]
    total = sum(p)
    return sum(1 - (1 - min(1.0, k * q / total)) ** tokens for q in p)


def work(case):
    path = case["path"]
    if path in ("moe", "int4_moe"):
        B, E, k, H, I = (case[n] for n in ("tokens", "experts", "top_k", "hidden", "inter"))
        per = 3 * H * I // 2
        per += 3 * H * I // 32 if path == "moe" else 3 * H * I // case["group"] * 2
        used = _distinct(E, k, B, case.get("skew", 0.0))
        return dict(bytes=int(used * per) + E * H * 2 + 2 * B * H * 2, flops=2 * 3 * B * k * H * I + 2 * B * H * E)
    if path == "int4":
        M, K, N, G = case["rows"], case["K"], case["N"], case["group"]
        aux = {"linear": 0, "linear_bias": N * 2, "linear_residual": M * N * 2}[case["op"]]
        z = K // G * N // 2 if case["zeros"] else 0
        return dict(bytes=K * N // 2 + K // G * N * 2 + z + 2 * M * (K + N) + aux, flops=2 * M * K * N)
    if path == "int8_mlp":
        M, H, I, G = case["rows"], case["hidden"], case["inter"], case["group"]
        return dict(bytes=3 * (H * I // 2 + H * I // G * 2) + 4 * M * H + 2 * H + 2 * M * I, flops=2 * 3 * M * H * I)
    M, K, N = case["rows"], case["K"], case["N"]
    grid = (N + case["block_rows"] - 1) // case["block_rows"] * ((K + 127) // 128) * 2
    return dict(bytes=N * K + grid + M * K * 2 + M * N * (4 if case["logits"] == "f32" else 2) + 4 * M,
                flops=2 * M * K * N)


def tolerance(case):
    """About four times what the same call shows with its sums in another
    order (the contraction's blocks permuted), or with the matrix unit's own
    error (1.4e-5 against double for e4m3 products) where that is larger.  A
    bf16 result that lands on the other side of a rounding edge moves by one
    place (2^-7 of its value at most); the blocks and the feed-forward also
    requantize an intermediate, where one place can move an e4m3 or int8 code."""
    path = case["path"]
    if path == "head":
        if case["logits"] == "f32":
            return dict(rel=6e-5, max=6e-4, differ=0.01)
        return dict(rel=5e-4, max=0.03, differ=0.01)
    if path == "int4":
        return dict(rel=5e-4, max=0.03)
    return dict(rel=2e-3, max=0.05)


# ---------------------------------------------------------------------------
# The same in 64 bits: the operands as the formats hold them, sums in double
# ---------------------------------------------------------------------------

def _nibbles(w):
    """Codes of packed words [..., n] (low nibble first), [..., 8 n]."""
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int64)
    return ((w.to(torch.int64)[..., None] >> sh) & 15).flatten(-2)


def _e2m1(w, s):
    """MXFP4 rows [R, K/2] with e8m0 scales [R, K/32] as double [R, K]."""
    table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64,
                         device=w.device)
    v = table[torch.stack([w & 15, w >> 4], -1).flatten(-2).long()]
    return v * torch.exp2(s.double() - 127).repeat_interleave(32, -1)


def _e4m3_blocks(x, pow2):
    """bf16 rows quantized per 128 columns to e4m3, as double.  (A division by
    a Python number would multiply by its reciprocal; the scale is a quotient.)"""
    K = x.shape[-1]
    xb = torch.nn.functional.pad(x.float(), (0, -K % 128)).unflatten(-1, (-1, 128))
    amax = xb.abs().amax(-1, keepdim=True)
    if pow2:
        mant, ex = torch.frexp(amax.clamp(min=1e-4) / torch.full_like(amax, 448))
        s = torch.ldexp(torch.ones_like(mant), torch.where(mant == 0.5, ex - 1, ex))
    else:
        s = torch.where(amax > 0, amax / torch.full_like(amax, 448), torch.ones_like(amax))
    q = (xb / s).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * s.double()).flatten(-2)[..., :K]


def _int8_blocks(x):
    xb = x.float().unflatten(-1, (-1, 32))
    amax = xb.abs().amax(-1, keepdim=True)
    s = torch.where(amax > 0, amax / torch.full_like(amax, 127), torch.ones_like(amax))
    return ((xb / s).clamp(-127, 127).round().double() * s.double()).flatten(-2)


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _top(logits, k):
    """The k largest (the lower id first among equals), with softmax weights over them, as bf16 words hold them."""
    v, i = torch.sort(logits, dim=-1, descending=True, stable=True)
    return i[:, :k], _bf16(torch.softmax(v[:, :k], -1))


def _experts(out, ids, wts, E, contract):
    for e in range(E):
        b, r = (ids == e).nonzero(as_tuple=True)
        if b.numel():
            out[b] += contract(e, b) * wts[b, r][:, None]
    return out


def _int4_dense(d, layout, group):
    """INT4 weights as double [K, N]."""
    if layout == "ct":
        q = _nibbles(d["w"]).double() - 8
        return (q * d["s"].double().repeat_interleave(group, -1)).T
    q = _nibbles(d["w"].T).T.double()
    z = 8.0 if d["z"] is None else _nibbles(d["z"]).double().repeat_interleave(group, 0)
    return (q - z) * d["s"].double().repeat_interleave(group, 0)


def exact(case, seed):
    path = case["path"]
    if path == "moe":
        d = _moe_inputs(case, seed)
        b = d["bank"]
        x = _e4m3_blocks(d["x"], True)
        ids, wts = _top(_bf16(d["x"].double() @ d["router"].double().T), case["top_k"])

        def contract(e, rows):
            g = _bf16(x[rows] @ _e2m1(b["gate_w"][e], b["gate_s"][e]).T).clamp(max=LIMIT)
            u = _bf16(x[rows] @ _e2m1(b["up_w"][e], b["up_s"][e]).T).clamp(-LIMIT, LIMIT)
            h = (g * torch.sigmoid(g) * u).to(torch.bfloat16)
            return _e4m3_blocks(h, True) @ _e2m1(b["down_w"][e], b["down_s"][e]).T

        return _experts(torch.zeros_like(x), ids, wts, case["experts"], contract)
    if path == "int4":
        d = _int4_inputs(case, seed)
        y = d["x"].double() @ _int4_dense(d, case["layout"], case["group"])
        return y if d["aux"] is None else y + d["aux"].double()
    if path == "int8_mlp":
        d = _int8_inputs(case, seed)
        G = case["group"]
        x = d["x"].double()
        n = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * d["norm"].double()).to(torch.bfloat16)
        q = _int8_blocks(n)
        g, u = (_bf16(q @ _int4_dense(d[w], "gptq", G)) for w in ("gate", "up"))
        act = _bf16(g * torch.sigmoid(g)) * u
        return act, _int8_blocks(act.to(torch.bfloat16)) @ _int4_dense(d["down"], "gptq", G) + x
    if path == "head":
        d = _head_inputs(case, seed)
        K, N, br = case["K"], case["N"], case["block_rows"]
        x = _e4m3_blocks(d["x"], False)
        y = torch.empty(case["rows"], N, dtype=torch.float64, device=DEV)
        step = 16384
        for r in range(0, N, step):
            w = d["W"][r:r + step].view(torch.float8_e4m3fn).double()
            s = d["scale"].double()[r // br:(r + step + br - 1) // br].repeat_interleave(br, 0)[:w.shape[0]]
            y[:, r:r + step] = x @ (w * s.repeat_interleave(128, 1)[:, :K]).T
        return y, None
    d = _int4_moe_inputs(case, seed)
    I, G = case["inter"], case["group"]
    x = d["x"].double()
    ids, wts = _top(_bf16(x @ d["router"].double().T), case["top_k"])

    def dense(n, e):
        return _int4_dense(dict(w=d[n + "_w"][e], s=d[n + "_s"][e]), "ct", G)

    def project(e, rows):
        gu = _bf16(x[rows] @ dense("gate_up", e))
        g, u = gu[:, :I], gu[:, I:]
        return _bf16(_bf16(g * torch.sigmoid(g)) * u) @ dense("down", e)

    return _experts(torch.zeros_like(x), ids, wts, case["experts"], project)
