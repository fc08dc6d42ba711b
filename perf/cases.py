"""The work that a program using larynx_amd has it do, as measurable cases.

Whole calls: FlowDecoder.infer (speech tokens -> mel), DiTEstimator.forward, the Qwen2
LM's prefill and token-by-token decode.  Single layers: attention, a projection and the
normalisations through larynx_amd.ops.  Geometry is the models' own (DiTConfig, FlowConfig
and Qwen2Config defaults); handles are built once for the longest input they serve, as a
program keeps them, and lengths range from the shortest call to the longest supported.

exact() restates each path in plain float64 torch.  Angles of the rotary embeddings, the
timestep sinusoid's arguments and the Euler schedule are fp32 by definition of the models
and are formed in fp32 there too.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from larynx_amd import ops
from larynx_amd.flow import (DiTConfig, DiTEstimator, FlowConfig, FlowDecoder, cfm_t_span,
                             dit_param_shapes, flow_frontend_param_shapes)
from larynx_amd.llm import Qwen2Config, Qwen2LM, qwen2_param_shapes

DEV = "cuda"
DIT, FLOW, LM = DiTConfig(), FlowConfig(), Qwen2Config()
MAX_TOKENS = 1500  # 60 s of speech at 25 tokens/s: a decoder serving any utterance up to that
MAX_FRAMES = FLOW.token_mel_ratio * MAX_TOKENS
MAX_CTX = 4096     # the LM's longest context

# (N, K, epilogue) of the estimator's projections
PROJ = {
    "qkv": (3 * DIT.dim, DIT.dim, "rope"),
    "out": (DIT.dim, DIT.dim, "none"),
    "ff0": (DIT.ff_inner, DIT.dim, "gelu"),
    "ff2": (DIT.dim, DIT.ff_inner, "none"),
}


def listed():
    return [
        # one short sentence: 1 s of speech after half a second of prompt voice
        dict(name="infer_1s", kind="infer", n_prompt=12, n_tokens=25),
        # the usual utterance: 8 s after a 2 s prompt (the benchmark's 10 s, T = 500)
        dict(name="infer_10s", kind="infer", n_prompt=50, n_tokens=200),
        # the longest utterance a decoder is built for (T = 3000)
        dict(name="infer_60s", kind="infer", n_prompt=300, n_tokens=1200),
        # one estimator evaluation of a caller with its own solver, at fp32-GEMM accuracy
        dict(name="dit_forward_six", kind="dit", B=2, T=211, products=6),
        # LM prompt without a reference voice: a few words
        dict(name="prefill_37", kind="prefill", L=37),
        # LM prompt with a reference voice (the benchmark's size)
        dict(name="prefill_256", kind="prefill", L=256),
        # LM prompt with a long reference voice and a long text
        dict(name="prefill_1531", kind="prefill", L=1531),
        # speech tokens one by one, soon after a short prompt
        dict(name="decode_at_30", kind="decode", cache=30, steps=8),
        # the same late in a long utterance
        dict(name="decode_at_2000", kind="decode", cache=2000, steps=8),
        # the estimator's attention layer at an odd length
        dict(name="attention_777", kind="attention", form="dit", B=2, T=777, products=3),
        # the estimator's q|k|v projection with bias and rotary, at an odd length
        dict(name="linear_qkv_333", kind="linear", proj="qkv", B=2, T=333, products=3),
        # the smallest call: the modulated LayerNorm over a very short utterance
        dict(name="ada_ln_24", kind="norm", form="ada_ln", B=2, T=24),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["infer", "dit", "prefill", "decode", "attention", "linear", "norm"])
    if kind == "infer":
        total = _log_int(rng, 12, MAX_TOKENS)
        n_prompt = max(1, min(total - 1, int(total * rng.uniform(0.1, 0.4))))
        return dict(kind=kind, n_prompt=n_prompt, n_tokens=total - n_prompt)
    if kind == "dit":
        B = rng.choice([1, 2, 2, 4])
        return dict(kind=kind, B=B, T=_log_int(rng, 24, 2 * MAX_FRAMES // max(B, 2)),
                    products=rng.choice([3, 3, 6]))
    if kind == "prefill":
        return dict(kind=kind, L=_log_int(rng, 8, 2048))
    if kind == "decode":
        return dict(kind=kind, cache=_log_int(rng, 1, 4000), steps=rng.randint(4, 16))
    if kind == "attention":
        if rng.random() < 0.6:
            return dict(kind=kind, form="dit", B=2, T=_log_int(rng, 24, MAX_FRAMES),
                        products=rng.choice([3, 3, 6]))
        return dict(kind=kind, form="lm", B=1, T=_log_int(rng, 8, 2048), products=6)
    if kind == "linear":
        return dict(kind=kind, proj=rng.choice(sorted(PROJ)), B=2, T=_log_int(rng, 24, MAX_FRAMES),
                    products=rng.choice([3, 3, 6]))
    if rng.random() < 0.5:
        return dict(kind="norm", form="ada_ln", B=2, T=_log_int(rng, 24, MAX_FRAMES))
    return dict(kind="norm", form="rms_norm", B=1, T=_log_int(rng, 1, 2048))


# ---- inputs ---------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g).mul_(std)


def _params(shapes, g):
    """Weights at a trained network's scale: matrices keep the variance of what they read
    (std 1 / sqrt(fan in)), norm gains near one, small biases, 0.02 embeddings."""
    out = {}
    for name, shape in shapes:
        if name.endswith("bias"):
            out[name] = _randn(g, *shape, std=0.02)
        elif len(shape) == 1:
            out[name] = _randn(g, *shape, std=0.1).add_(1.0)
        elif "embed" in name and "proj" not in name and "time" not in name and len(shape) == 2 \
                and "affine" not in name:
            out[name] = _randn(g, *shape, std=0.02 if shape[1] == LM.hidden else 0.5)
        else:
            fan = 1
            for n in shape[1:]:
                fan *= n
            out[name] = _randn(g, *shape, std=fan ** -0.5)
    return out


def _infer_sizes(case):
    total = case["n_prompt"] + case["n_tokens"]
    return FLOW.token_mel_ratio * total, FLOW.token_mel_ratio * case["n_prompt"]


def _draw_infer(case, seed):
    g = _gen(seed)
    MT, L1 = _infer_sizes(case)
    ids = torch.randint(0, FLOW.vocab, (case["n_prompt"] + case["n_tokens"],), device=DEV,
                        generator=g).cpu().numpy().astype(np.int32)
    return dict(front=_params(flow_frontend_param_shapes(DIT, FLOW), g),
                dit=_params(dit_param_shapes(DIT), g),
                prompt=ids[:case["n_prompt"]].copy(), tokens=ids[case["n_prompt"]:].copy(),
                feat=_randn(g, L1, DIT.mel_dim), spk=_randn(g, FLOW.spk_in),
                z=_randn(g, DIT.mel_dim, MT))


def _draw_dit(case, seed):
    g = _gen(seed)
    B, T = case["B"], case["T"]
    return dict(dit=_params(dit_param_shapes(DIT), g), x=_randn(g, B, DIT.mel_dim, T),
                mu=_randn(g, B, DIT.mel_dim, T), cond=_randn(g, B, DIT.mel_dim, T),
                spks=_randn(g, B, DIT.mel_dim, std=0.3),
                t=torch.rand(B, device=DEV, generator=g))


def _draw_prefill(case, seed):
    g = _gen(seed)
    L = case["L"]
    n_text = max(1, (L - 2) * 5 // 8)
    return dict(lm=_params(qwen2_param_shapes(LM), g),
                text=torch.randint(0, LM.text_vocab, (n_text,), device=DEV, generator=g).tolist(),
                speech=torch.randint(0, 6561, (L - 2 - n_text,), device=DEV, generator=g).tolist())


def _draw_decode(case, seed):
    g = _gen(seed)
    KV = LM.n_kv_heads * LM.head_dim
    c = case["cache"]
    return dict(lm=_params(qwen2_param_shapes(LM), g),
                k=_randn(g, LM.n_layers, c, KV), v=_randn(g, LM.n_layers, c, KV, std=0.5),
                tokens=torch.randint(0, 6561, (case["steps"],), device=DEV, generator=g).tolist())


def _attn_heads(case):
    return (DIT.heads, DIT.heads) if case["form"] == "dit" else (LM.n_heads, LM.n_kv_heads)


def _draw_attention(case, seed):
    g = _gen(seed)
    nh, nkv = _attn_heads(case)
    B, T, hd = case["B"], case["T"], DIT.head_dim
    # one fused q|k|v buffer, as the projection leaves it
    return dict(qkv=_randn(g, B, T, (nh + 2 * nkv) * hd))


def _draw_linear(case, seed):
    g = _gen(seed)
    N, K, _ = PROJ[case["proj"]]
    return dict(x=_randn(g, case["B"] * case["T"], K), W=_randn(g, N, K, std=K ** -0.5),
                b=_randn(g, N, std=0.02))


def _draw_norm(case, seed):
    g = _gen(seed)
    B, T = case["B"], case["T"]
    if case["form"] == "ada_ln":
        # shift and scale are chunks of one stacked modulation row
        return dict(x=_randn(g, B, T, DIT.dim), emb=_randn(g, B, 6 * DIT.dim, std=0.3))
    return dict(x=_randn(g, T, LM.hidden), w=_randn(g, LM.hidden, std=0.1).add_(1.0))


_DRAW = dict(infer=_draw_infer, dit=_draw_dit, prefill=_draw_prefill, decode=_draw_decode,
             attention=_draw_attention, linear=_draw_linear, norm=_draw_norm)


def prepare(case, seed):
    s = _DRAW[case["kind"]](case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind == "infer":
        s["decoder"] = FlowDecoder(s.pop("front"), s.pop("dit"), DIT, FLOW, MAX_TOKENS)
    elif kind == "dit":
        s["est"] = DiTEstimator(s.pop("dit"), DIT, B=case["B"], max_T=MAX_FRAMES)
        s["est"].set_products(case["products"])
    elif kind == "prefill":
        s["model"] = Qwen2LM(s.pop("lm"), LM, MAX_CTX)
        s["cache"] = [tuple(c[:case["L"]] for c in s["model"].cache_views(i))
                      for i in range(LM.n_layers)]
    elif kind == "decode":
        m = s["model"] = Qwen2LM(s.pop("lm"), LM, MAX_CTX)
        c, n = case["cache"], case["steps"]
        s["rows"] = []
        for i in range(LM.n_layers):
            kc, vc = m.cache_views(i)
            kc[:c].copy_(s["k"][i])
            vc[:c].copy_(s["v"][i])
            s["rows"].append((kc[c:c + n], vc[c:c + n]))
    elif kind == "attention":
        nh, nkv = _attn_heads(case)
        hd = DIT.head_dim
        s["q"], s["k"], s["v"] = s["qkv"].split([nh * hd, nkv * hd, nkv * hd], dim=-1)
    elif kind == "linear":
        N, K, epi = PROJ[case["proj"]]
        s["wf"] = ops.wfrag_pack(s["W"])
        s["epi"] = None
        if epi == "gelu":
            s["epi"] = ops.Epilogue(kind=ops.LX_EPI_GELU_TANH)
        elif epi == "rope":
            s["pos"] = torch.arange(case["T"], device=DEV, dtype=torch.int32)
            e = s["epi"] = ops.Epilogue(kind=ops.LX_EPI_ROPE_PARTIAL)
            e.rows_per_batch, e.pos = case["T"], s["pos"].data_ptr()
            e.rot_dim, e.rope_section, e.rope_sections, e.rope_base = 64, DIT.dim, 2, 10000.0
    return s


def _held(logits, model):
    """The cache rows beside `logits` are views of the model's memory, which lives as long as
    the model does: whoever holds the logits holds the model."""
    logits.model = model
    return logits


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "infer":
        return s["decoder"].infer(s["prompt"], s["tokens"], s["feat"], s["spk"], s["z"])
    if kind == "dit":
        return s["est"].forward(s["x"], s["mu"], s["cond"], s["spks"], s["t"])
    if kind == "prefill":
        m = s["model"]
        logits = m.prefill(m.build_lm_input(s["text"], s["speech"]))
        return dict(logits=_held(logits, m), cache=s["cache"])
    if kind == "decode":
        m = s["model"]
        m.set_cache_len(case["cache"])
        return dict(logits=[_held(m.decode(t), m) for t in s["tokens"]],
                    rows=[s["rows"][i] for i in (0, LM.n_layers // 2, LM.n_layers - 1)])
    if kind == "attention":
        nh, nkv = _attn_heads(case)
        return ops.attention(s["q"], s["k"], s["v"], nh, nkv, causal=case["form"] == "lm",
                             products=case["products"])
    if kind == "linear":
        return ops.linear_bx(s["x"], s["wf"], PROJ[case["proj"]][0], s["b"], s["epi"], bm=64,
                             products=case["products"])
    if case["form"] == "ada_ln":
        D = DIT.dim
        return ops.ada_ln(s["x"], s["emb"][:, D:2 * D], s["emb"][:, :D])
    return ops.rms_norm(s["x"], s["w"])


# ---- what a pass cannot do without ----------------------------------------------------


def _dit_work(rows, B, T, steps=1):
    """Estimator: per-row matrix work of `steps` evaluations, attention, conv_pos, and the
    modulation GEMV once per evaluation input; weights read once in fp32."""
    D, ff, mel = DIT.dim, DIT.ff_inner, DIT.mel_dim
    per_row = DIT.depth * 2 * (4 * D * D + 2 * D * ff) + 2 * 4 * mel * D + 2 * mel * D \
        + 2 * 2 * D * 64 * DIT.conv_kernel
    attn = DIT.depth * 4 * B * T * T * D
    mod = 2 * (DIT.depth * 6 * D * D + 2 * D * D)
    weights = DIT.depth * (4 * D * D + 2 * D * ff + 6 * D * D) + 2 * D * D + 5 * mel * D \
        + 2 * D * 64 * DIT.conv_kernel + D * (DIT.freq_dim + D)
    return steps * (rows * per_row + attn + mod), 4 * weights


def _lm_layer_weights():
    KV = LM.n_kv_heads * LM.head_dim
    return LM.hidden * (2 * LM.hidden + 2 * KV + 3 * LM.intermediate)


def work(case):
    kind = case["kind"]
    if kind == "infer":
        MT, L1 = _infer_sizes(case)
        seq = MT // 2
        flops, wbytes = _dit_work(2 * MT, 2, MT, DIT.n_timesteps)
        conv = FLOW.channels * DIT.mel_dim * (FLOW.pre_lookahead + 1 + 3)
        io = 4 * DIT.mel_dim * (seq + L1 + MT + MT - L1)
        return dict(flops=flops + 2 * seq * conv, bytes=wbytes + 4 * conv + io)
    if kind == "dit":
        B, T = case["B"], case["T"]
        flops, wbytes = _dit_work(B * T, B, T)
        return dict(flops=flops, bytes=wbytes + 4 * 4 * B * DIT.mel_dim * T)
    if kind == "prefill":
        L, H = case["L"], LM.hidden
        KV = LM.n_kv_heads * LM.head_dim
        flops = LM.n_layers * (2 * L * _lm_layer_weights() + 2 * L * (L + 1) * H) \
            + 2 * L * H * LM.speech_vocab
        return dict(flops=flops, bytes=4 * (LM.n_layers * (_lm_layer_weights() + 2 * L * KV)
                                            + LM.speech_vocab * (H + L) + L * H))
    if kind == "decode":
        n, c, H = case["steps"], case["cache"], LM.hidden
        KV = LM.n_kv_heads * LM.head_dim
        w = LM.n_layers * _lm_layer_weights() + LM.speech_vocab * H
        keys = n * c + n * (n + 1) // 2
        return dict(flops=2 * n * w + LM.n_layers * 4 * keys * H,
                    bytes=4 * (n * w + LM.n_layers * 2 * (keys + n) * KV + n * (LM.speech_vocab + H)))
    B, T = case["B"], case["T"]
    if kind == "attention":
        nh, nkv = _attn_heads(case)
        hd = DIT.head_dim
        pairs = T * (T + 1) // 2 if case["form"] == "lm" else T * T
        return dict(flops=4 * B * nh * pairs * hd, bytes=4 * B * T * hd * (2 * nh + 2 * nkv))
    if kind == "linear":
        N, K, _ = PROJ[case["proj"]]
        return dict(flops=2 * B * T * N * K, bytes=4 * (B * T * (N + K) + N * K + N))
    if case["form"] == "ada_ln":
        return dict(flops=8 * B * T * DIT.dim, bytes=4 * (2 * B * T * DIT.dim + 2 * B * DIT.dim))
    return dict(flops=4 * T * LM.hidden, bytes=4 * (2 * T * LM.hidden + LM.hidden))


def tolerance(case):
    """Four to five times the error against exact() that each path shows: three-product paths
    carry 16 significant bits per operand, six-product ones are at the fp32 level, and the
    LM's 24 layers multiply the prefill's (2.3e-5 in the deepest cache rows)."""
    kind = case["kind"]
    if kind == "prefill":
        return dict(rel=1e-4)
    if kind in ("infer", "dit"):
        return dict(rel=2e-5)
    if kind == "decode":
        return dict(rel=1e-5)
    if kind in ("attention", "linear"):
        return dict(rel=3e-5 if case["products"] == 3 else 5e-6)
    return dict(rel=1e-6)


# ---- float64 restatement --------------------------------------------------------------


def _f64(params):
    return {k: v.double() for k, v in params.items()}


def _rope_table(n, dim, base):
    inv = 1.0 / torch.pow(torch.tensor(base, dtype=torch.float64),
                          torch.arange(0, dim, 2).double() / dim).float()
    ang = (torch.arange(n).float()[:, None] * inv[None, :]).to(DEV).double()
    return ang.cos(), ang.sin()


def _softmax_attention(q, k, v, causal=False, offset=0):
    """q (B, H, Tq, d), k/v (B, H, Tk, d), head by head."""
    out = torch.empty_like(q)
    scale = q.shape[-1] ** -0.5
    mask = None
    if causal:
        i = torch.arange(q.shape[2], device=DEV)[:, None] + offset
        mask = torch.arange(k.shape[2], device=DEV)[None, :] > i
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = torch.mm(q[b, h], k[b, h].t().contiguous()) * scale
            if mask is not None:
                s.masked_fill_(mask, -math.inf)
            out[b, h] = torch.mm(torch.softmax(s, -1), v[b, h])
    return out


def _heads(x, n):
    B, T, _ = x.shape
    return x.reshape(B, T, n, -1).transpose(1, 2).contiguous()


def _rope_partial(x, cos, sin, rot=64):
    """Interleaved pairs of the first `rot` channels of x (B, T, D)."""
    a, b = x[..., 0:rot:2].clone(), x[..., 1:rot:2].clone()
    x[..., 0:rot:2] = a * cos - b * sin
    x[..., 1:rot:2] = b * cos + a * sin
    return x


def _ada_ln(x, shift, scale):
    return F.layer_norm(x, x.shape[-1:], eps=1e-6) * (1 + scale[:, None]) + shift[:, None]


def _conv_pos(x, w, b):
    """mish(causal grouped conv), x (B, T, C), w (C, C/G, K)."""
    B, T, C = x.shape
    K, G = w.shape[2], DIT.conv_groups
    xp = F.pad(x, (0, 0, K - 1, 0))
    y = torch.zeros_like(x)
    for k in range(K):
        tap = w[:, :, k].reshape(G, C // G, -1)
        for g in range(G):
            c = slice(g * (C // G), (g + 1) * (C // G))
            for i in range(B):
                y[i, :, c] += torch.mm(xp[i, k:k + T, c].contiguous(), tap[g].t().contiguous())
    return F.mish(y + b)


def _dit64(p, x, mu, cond, spks, t):
    B, mel, T = x.shape
    half = DIT.freq_dim // 2
    coeff = torch.exp(-torch.arange(half).float() * (math.log(10000.0) / (half - 1))).to(DEV)
    ang = ((1000.0 * t.float())[:, None] * coeff[None, :]).double()
    e = torch.cat([ang.sin(), ang.cos()], -1)
    e = F.linear(e, p["time_embed.time_mlp.0.weight"], p["time_embed.time_mlp.0.bias"])
    e = F.linear(F.silu(e), p["time_embed.time_mlp.2.weight"], p["time_embed.time_mlp.2.bias"])
    se = F.silu(e)
    a0 = torch.cat([x.transpose(1, 2), cond.transpose(1, 2), mu.transpose(1, 2),
                    spks[:, None].expand(B, T, mel)], -1)
    h = F.linear(a0, p["input_embed.proj.weight"], p["input_embed.proj.bias"])
    c = "input_embed.conv_pos_embed.conv"
    c1 = _conv_pos(h, p[c + "1.0.weight"], p[c + "1.0.bias"])
    h = h + _conv_pos(c1, p[c + "2.0.weight"], p[c + "2.0.bias"])
    cos, sin = _rope_table(T, 64, 10000.0)
    for i in range(DIT.depth):
        b = f"transformer_blocks.{i}."

        def lin(y, name):
            return F.linear(y, p[b + name + ".weight"], p[b + name + ".bias"])

        sh1, sc1, g1, sh2, sc2, g2 = lin(se, "attn_norm.linear").chunk(6, -1)
        n = _ada_ln(h, sh1, sc1)
        q = _rope_partial(lin(n, "attn.to_q"), cos, sin)
        k = _rope_partial(lin(n, "attn.to_k"), cos, sin)
        o = _softmax_attention(_heads(q, DIT.heads), _heads(k, DIT.heads),
                               _heads(lin(n, "attn.to_v"), DIT.heads))
        o = o.transpose(1, 2).reshape(B, T, DIT.dim)
        h = h + g1[:, None] * lin(o, "attn.to_out.0")
        n = F.gelu(lin(_ada_ln(h, sh2, sc2), "ff.ff.0.0"), approximate="tanh")
        h = h + g2[:, None] * lin(n, "ff.ff.2")
    sc, sh = F.linear(se, p["norm_out.linear.weight"], p["norm_out.linear.bias"]).chunk(2, -1)
    out = F.linear(_ada_ln(h, sh, sc), p["proj_out.weight"], p["proj_out.bias"])
    return out.transpose(1, 2).contiguous()


def _infer64(case, s):
    w, p = _f64(s["front"]), _f64(s["dit"])
    MT, L1 = _infer_sizes(case)
    e = s["spk"].double()
    spk = F.linear(e / e.square().sum().clamp(min=1e-12).sqrt(),
                   w["spk_embed_affine_layer.weight"], w["spk_embed_affine_layer.bias"])
    ids = torch.from_numpy(np.concatenate([s["prompt"], s["tokens"]]).astype(np.int64)).to(DEV)
    x = w["input_embedding.weight"][ids]

    def conv(y, name):
        k = w[name + ".weight"].shape[2]
        n = y.shape[0] - k + 1
        cols = torch.cat([y[i:i + n] for i in range(k)], -1)
        return F.linear(cols, w[name + ".weight"].permute(0, 2, 1).reshape(-1, cols.shape[1])
                        .contiguous(), w[name + ".bias"])

    y = F.leaky_relu(conv(F.pad(x, (0, 0, 0, FLOW.pre_lookahead)), "pre_lookahead_layer.conv1"),
                     0.01)
    y = conv(F.pad(y, (0, 0, 2, 0)), "pre_lookahead_layer.conv2") + x
    mu = y.repeat_interleave(FLOW.token_mel_ratio, 0).t()
    cond = torch.zeros(DIT.mel_dim, MT, device=DEV, dtype=torch.float64)
    cond[:, :L1] = s["feat"].double().t()

    def pair(v):
        return torch.stack([v, torch.zeros_like(v)])

    z = s["z"].double()
    span = cfm_t_span(DIT.n_timesteps)
    t, dt = span[0], np.float32(span[1] - span[0])
    for step in range(1, DIT.n_timesteps + 1):
        tt = torch.full((2,), float(t), device=DEV)
        d = _dit64(p, torch.stack([z, z]), pair(mu), pair(cond), pair(spk), tt)
        z = z + float(dt) * ((1.0 + DIT.cfg_rate) * d[0] - DIT.cfg_rate * d[1])
        t = np.float32(t + dt)
        if step < DIT.n_timesteps:
            dt = np.float32(span[step + 1] - t)
    return z[:, L1:].contiguous()


def _lm64(p, x, past_k=None, past_v=None):
    """x (L, H) after the given cache rows; returns logits, new k rows and v rows per layer."""
    L, past = x.shape[0], 0 if past_k is None else past_k[0].shape[0]
    cos, sin = _rope_table(past + L, LM.head_dim, LM.rope_theta)
    cos, sin = cos[past:], sin[past:]

    def norm(y, w):
        return y * torch.rsqrt(y.square().mean(-1, keepdim=True) + LM.rms_eps) * w

    def rope(y, n):
        a, b = y.reshape(L, n, 2, LM.head_dim // 2).unbind(2)
        c, s = cos[:, None], sin[:, None]
        return torch.cat([a * c - b * s, b * c + a * s], -1).reshape(L, -1)

    ks, vs = [], []
    rep = LM.n_heads // LM.n_kv_heads
    for i in range(LM.n_layers):
        b = f"layers.{i}."

        def lin(y, name):
            return F.linear(y, p[b + name + ".weight"], p.get(b + name + ".bias"))

        n = norm(x, p[b + "input_layernorm.weight"])
        q = rope(lin(n, "self_attn.q_proj"), LM.n_heads)
        k = rope(lin(n, "self_attn.k_proj"), LM.n_kv_heads)
        v = lin(n, "self_attn.v_proj")
        ks.append(k)
        vs.append(v)
        if past:
            k, v = torch.cat([past_k[i], k]), torch.cat([past_v[i], v])
        kh = _heads(k[None], LM.n_kv_heads).repeat_interleave(rep, 1)
        vh = _heads(v[None], LM.n_kv_heads).repeat_interleave(rep, 1)
        o = _softmax_attention(_heads(q[None], LM.n_heads), kh, vh, causal=True, offset=past)
        x = x + lin(o.transpose(1, 2).reshape(L, -1), "self_attn.o_proj")
        n = norm(x, p[b + "post_attention_layernorm.weight"])
        n = F.silu(lin(n, "mlp.gate_proj")) * lin(n, "mlp.up_proj")
        x = x + lin(n, "mlp.down_proj")
    logits = F.linear(norm(x, p["norm.weight"]), p["llm_decoder.weight"])
    return logits, ks, vs


def exact(case, seed):
    s = _DRAW[case["kind"]](case, seed)
    kind = case["kind"]
    if kind == "infer":
        return _infer64(case, s)
    if kind == "dit":
        return _dit64(_f64(s["dit"]), *(s[k].double() for k in ("x", "mu", "cond", "spks")), s["t"])
    if kind in ("prefill", "decode"):
        text_table = s["lm"].pop("embed_tokens.weight")
        p = _f64(s["lm"])
        speech = p["speech_embedding.weight"]
    if kind == "prefill":
        x = torch.cat([speech[6561:6562], text_table[s["text"]].double(), speech[6563:6564],
                       speech[s["speech"]]])
        logits, ks, vs = _lm64(p, x)
        return dict(logits=logits, cache=list(zip(ks, vs)))
    if kind == "decode":
        # causal attention makes the tokens one pass over the cache and each other
        logits, ks, vs = _lm64(p, speech[s["tokens"]], [k.double() for k in s["k"]],
                               [v.double() for v in s["v"]])
        at = (0, LM.n_layers // 2, LM.n_layers - 1)
        return dict(logits=list(logits), rows=[(ks[i], vs[i]) for i in at])
    if kind == "attention":
        nh, nkv = _attn_heads(case)
        hd = DIT.head_dim
        q, k, v = s["qkv"].double().split([nh * hd, nkv * hd, nkv * hd], dim=-1)
        k = _heads(k, nkv).repeat_interleave(nh // nkv, 1)
        v = _heads(v, nkv).repeat_interleave(nh // nkv, 1)
        o = _softmax_attention(_heads(q, nh), k, v, causal=case["form"] == "lm")
        return o.transpose(1, 2).reshape(case["B"], case["T"], nh * hd).contiguous()
    if kind == "linear":
        y = F.linear(s["x"].double(), s["W"].double(), s["b"].double())
        epi = PROJ[case["proj"]][2]
        if epi == "gelu":
            return F.gelu(y, approximate="tanh")
        if epi == "rope":
            y = y.view(case["B"], case["T"], -1)
            cos, sin = _rope_table(case["T"], 64, 10000.0)
            for sec in range(2):
                _rope_partial(y[..., sec * DIT.dim:(sec + 1) * DIT.dim], cos, sin)
            y = y.view(case["B"] * case["T"], -1)
        return y
    x = s["x"].double()
    if case["form"] == "ada_ln":
        D = DIT.dim
        e = s["emb"].double()
        return _ada_ln(x, e[:, :D], e[:, D:2 * D])
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * s["w"].double()
