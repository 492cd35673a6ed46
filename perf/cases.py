"""Performance cases of the MoE decode / prefill library: one pass of a public entry point each.

Sizes are those of the two model shapes the library is configured for (Qwen3-30B-A3B and
GPT-OSS-20B) over the batch sizes, KV lengths and prompt lengths that a serving program meets.
All inputs and weights are drawn on the GPU from the seed alone; `exact` restates every path in
float64 torch.  A case is a dict: `kind` names the path, the rest are its sizes.
"""
from __future__ import annotations

import math

import torch

from __graft_entry__ import load_package

DEV = "cuda:0"
BF16, F32, F64, I32 = torch.bfloat16, torch.float32, torch.float64, torch.int32
SHAPES = {
    "qwen": dict(H=2048, Hp=2048, nq=32, nkv=4, d=128, E=128, K=8, I=768, V=151936, eps=1e-6),
    "gpt": dict(H=2880, Hp=3072, nq=64, nkv=8, d=64, E=32, K=4, I=2880, V=201088, eps=1e-5),
}
THETA = 1e6                      # Qwen RoPE base
WINDOW, ALPHA, LIMIT = 128, 1.702, 7.0   # GPT-OSS sliding window, Swish alpha, expert clamp
W_STD = 0.02                     # linear weights
# GPT-OSS residual-writing projections (o_proj, down), scaled by 1 / sqrt(2 x 24 layers) as trained
# models are initialised: at 0.02 one layer's MXFP8 rounding would swamp the residual stream
OUT_STD = W_STD / 48 ** 0.5
ROUTER_STD = 0.05                # logits of std ~2.3: the peaked routing of a trained router
KV_SCALE = 32.0                  # FP8 KV cache: unit-variance rows use e4m3's middle binades
FP8_CLIP = 240.0
FMT = {"mxfp8": 1, "mxfp4": 2}   # the library's MX format numbers
BYTES = {"bf16": 2.0, "mxfp8": 1 + 1 / 32, "mxfp4": 0.5 + 1 / 32, "fp8row": 1.0}
GRID4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)   # E2M1 magnitudes by code


def listed():
    return [
        # one token through one norm: the smallest call, whose cost is the call itself
        dict(name="norm_1", kind="norm", rows=1, H=2048, dtype="bf16"),
        # the router of a small decode batch (softmax, top 8 of 128, renormalised)
        dict(name="router_16", kind="router", T=16, H=2048, E=128, K=8, dtype="f32"),
        # attention block of a small batch at a context of 2048: flat bf16 cache, q/k norms
        dict(name="attn_4x2048", kind="attn", B=4, S=2048, shape="qwen", kv="bf16", block=0),
        # attention block of a serving batch on a paged FP8 cache, which halves the KV memory
        dict(name="attn_fp8_16x4096", kind="attn", B=16, S=4096, shape="qwen", kv="fp8", block=64),
        # the experts of a full decode batch, and of half a batch with MXFP8 weights
        dict(name="moe_64", kind="moe", T=64, fmt="bf16"),
        dict(name="moe_mxfp8_32", kind="moe", T=32, fmt="mxfp8"),
        # the experts of a short prompt of odd length, and of a large prompt batch
        dict(name="moe_prefill_1003", kind="moe_prefill", T=1003),
        dict(name="moe_prefill_8192", kind="moe_prefill", T=8192),
        # one decoder layer for a full serving batch: paged cache, ragged lengths up to 8192
        dict(name="layer_decode_64", kind="layer_decode", B=64, S=8192, block=64, fmt="bf16"),
        # one decoder layer over a 2048-token prompt (context encoding)
        dict(name="layer_prefill_2048", kind="layer_prefill", T=2048),
        # whole greedy steps: one stream's latency (8 layers), a GPT-OSS MXFP4 batch (4 layers)
        dict(name="step_1", kind="step", B=1, S=2048, layers=8),
        dict(name="gptoss_step_32", kind="gptoss_step", B=32, S=4096, layers=4),
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))
    kind = rng.choice(["norm", "router", "attn", "attn", "moe", "moe", "moe_prefill", "moe_prefill",
                       "layer_decode", "layer_decode", "layer_prefill", "layer_prefill", "step",
                       "gptoss_step"])
    if kind == "norm":
        return dict(kind=kind, rows=log(1, 4096), H=rng.choice([2048, 3072, 4096]),
                    dtype=rng.choice(["bf16", "f32"]))
    if kind == "router":
        E, K = rng.choice([(128, 8), (32, 4)])
        return dict(kind=kind, T=log(1, 2048), H=rng.choice([2048, 3072]), E=E, K=K,
                    dtype=rng.choice(["bf16", "f32"]))
    if kind == "attn":
        kv, block = rng.choice(["bf16", "fp8"]), rng.choice([0, 64])
        B = log(1, 64)
        S = log(128, min(8192, 65536 // B))
        return dict(kind=kind, B=B, S=(S + 63) // 64 * 64 if block else S, kv=kv, block=block,
                    shape=rng.choice(["qwen", "qwen", "gpt"]))
    if kind == "moe":
        return dict(kind=kind, T=log(1, 128), fmt=rng.choice(["bf16", "mxfp8", "mxfp4", "fp8row"]))
    if kind == "moe_prefill":
        return dict(kind=kind, T=log(129, 8192))
    if kind == "layer_decode":
        return dict(kind=kind, B=log(1, 64), S=log(512, 8192) // 64 * 64, block=rng.choice([0, 64]),
                    fmt=rng.choice(["bf16", "bf16", "mxfp8", "mxfp4"]))
    if kind == "layer_prefill":
        return dict(kind=kind, T=log(16, 4096))
    if kind == "step":
        return dict(kind=kind, B=log(1, 16), S=log(256, 4096), layers=rng.randint(1, 8))
    return dict(kind=kind, B=log(1, 32), S=log(256, 4096), layers=rng.choice([2, 4]))


# ------------------------------------------------------------------------------ inputs
class Rand:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed) + 1)

    def n(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(*shape, generator=self.g, device=DEV)
        return t.mul_(std).add_(mean).to(dtype)

    def ints(self, lo, hi, n):
        return torch.randint(lo, hi + 1, (n,), generator=self.g, device=DEV, dtype=I32)


def _dt(name):
    return {"bf16": BF16, "f32": F32}[name]


def _routing(r, T, E, K):
    """Expert ids [T, K] and scattered affinities [T, E]: some experts are busier than others."""
    logits = r.n(T, E, dtype=F32) + r.n(E, std=0.5, dtype=F32)
    top, idx = torch.topk(logits, K, dim=-1)
    aff = torch.zeros(T, E, device=DEV).scatter_(1, idx, torch.softmax(top, -1))
    return idx.to(I32), aff


def _norm_inputs(c, seed):
    r = Rand(seed)
    return dict(x=r.n(c["rows"], c["H"], dtype=_dt(c["dtype"])), g=r.n(c["H"], std=0.02, mean=1.0))


def _router_inputs(c, seed):
    r = Rand(seed)
    w = r.n(c["H"], c["E"], std=ROUTER_STD)
    return dict(x=r.n(c["T"], c["H"], dtype=_dt(c["dtype"])), w=w.to(_dt(c["dtype"])))


def _attn_inputs(c, seed):
    """X, weights, caches and the 0/1 mask of ragged lengths in [S/2, S - 1] (the longest S - 1)."""
    r, m, B, S = Rand(seed), SHAPES[c["shape"]], c["B"], c["S"]
    Hp, nq, nkv, d = m["Hp"], m["nq"], m["nkv"], m["d"]
    fp8, blk = c["kv"] == "fp8", c["block"]
    x = r.n(B, 1, Hp)
    x[..., m["H"]:] = 0
    g = r.n(Hp, std=0.02, mean=1.0)
    lens = r.ints(max(1, S // 2), max(1, S - 1), B)
    lens[0] = S - 1
    w = r.n(Hp, (nq + 2 * nkv) * d, std=W_STD)
    wo = r.n(nq * d, Hp, std=W_STD / (KV_SCALE if fp8 else 1.0))
    shape = (B * (S // blk), blk, nkv, d) if blk else (B, nkv, S, d)
    kc, vc = r.n(*shape), r.n(*shape)
    if fp8:
        kc, vc = [(t.float() * KV_SCALE).clamp_(-FP8_CLIP, FP8_CLIP).to(torch.float8_e4m3fn) for t in (kc, vc)]
    table = None
    pos = lens.long()
    if blk:
        table = torch.randperm(B * (S // blk), generator=r.g, device=DEV).to(I32).reshape(B, S // blk)
        pos = table.long().gather(1, (pos // blk)[:, None])[:, 0] * blk + pos % blk
    mask = torch.arange(S, device=DEV)[:, None] < lens[None, :]
    mask[S - 1] = True                                          # the new token's own slot
    mask = mask[:, :, None, None].expand(S, B, nq, 1).to(torch.uint8).contiguous()
    ang = lens.float()[None] * (THETA ** (-torch.arange(0, d, 2, device=DEV).float() / d))[:, None]
    s = dict(x=x, g=g, w=w, wo=wo, kc=kc, vc=vc, table=table, mask=mask, lens=lens, pos=pos.to(I32),
             cos=ang.cos()[:, :, None].contiguous(), sin=ang.sin()[:, :, None].contiguous(),
             bq=None, bo=None, qn=None, kn=None, sink=None)
    if c["shape"] == "qwen":
        s.update(qn=r.n(d, std=0.02, mean=1.0), kn=r.n(d, std=0.02, mean=1.0))
    else:
        s.update(bq=r.n((nq + 2 * nkv) * d, std=W_STD), bo=r.n(Hp, std=W_STD),
                 sink=r.n(nq, 1, dtype=F32))
    return s


def _moe_inputs(c, seed):
    """Hidden rows, routing, and expert weights in the operator's layouts, of std 0.02."""
    r, m, T, fmt = Rand(seed), SHAPES["qwen"], c["T"], c.get("fmt", "bf16")
    H, E, K, I = m["H"], m["E"], m["K"], m["I"]
    x = r.n(T, H)
    idx, aff = _routing(r, T, E, K)
    s = dict(x=x, idx=idx, aff=aff, gs=None, ds=None)
    if fmt == "bf16":
        s.update(gu=r.n(E, H, 2, I, std=W_STD), dn=r.n(E, I, H, std=W_STD))
    elif fmt == "fp8row":       # e4m3 codes around +-100, one scale per output column
        s.update(gu=r.n(E, H, 2, I, std=100.0, dtype=F32).clamp_(-240, 240).to(torch.float8_e4m3fn),
                 dn=r.n(E, I, H, std=100.0, dtype=F32).clamp_(-240, 240).to(torch.float8_e4m3fn),
                 gs=r.n(E, 2, I, std=2e-5, mean=2e-4, dtype=F32),
                 ds=r.n(E, H, std=2e-5, mean=2e-4, dtype=F32))
    else:                        # MX codes as a quantiser leaves them, E8M0 scales per 32
        t_h, t_i = H // 512, (I + 511) // 512
        lead_g, lead_d = (E, 128, 2, t_h, I), (E, 128, t_i, H)
        if fmt == "mxfp8":
            def code(lead):
                return r.n(*lead, 4, std=128.0, dtype=F32).clamp_(-448, 448).to(torch.float8_e4m3fn)
            e0 = 127 - 13
        else:
            cuts = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)

            def code(lead):
                v = r.n(*lead, 4, std=2.0, dtype=F32)
                q = (torch.bucketize(v.abs(), cuts) + 8 * (v < 0)).to(torch.uint8)
                return (q[..., 0::2] + 16 * q[..., 1::2]).contiguous()
            e0 = 127 - 7

        def scales(*shape):
            return (e0 + r.ints(0, 1, math.prod(shape))).to(torch.uint8).reshape(shape)
        gu, dn = code(lead_g), code(lead_d)
        gs, ds = scales(E, 16, 2, t_h, I), scales(E, 16, t_i, H)
        last = (I - 512 * (t_i - 1)) // 4            # positions past I hold zeros
        dn.view(torch.uint8)[:, last:, t_i - 1] = 0
        ds[:, last // 8:, t_i - 1] = 0
        s.update(gu=gu, dn=dn, gs=gs, ds=ds)
    return s


def _qwen_layer_weights(r):
    m = SHAPES["qwen"]
    H, nq, nkv, d, E, I = (m[k] for k in ("H", "nq", "nkv", "d", "E", "I"))
    return dict(q_proj=r.n(nq * d, H, std=W_STD), k_proj=r.n(nkv * d, H, std=W_STD),
                v_proj=r.n(nkv * d, H, std=W_STD), o_proj=r.n(H, nq * d, std=W_STD),
                q_norm=r.n(d, std=0.02, mean=1.0), k_norm=r.n(d, std=0.02, mean=1.0),
                input_layernorm=r.n(H, std=0.02, mean=1.0),
                post_attention_layernorm=r.n(H, std=0.02, mean=1.0),
                gate=r.n(E, H, std=ROUTER_STD), gate_up_proj=r.n(E, 2 * I, H, std=W_STD),
                down_proj=r.n(E, H, I, std=W_STD))


def _gpt_layer_weights(r):
    m = SHAPES["gpt"]
    H, nq, nkv, d, E, I = (m[k] for k in ("H", "nq", "nkv", "d", "E", "I"))
    w = {}
    for n, rows, cols, std in (("q_proj", nq * d, H, W_STD), ("k_proj", nkv * d, H, W_STD),
                               ("v_proj", nkv * d, H, W_STD), ("o_proj", H, nq * d, OUT_STD)):
        w[n + ".weight"], w[n + ".bias"] = r.n(rows, cols, std=std), r.n(rows, std=W_STD)
    w.update({"sinks": r.n(nq, dtype=F32), "input_layernorm": r.n(H, std=0.02, mean=1.0),
              "post_attention_layernorm": r.n(H, std=0.02, mean=1.0),
              "router.weight": r.n(E, H, std=ROUTER_STD), "router.bias": r.n(E, std=W_STD),
              "experts.gate_up_proj": r.n(E, H, 2 * I, std=W_STD),
              "experts.gate_up_proj_bias": r.n(E, 2 * I, std=W_STD),
              "experts.down_proj": r.n(E, I, H, std=OUT_STD),
              "experts.down_proj_bias": r.n(E, H, std=W_STD)})
    return w


def _layers_of(c):
    return c.get("layers", 1)


def _model_inputs(c, seed, visit):
    """Everything of a model case: `visit(layer, weights)` sees each layer's weights in turn.
    Residual rows have unit variance (the residual stream outweighs one layer's update)."""
    r, kind = Rand(seed), c["kind"]
    gpt = kind == "gptoss_step"
    m = SHAPES["gpt" if gpt else "qwen"]
    for l in range(_layers_of(c)):
        visit(l, _gpt_layer_weights(r) if gpt else _qwen_layer_weights(r))
    s = {}
    if kind == "layer_prefill":
        s["hidden"] = r.n(1, c["T"], m["H"])
        return s
    B, S = c["B"], c["S"]
    s["lens"] = r.ints(S // 16 if kind == "layer_decode" else max(1, S // 4), S, B)
    s["lens"][0] = S
    if kind == "layer_decode":
        s["hidden"] = r.n(B, 1, m["H"])
    else:
        s["ids"] = r.ints(0, m["V"] - 1, B)
        s["embed"] = r.n(m["V"], m["H"])
        s["ln_f"] = r.n(m["H"], std=0.02, mean=1.0)
        s["lm"] = r.n(m["V"], m["H"], std=W_STD)
    rows = S + 64                                    # cache rows (a multiple of 64 when paged)
    s["caches"], s["table"] = [], None
    blk = c.get("block", 0)
    for l in range(_layers_of(c)):
        n = WINDOW if gpt and l % 2 == 0 else rows
        shape = (B * (n // blk), blk, m["nkv"], m["d"]) if blk else (B, m["nkv"], n, m["d"])
        s["caches"] += [r.n(*shape), r.n(*shape)]
    if blk:
        s["table"] = torch.randperm(B * (rows // blk), generator=r.g, device=DEV).to(I32).reshape(B, -1)
    return s


# ------------------------------------------------------------------------------ prepare / run
def prepare(case, seed):
    mk, kind = load_package(), case["kind"]
    if kind == "norm":
        s = _norm_inputs(case, seed)
        s["out"] = torch.empty_like(s["x"])
    elif kind == "router":
        s = _router_inputs(case, seed)
        T, E, K = case["T"], case["E"], case["K"]
        s["logits"] = torch.empty(T, E, dtype=F32, device=DEV)
        s["aff"] = torch.empty(T, E, dtype=F32, device=DEV)
        s["idx"] = torch.empty(T, K, dtype=I32, device=DEV)
    elif kind == "attn":
        s = _attn_inputs(case, seed)
        s["kv_scale"] = torch.full((1, 1), KV_SCALE, device=DEV) if case["kv"] == "fp8" else None
    elif kind in ("moe", "moe_prefill"):
        s = _moe_inputs(case, seed)
    else:
        s = _prepare_model(mk, case, seed)
    s["case"] = case
    if kind in ("router", "attn", "moe", "moe_prefill"):
        run(s)                   # the operators lay their weights out on a tensor's first use
    return s


def _prepare_model(mk, c, seed):
    import importlib
    Q = importlib.import_module(mk.__name__ + ".qwen_with_megakernel")
    G = importlib.import_module(mk.__name__ + ".gpt_oss_with_megakernel")
    kind, L, B = c["kind"], _layers_of(c), c.get("B", 1)
    packed, rows = [], c["S"] + 64 if "S" in c else c["T"] + 64
    if kind == "gptoss_step":
        cfg = G.GptOssMKConfig(num_hidden_layers=L, max_batch=B, max_seq=rows, expert_format="mxfp4")
        s = _model_inputs(c, seed, lambda l, w: packed.append(G.pack_layer(w, cfg)))
        model = G.GptOssMegakernelModel(cfg, packed, B, DEV, embed=s.pop("embed"), ln_f=s["ln_f"],
                                        lm_head=s.pop("lm"))
    else:
        cfg = Q.Qwen3MoeMKConfig(num_hidden_layers=L, max_batch=B, max_seq=rows,
                                 expert_format=c.get("fmt", "bf16"), kv_block_len=c.get("block", 0))
        s = _model_inputs(c, seed, lambda l, w: packed.append(Q.pack_layer(w, cfg.expert_format)))
        model = Q.Qwen3MoeMegakernelModel(cfg, packed, B, DEV, embed=s.pop("embed", None),
                                          ln_f=s.get("ln_f"), lm_head=s.pop("lm", None))
    s["model"] = model
    if kind == "layer_prefill":
        s["pos"] = torch.arange(c["T"], device=DEV)[None]
        return s
    for mine, theirs in zip(s.pop("caches"), model.kv_mgr.past_key_values):
        theirs.copy_(mine)
    if s["table"] is not None:
        model.kv_mgr.block_table.copy_(s["table"])
    if kind == "layer_decode":
        s["pos"] = s["lens"][:, None].contiguous()
        return s
    s["hidden"] = torch.empty(B, SHAPES["gpt" if kind == "gptoss_step" else "qwen"]["Hp"], dtype=BF16, device=DEV)
    s["logits"] = torch.empty(B, cfg.vocab_size, dtype=F32, device=DEV)
    s["next"] = torch.empty(B, dtype=I32, device=DEV)
    return s


def run(s):
    mk, c = load_package(), s["case"]
    kind = c["kind"]
    if kind == "norm":
        return mk.rmsnorm_tkg(s["x"], s["g"], s["out"], eps=1e-6)
    if kind == "router":
        return mk.router_topk(s["x"], s["w"], None, s["logits"], s["aff"], s["idx"],
                              mk.RouterActFnType.SOFTMAX, c["K"], 1, 0, router_pre_norm=True,
                              norm_topk_prob=True)
    if kind == "attn":
        m, none = SHAPES[c["shape"]], mk.QuantizationType.NONE
        return mk.attention_block_tkg(
            s["x"], m["H"], True, m["eps"], s["g"], s["w"], s["bq"], none, None, None,
            s["qn"] is not None, m["eps"], s["qn"], s["kn"], s["cos"], s["sin"], True, False, 0.0, None,
            None, False, s["table"], s["kc"], s["vc"], s["mask"], s["sink"], True, s["pos"], s["wo"],
            s["bo"], none, None, None, False, False, softmax_scale=_softmax_scale(c),
            k_scale=s["kv_scale"], v_scale=s["kv_scale"])
    if kind in ("moe", "moe_prefill"):
        post = mk.ExpertAffinityScaleMode.POST_SCALE
        if kind == "moe_prefill":
            return mk.moe_prefill(s["x"], s["gu"], s["dn"], s["aff"], s["idx"],
                                  expert_affinities_scaling_mode=post)
        return mk.moe_tkg(s["x"], s["gu"], s["dn"], s["aff"], s["idx"], False,
                          expert_gate_up_weights_scale=s["gs"], expert_down_weights_scale=s["ds"],
                          expert_affinities_scaling_mode=post)
    model = s["model"]
    if kind in ("layer_decode", "layer_prefill"):
        y, kv, _, _, _ = model.layers[0](s["hidden"], position_ids=s["pos"],
                                         is_for_context_encoding=kind == "layer_prefill")
        return [y, kv[0], kv[1]]
    model.step(s["ids"], s["lens"], s["hidden"], s["logits"], s["next"])
    return [s["logits"]] + list(model.kv_mgr.past_key_values)


def _softmax_scale(c):
    return SHAPES[c["shape"]]["d"] ** -0.5 / (KV_SCALE if c["kv"] == "fp8" else 1.0)


# ------------------------------------------------------------------------------ work
def _distinct(E, K, T):
    return E * (1 - (1 - K / E) ** T)


def _expert_work(m, T, fmt):
    pairs = 6.0 * T * m["K"] * m["H"] * m["I"]
    return _distinct(m["E"], m["K"], T) * 3 * m["H"] * m["I"] * BYTES[fmt], pairs


def _attn_work(m, rows, kv_rows, kv_bytes):
    wide = m["H"] * (2 * m["nq"] + 2 * m["nkv"]) * m["d"]
    by = 2.0 * wide + kv_rows * 2 * m["nkv"] * m["d"] * kv_bytes
    return by, 2.0 * rows * wide + 4.0 * kv_rows * m["nq"] * m["d"]


def work(case):
    c, kind = case, case["kind"]
    if kind == "norm":
        n = c["rows"] * c["H"]
        return {"bytes": 2.0 * n * (2 if c["dtype"] == "bf16" else 4) + 2 * c["H"], "flops": 4.0 * n}
    if kind == "router":
        T, H, E = c["T"], c["H"], c["E"]
        return {"bytes": (T + E) * H * (2.0 if c["dtype"] == "bf16" else 4.0) + T * (8.0 * E + 4 * c["K"]),
                "flops": 2.0 * T * H * E}
    if kind == "attn":
        m, B, S = SHAPES[c["shape"]], c["B"], c["S"]
        by, fl = _attn_work(m, B, B * 0.75 * S, 1 if c["kv"] == "fp8" else 2)
        return {"bytes": by + S * B * m["nq"] + 4.0 * B * m["H"], "flops": fl}
    m = SHAPES["gpt" if kind == "gptoss_step" else "qwen"]
    if kind in ("moe", "moe_prefill"):
        by, fl = _expert_work(m, c["T"], c.get("fmt", "bf16"))
        return {"bytes": by + 4.0 * c["T"] * m["H"], "flops": fl}
    T = c["T"] if kind == "layer_prefill" else c["B"]
    by, fl = _expert_work(m, T, "mxfp4" if kind == "gptoss_step" else c.get("fmt", "bf16"))
    fixed = 2.0 * m["H"] * m["E"] + 4.0 * T * m["H"]
    router = 2.0 * T * m["H"] * m["E"]
    if kind == "layer_prefill":      # K / V rows written once; every prefix position is scored
        a, f = _attn_work(m, T, T, 2)
        return {"bytes": by + a + fixed, "flops": fl + f + router + 2.0 * T * T * m["nq"] * m["d"]}
    S = c["S"]
    full = c["B"] * (S * 17 / 32 if kind == "layer_decode" else S * 5 / 8)
    bytes_, flops = 0.0, 0.0
    for l in range(_layers_of(c)):
        rows = c["B"] * min(WINDOW - 1, S * 5 / 8) if kind == "gptoss_step" and l % 2 == 0 else full
        a, f = _attn_work(m, T, rows, 2)
        bytes_, flops = bytes_ + by + a + fixed, flops + fl + f + router
    if kind != "layer_decode":
        bytes_, flops = bytes_ + 2.0 * m["V"] * m["H"] + 4.0 * T * m["V"], flops + 2.0 * T * m["V"] * m["H"]
    return {"bytes": bytes_, "flops": flops}


# ------------------------------------------------------------------------------ tolerance
def tolerance(case):
    kind = case["kind"]
    if kind == "norm":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1e-5}
    if kind == "router":            # fp32 sums over H; a near-tie may swap two experts of a row
        return {"rel": 1e-4, "max": 0.5, "differ": 0.01}
    if kind == "attn":              # bf16 rounding of the heads; FP8: of the new rows' codes
        return {"rel": 1.5e-2}
    if kind in ("moe", "moe_prefill"):   # MX: a hidden value one bf16 step off may take another code
        return {"rel": 3e-2 if case.get("fmt", "bf16") in FMT else 1e-2}
    # a near-tie of the router sends a token to another expert: `max` of single values is loose
    loose = kind in ("step", "gptoss_step") or case.get("fmt") in FMT
    return {"rel": 3e-2 if loose else 1.5e-2, "max": 0.9}


# ------------------------------------------------------------------------------ float64
def _rms(x, g, eps, n=None):
    return x * g.double() / torch.sqrt((x * x).sum(-1, keepdim=True) / (n or x.shape[-1]) + eps)


def _rope(x, cos, sin):
    """Contiguous-halves rotation; cos / sin broadcast against x[..., :d/2]."""
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend(q, k, v, scale, sink=None):
    """q [nq, d] over k, v [n, nkv, d] -> [nq, d]."""
    nq, d = q.shape
    nkv = k.shape[1]
    qg = q.reshape(nkv, nq // nkv, d)
    sc = torch.matmul(qg, k.permute(1, 2, 0).contiguous()) * scale          # [nkv, g, n]
    if sink is not None:
        sc = torch.cat([sc, sink.double().reshape(nkv, -1, 1)], -1)
    p = torch.softmax(sc, -1)
    if sink is not None:
        p = p[..., :-1]
    return torch.matmul(p, v.permute(1, 0, 2).contiguous()).reshape(nq, d)


def _mx_qdq(x, fmt=1):
    """OCP MX quantise and dequantise along the last dim (a multiple of 32)."""
    b = x.double().reshape(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    e = torch.floor(torch.log2(torch.where(amax > 0, amax, torch.ones_like(amax)))) - (8 if fmt == 1 else 2)
    X = torch.exp2(e)
    v = b / X
    if fmt == 1:
        q = v.clamp(-448, 448).float().to(torch.float8_e4m3fn).double()
    else:
        a = v.abs()
        code = ((a > 0.25).to(torch.int64) + (a >= 0.75) + (a > 1.25) + (a >= 1.75) + (a > 2.5) + (a >= 3.5)
                + (a > 5.0))
        q = torch.tensor(GRID4, device=x.device, dtype=F64)[code] * v.sign()
    return (q * X).reshape(x.shape)


def _experts(x, idx, wgt, gate_up, down, act, act_q=None):
    """sum_k wgt * down(act(gate_up(x))) with gate_up(e) -> ([H, 2I], bias), down(e) -> ([I, H], bias)."""
    y = torch.zeros_like(x)
    xin = _mx_qdq(x) if act_q else x
    for e in torch.unique(idx).tolist():
        t, k = torch.nonzero(idx == e, as_tuple=True)
        w, b = gate_up(e)
        h = act(xin[t] @ w + b)
        if act_q:
            h = _mx_qdq(h)
        w, b = down(e)
        y.index_add_(0, t, wgt[t, k][:, None] * (h @ w + b))
    return y


def _silu_mul(z):
    g, u = z.chunk(2, -1)
    return g * torch.sigmoid(g) * u


def _e2m1(codes):
    both = torch.stack([codes & 15, codes >> 4], -1).flatten(-2).long()
    v = torch.tensor(GRID4, device=codes.device, dtype=F64)[both & 7]
    return torch.where(both >= 8, -v, v)


def _moe_weights(s, fmt):
    """Per-expert float64 [H, 2I] and [I, H] of the operator's layouts."""
    m = SHAPES["qwen"]
    H, I = m["H"], m["I"]
    if fmt == "bf16":
        return (lambda e: (s["gu"][e].double().reshape(H, 2 * I), 0.0)), lambda e: (s["dn"][e].double(), 0.0)
    if fmt == "fp8row":
        return ((lambda e: (s["gu"][e].double().reshape(H, 2 * I) * s["gs"][e].double().reshape(-1), 0.0)),
                lambda e: (s["dn"][e].double() * s["ds"][e].double(), 0.0))
    dec = (lambda t: t.double()) if fmt == "mxfp8" else _e2m1

    def gate_up(e):     # [128 p, 2, t, I, 4 j], h = 512 t + 4 p + j; scale block t * 16 + p // 8
        v = dec(s["gu"][e]) * torch.exp2(s["gs"][e].double() - 127).repeat_interleave(8, 0)[..., None]
        return v.permute(2, 0, 4, 1, 3).reshape(H, 2 * I), 0.0

    def down(e):        # [128 p, t, H, 4 j], i = 512 t + 4 p + j
        v = dec(s["dn"][e]) * torch.exp2(s["ds"][e].double() - 127).repeat_interleave(8, 0)[..., None]
        return v.permute(1, 0, 3, 2).reshape(-1, H)[:I], 0.0
    return gate_up, down


def _qwen_layer64(x, w, attend, rope, fmt):
    """x [T, H] -> (x', k [T, nkv, d], v); attend(q, k, v) -> [T, nq, d]."""
    m = SHAPES["qwen"]
    T, d, I = x.shape[0], m["d"], m["I"]
    h = _rms(x, w["input_layernorm"], m["eps"])
    q = _rms((h @ w["q_proj"].double().t()).reshape(T, -1, d), w["q_norm"], m["eps"])
    k = _rms((h @ w["k_proj"].double().t()).reshape(T, -1, d), w["k_norm"], m["eps"])
    v = (h @ w["v_proj"].double().t()).reshape(T, -1, d)
    q, k = _rope(q, *rope), _rope(k, *rope)
    x = x + attend(q, k, v).reshape(T, -1) @ w["o_proj"].double().t()
    n = _rms(x, w["post_attention_layernorm"], m["eps"])
    top, idx = torch.topk(torch.softmax(n @ w["gate"].double().t(), -1), m["K"], dim=-1)
    qd = (lambda t: _mx_qdq(t, FMT[fmt])) if fmt in FMT else (lambda t: t.double())
    moe = _experts(n, idx, top / top.sum(-1, keepdim=True),
                   lambda e: (qd(w["gate_up_proj"][e]).t(), 0.0), lambda e: (qd(w["down_proj"][e]).t(), 0.0),
                   _silu_mul, fmt in FMT)
    return x + moe, k, v


def _gpt_layer64(x, w, attend, rope):
    m = SHAPES["gpt"]
    T, d = x.shape[0], m["d"]

    def lin(t, n):
        return t @ w[n + ".weight"].double().t() + w[n + ".bias"].double()
    h = _rms(x, w["input_layernorm"], m["eps"])
    q, k, v = (lin(h, n).reshape(T, -1, d) for n in ("q_proj", "k_proj", "v_proj"))
    q, k = _rope(q, *rope), _rope(k, *rope)
    x = x + lin(attend(q, k, v).reshape(T, -1), "o_proj")
    n = _rms(x, w["post_attention_layernorm"], m["eps"])
    top, idx = torch.topk(lin(n, "router"), m["K"], dim=-1)

    def gate_up(e):     # gate / up columns alternate; "up + 1" sits in the bias
        g, b = w["experts.gate_up_proj"][e], w["experts.gate_up_proj_bias"][e].double()
        g = torch.cat([_mx_qdq(g[:, i::2].t().contiguous(), 2).t() for i in (0, 1)], 1)
        return g, torch.cat([b[0::2], (b[1::2] + 1.0).to(BF16).double()])

    def down(e):
        g = w["experts.down_proj"][e]
        return _mx_qdq(g.t().contiguous(), 2).t(), w["experts.down_proj_bias"][e].double()

    def act(z):
        g, u = z.chunk(2, -1)
        g, u = g.clamp(max=LIMIT), u.clamp(1 - LIMIT, 1 + LIMIT)
        return g * torch.sigmoid(ALPHA * g) * u
    return x + _experts(n, idx, torch.softmax(top, -1), gate_up, down, act, True), k, v


def _yarn(pos):
    """GPT-OSS RoPE tables (YaRN, theta 150000, factor 32, 4096 original positions)."""
    d, base, factor = 64, 150000.0, 32.0

    def corr(rot):
        return d * math.log(4096 / (rot * 2 * math.pi)) / (2 * math.log(base))
    i = torch.arange(d // 2, dtype=F64, device=DEV)
    extra = base ** (-2 * i / d)
    lo, hi = max(corr(32.0), 0.0), min(corr(1.0), d - 1.0)
    keep = 1 - ((i - lo) / (hi - lo)).clamp(0, 1)
    ang = pos.double()[:, None, None] * (extra / factor * (1 - keep) + extra * keep)
    s = 0.1 * math.log(factor) + 1
    return ang.cos() * s, ang.sin() * s


def _qwen_rope(pos):
    d = SHAPES["qwen"]["d"]
    ang = pos.double()[:, None, None] * THETA ** (-torch.arange(0, d, 2, dtype=F64, device=DEV) / d)
    return ang.cos(), ang.sin()


def _rows(cache, table, b, n):
    """The first n positions of sequence b as float64 [n, nkv, d]."""
    if table is None:
        return cache[b, :, :n].transpose(0, 1).double()
    blk = cache.shape[1]
    used = table[b, : (n + blk - 1) // blk].long()
    return cache[used].flatten(0, 1)[:n].double()


def _store(cache, table, b, t, row):
    if table is None:
        cache[b, :, t] = row
    else:
        cache[int(table[b, t // cache.shape[1]]), t % cache.shape[1]] = row


def _exact_attn(c, seed):
    s, m, fp8 = _attn_inputs(c, seed), SHAPES[c["shape"]], c["kv"] == "fp8"
    B, d, nq, nkv = c["B"], m["d"], m["nq"], m["nkv"]
    h = _rms(s["x"][:, 0].double(), s["g"], m["eps"], m["H"])
    z = h @ s["w"].double() + (s["bq"].double() if s["bq"] is not None else 0.0)
    q, k, v = z.reshape(B, -1, d).split([nq, nkv, nkv], 1)
    if s["qn"] is not None:
        q, k = _rms(q, s["qn"], m["eps"]), _rms(k, s["kn"], m["eps"])
    cos, sin = s["cos"][:, :, 0].t()[:, None].double(), s["sin"][:, :, 0].t()[:, None].double()
    q, k = _rope(q, cos, sin), _rope(k, cos, sin)
    if fp8:
        k, v = [(t * KV_SCALE).clamp(-FP8_CLIP, FP8_CLIP).float().to(torch.float8_e4m3fn).double()
                for t in (k, v)]
    kc, vc = s["kc"].double(), s["vc"].double()
    o = torch.empty(B, nq, d, dtype=F64, device=DEV)
    for b in range(B):
        n = int(s["lens"][b])
        kk = torch.cat([_rows(s["kc"], s["table"], b, n), k[b][None]])
        vv = torch.cat([_rows(s["vc"], s["table"], b, n), v[b][None]])
        o[b] = _attend(q[b], kk, vv, _softmax_scale(c), s["sink"])
        _store(kc, s["table"], b, n, k[b])
        _store(vc, s["table"], b, n, v[b])
    out = o.reshape(B, -1) @ s["wo"].double() + (s["bo"].double() if s["bo"] is not None else 0.0)
    return [out, kc, vc]


def _exact_model(c, seed):
    kind, gpt = c["kind"], c["kind"] == "gptoss_step"
    weights = []
    s = _model_inputs(c, seed, lambda l, w: weights.append(w))
    if kind == "layer_prefill":
        T, m = c["T"], SHAPES["qwen"]
        g = m["nq"] // m["nkv"]
        causal = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()

        def prompt(q, k, v):
            o = torch.empty_like(q)
            for i in range(m["nq"]):
                sc = (q[:, i] @ k[:, i // g].t().contiguous()) * m["d"] ** -0.5
                o[:, i] = torch.softmax(sc.masked_fill_(~causal, -math.inf), -1) @ v[:, i // g]
            return o
        x, k, v = _qwen_layer64(s["hidden"][0].double(), weights[0], prompt,
                                _qwen_rope(torch.arange(T, device=DEV)), "bf16")
        pad = [torch.zeros(1, m["nkv"], T + 64, m["d"], dtype=F64, device=DEV) for _ in range(2)]
        pad[0][0, :, :T], pad[1][0, :, :T] = k.transpose(0, 1), v.transpose(0, 1)
        return [x[None], pad[0], pad[1]]
    pos, table = s["lens"], s["table"]
    rope = _yarn(pos) if gpt else _qwen_rope(pos)
    x = s["hidden"][:, 0].double() if kind == "layer_decode" else s["embed"][s["ids"].long()].double()
    caches = []
    for l, w in enumerate(weights):
        kc, vc = s["caches"][2 * l], s["caches"][2 * l + 1]
        ring = gpt and l % 2 == 0

        def step(q, k, v):
            o = torch.empty_like(q)
            for b in range(c["B"]):
                n = int(pos[b])
                n = min(n, WINDOW - 1) if ring else n
                kk = torch.cat([_rows(kc, table, b, n), k[b][None]])
                vv = torch.cat([_rows(vc, table, b, n), v[b][None]])
                o[b] = _attend(q[b], kk, vv, q.shape[-1] ** -0.5, w["sinks"] if gpt else None)
            return o
        x, k, v = _gpt_layer64(x, w, step, rope) if gpt else _qwen_layer64(x, w, step, rope, c.get("fmt", "bf16"))
        new = [kc.double(), vc.double()]
        for b in range(c["B"]):
            t = int(pos[b]) % (WINDOW - 1) if ring else int(pos[b])
            _store(new[0], table, b, t, k[b])
            _store(new[1], table, b, t, v[b])
        caches += new
        weights[l] = None
    if kind == "layer_decode":
        return [x[:, None]] + caches
    f = _rms(x, s["ln_f"], SHAPES["gpt" if gpt else "qwen"]["eps"])
    logits = torch.cat([f @ part.double().t() for part in s["lm"].split(32768)], 1)
    return [logits] + caches


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm":
        s = _norm_inputs(case, seed)
        return _rms(s["x"].double(), s["g"], 1e-6)
    if kind == "router":
        s = _router_inputs(case, seed)
        logits = s["x"].double() @ s["w"].double()
        top, idx = torch.topk(torch.softmax(logits, -1), case["K"], dim=-1)
        aff = torch.zeros_like(logits).scatter_(1, idx, top / top.sum(-1, keepdim=True))
        return [logits, None, aff]
    if kind == "attn":
        return _exact_attn(case, seed)
    if kind in ("moe", "moe_prefill"):
        s, fmt = _moe_inputs(case, seed), case.get("fmt", "bf16")
        gate_up, down = _moe_weights(s, fmt)
        wgt = s["aff"].double().gather(1, s["idx"].long())
        return _experts(s["x"].double(), s["idx"], wgt, gate_up, down, _silu_mul, fmt in FMT)
    return _exact_model(case, seed)
