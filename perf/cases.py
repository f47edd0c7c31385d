"""The steps a user of this framework has it run, at the sizes they come in: one case is one step of a model - a prefill
step over prompts, a decode step over a batch, or a step that mixes portions of prompts with decoded tokens - through the
model classes, the step context and the paged caches, from token ids to logits, cache rows and recurrent state.

Models (random weights in the architectures' shapes):

  dense     Qwen3-0.6B as it is: 28 layers, hidden 1024, 16 / 8 heads of 128, vocabulary 151936, tied; bf16 weights, or the
            framework's fp8 weights (e4m3, a power-of-two scale per row)
  moe       Qwen3-MoE layers at the sizes of the design benchmark (w1024: 32 experts of 512, 4 per token; w2048: 64 of 768, 8)
  gazutar   window attention / channel delta rule layers with group-routed experts at those sizes, bf16 or true float32
  felolorn  forget-gate linear attention / latent attention / head-decay linear attention / latent attention at those sizes

A step is described by `prompts` sequences of `lo`..`hi` new rows behind `past` rows each already has, and `decodes`
sequences of one new row behind `past_lo`..`past_hi` rows.  Decode steps are captured as the engine captures them (one
hipGraph per batch, held by the program and replayed); so are the dense model's prefill steps.  Steps of the other models
that bring prompts are launched eagerly, as the engine launches them.
"""
import math
import os
import sys
import types

import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-ascend_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

SIZES = {
    "w1024": dict(width=1024, layers=4, heads=8, kv_heads=4, dim=128, experts=32, ff=512, top=4, vocab=32768, window=512),
    "w2048": dict(width=2048, layers=4, heads=16, kv_heads=8, dim=128, experts=64, ff=768, top=8, vocab=32768, window=1024),
}
DENSE = dict(width=1024, layers=28, heads=16, kv_heads=8, dim=128, ff=3072, vocab=151936)
EPS = 1e-6
THETA = 1e6
TAPS = 4
BLOCK = {"dense": 16, "moe": 64, "gazutar": 64, "felolorn": 64}


def _case(name, model, size="", weights="bf16", prompts=0, lo=0, hi=0, past=0, decodes=0, past_lo=0, past_hi=0):
    return dict(name=name, model=model, size=size, weights=weights, prompts=prompts, lo=lo, hi=hi, past=past, decodes=decodes,
                past_lo=past_lo, past_hi=past_hi)


def listed():
    return [
        # one user waiting for one token: the latency of a step that is nothing but launches and weights
        _case("dense decode 1 x 128", "dense", decodes=1, past_lo=128, past_hi=128),
        # the headline workload: 32 sequences at 1024 tokens of context
        _case("dense decode 32 x 1024", "dense", decodes=32, past_lo=1024, past_hi=1024),
        # a busy server (up to 256 requests in flight, 100-1024 tokens each): ragged contexts
        _case("dense decode 200 ragged", "dense", decodes=200, past_lo=100, past_hi=1024),
        # fp8 weights, the batch of the shared-prefix workload
        _case("dense decode fp8 weights", "dense", weights="fp8", decodes=64, past_lo=512, past_hi=1100),
        # one short question arriving: what its time to first token consists of
        _case("dense prefill 137 tokens", "dense", prompts=1, lo=137, hi=137),
        # a full house of prompts: the step that sets the headline's time to first token
        _case("dense prefill 16 x 1024", "dense", prompts=16, lo=1024, hi=1024),
        # sparse feed-forwards: every expert is hit in a decode batch
        _case("moe decode 32 x 1024", "moe", "w2048", decodes=32, past_lo=1024, past_hi=1024),
        # recurrent + window-attention layers: a decode batch, ...
        _case("gazutar decode 32 x 1024", "gazutar", "w2048", decodes=32, past_lo=1024, past_hi=1024),
        # ... a prefill step of ragged prompts, ...
        _case("gazutar prefill 11 ragged", "gazutar", "w1024", prompts=11, lo=77, hi=1400),
        # ... and the exact serving mode: portions of prompts beside decoded tokens, everything in 32 bits
        _case("gazutar float32 mixed step", "gazutar", "w1024", "f32", prompts=3, lo=101, hi=400, past=130, decodes=13, past_lo=60, past_hi=700),
        # latent attention and linear attention: a prefill step at the larger size, a decode batch at the smaller one
        _case("felolorn prefill 8 x 1024", "felolorn", "w2048", prompts=8, lo=1024, hi=1024),
        _case("felolorn decode 24 ragged", "felolorn", "w1024", decodes=24, past_lo=30, past_hi=1500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dense decode", "dense decode", "dense prefill", "dense prefill", "moe", "gazutar", "gazutar", "gazutar f32",
                       "felolorn", "felolorn"])
    model = kind.split()[0]
    size = "" if model == "dense" else rng.choice(["w1024", "w2048"])
    weights = "f32" if kind.endswith("f32") else "fp8" if kind == "dense decode" and rng.random() < 0.25 else "bf16"
    c = _case(None, model, size, weights)
    del c["name"]
    if kind == "dense prefill":
        c["prompts"] = _log_int(rng, 1, 16)
        c["hi"] = _log_int(rng, 64, 1024)
        c["lo"] = rng.randint(max(1, c["hi"] // 4), c["hi"])
        c["past"] = rng.choice([0, 0, 16 * rng.randint(1, 20)])   # pages of a shared prefix that are in the cache already
        return c
    decode = model == "dense" or rng.random() < 0.5
    if decode:
        c["decodes"] = _log_int(rng, 1, 200 if model == "dense" else 64)
        c["past_hi"] = min(_log_int(rng, 100, 2047 if model == "dense" else 1500), 120000 // c["decodes"])
        c["past_lo"] = rng.randint(c["past_hi"] // 8 + 1, c["past_hi"])
        return c
    c["prompts"] = _log_int(rng, 1, 8)
    c["hi"] = _log_int(rng, 32, 400 if weights == "f32" else 1024)
    c["lo"] = rng.randint(max(1, c["hi"] // 8), c["hi"])
    if model != "moe" and rng.random() < 0.4:
        c["past"] = rng.randint(1, 300)
        c["decodes"] = rng.randint(0, 20)
        c["past_hi"] = rng.randint(100, 800)
        c["past_lo"] = rng.randint(20, c["past_hi"])
    return c


def sequences(case):
    """[(rows it has, rows the step brings)]: lengths spread over their range in no particular order, the same for every seed"""
    def spread(n, lo, hi):
        if n == 1:
            return [hi]
        return [lo + int(round((hi - lo) * ((0.5 + 0.618034 * i) % 1.0))) for i in range(n)]

    return [(case["past"], n) for n in spread(case["prompts"], case["lo"], case["hi"])] + \
           [(n, 1) for n in spread(case["decodes"], case["past_lo"], case["past_hi"])]


def dims(case):
    return dict(DENSE) if case["model"] == "dense" else dict(SIZES[case["size"]])


# ---------------------------------------------------------------------------------------------------------------------
# weights and inputs, made from the seed alone
# ---------------------------------------------------------------------------------------------------------------------
class _Draws:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.dtype = dtype

    def normal(self, *shape, std=1.0, mean=0.0, dtype=None):
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=self.g)
        return t.to(dtype or torch.float32)

    def mat(self, *shape, std=None):
        return self.normal(*shape, std=std if std is not None else shape[-1] ** -0.5, dtype=self.dtype)

    def uniform(self, *shape):
        return torch.rand(shape, dtype=torch.float32, device="cuda", generator=self.g)


def _routers(d, s, groups, keep, gain):
    """Routers and an embedding table that have a preference, as trained ones do: in every layer a token leans clearly towards
    `top` experts (spread over `keep` of `groups` groups), so that its choice does not hang on the last bits of its row.
    -> ([router of each layer], [vocab, width] table)"""
    W, E, top, V = s["width"], s["experts"], s["top"], s["vocab"]
    table = d.normal(V, W)
    routers = []
    per = E // groups
    for _ in range(s["layers"]):
        r = d.normal(E, W, std=W ** -0.5)
        routers.append((r * gain).to(d.dtype))
        kept = torch.rand(V, groups, device="cuda", generator=d.g).topk(keep, 1).indices
        each = top // keep
        for j in range(keep):
            ids = kept[:, j:j + 1] * per + torch.rand(V, per, device="cuda", generator=d.g).topk(each, 1).indices
            for k in range(each):
                table += 8.0 * r[ids[:, k]]
    return routers, table


def _qwen_weights(case, d):
    s, w = dims(case), {}
    W, H, G, D = s["width"], s["heads"], s["kv_heads"], s["dim"]
    moe = case["model"] == "moe"
    if moe:
        routers, table = _routers(d, s, 1, 1, 0.5)
        w["model.embed_tokens.weight"] = table.to(d.dtype)
        w["lm_head.weight"] = d.mat(s["vocab"], W)
    else:
        w["model.embed_tokens.weight"] = d.mat(s["vocab"], W, std=0.02)
    for i in range(s["layers"]):
        p = f"model.layers.{i}."
        w[p + "self_attn.qkv_proj.weight"] = d.mat((H + 2 * G) * D, W, std=0.02)
        w[p + "self_attn.o_proj.weight"] = d.mat(W, H * D, std=0.02)
        for n in ("self_attn.q_norm", "self_attn.k_norm"):
            w[p + n + ".weight"] = d.normal(D, mean=1.0, std=0.05, dtype=d.dtype)
        for n in ("input_layernorm", "post_attention_layernorm"):
            w[p + n + ".weight"] = d.normal(W, mean=1.0, std=0.05, dtype=d.dtype)
        if moe:
            w[p + "mlp.gate.weight"] = routers[i]
            w[p + "mlp.gate_up_stacked"] = d.mat(s["experts"], 2 * s["ff"], W, std=0.02)
            w[p + "mlp.down_stacked"] = d.mat(s["experts"], W, s["ff"], std=0.02)
        else:
            w[p + "mlp.gate_up_proj.weight"] = d.mat(2 * s["ff"], W, std=0.02)
            w[p + "mlp.down_proj.weight"] = d.mat(W, s["ff"], std=0.02)
    w["model.norm.weight"] = d.normal(W, mean=1.0, std=0.05, dtype=d.dtype)
    return w


def _expert_weights(w, p, d, s, router):
    E, ff, W = s["experts"], s["ff"], s["width"]
    w[p + "mlp.router"] = router
    w[p + "mlp.correction"] = d.normal(E, std=0.02)
    w[p + "mlp.gate"], w[p + "mlp.up"], w[p + "mlp.down"] = d.mat(E, ff, W), d.mat(E, ff, W), d.mat(E, W, ff)


def gazutar_config(s):
    att = {"type": "attention", "mixer": {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"],
                                          "mask": {"size": s["window"]}, "scale": s["dim"] ** -0.5, "v_mix": True}}
    rec = {"type": "channel_delta", "mixer": {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": s["dim"], "vdim": s["dim"],
                                              "conv": TAPS, "rank": s["width"] // 16}}
    ff = {"kind": "moe", "expert": {"ff": s["ff"]},
          "router": {"experts": s["experts"], "identity": 0, "top": s["top"], "groups": {"count": 4, "keep": 2}}}
    return {"architecture": "Gazutar", "vocab": s["vocab"], "width": s["width"], "logit_scale": 1.0, "norm": {"eps": EPS},
            "layers": [dict((rec, att)[i % 2], mlp=ff) for i in range(s["layers"])]}


def _gazutar_weights(case, d):
    s, w = dims(case), {}
    W, H, G, D = s["width"], s["heads"], s["kv_heads"], s["dim"]
    R = W // 16
    routers, table = _routers(d, s, 4, 2, 0.5)
    w["embed"], w["head"] = table.to(d.dtype), d.mat(s["vocab"], W)
    w["final_norm.weight"], w["final_norm.bias"] = d.normal(W, mean=1.0, std=0.05), d.normal(W, std=0.05)
    for i in range(s["layers"]):
        p = f"layers.{i}."
        for n in ("norm1", "norm2"):
            w[p + n + ".weight"], w[p + n + ".bias"] = d.normal(W, mean=0.25, std=0.02), d.normal(W, std=0.02)
        m = p + "mix."
        if i % 2:
            w[m + "qkvg.weight"] = d.mat((2 * H + 2 * G) * D, W)
            w[m + "q_norm"], w[m + "k_norm"] = d.normal(H * D, mean=1.0, std=0.05), d.normal(G * D, mean=1.0, std=0.05)
            w[m + "vmix"] = d.normal(1, mean=0.4, std=0.05)
        else:
            w[m + "qkv.weight"] = d.mat((2 * G + H) * D, W)
            w[m + "conv.weight"] = d.normal((2 * G + H) * D, TAPS, std=0.5)
            w[m + "low.weight"] = d.mat(2 * R + H, W)
            w[m + "a2"], w[m + "g2"] = d.mat(H * D, R), d.mat(H * D, R)
            w[m + "dt_bias"], w[m + "A_log"] = d.normal(H * D, mean=-1.0), d.normal(H, mean=-1.0, std=0.5)
            w[m + "norm"] = d.normal(D, mean=1.0, std=0.05)
        w[m + "o"] = d.mat(W, H * D)
        _expert_weights(w, p, d, s, routers[i])
    return w


FELOLORN_KINDS = ("hgrn2", "latent_attention", "lightning", "latent_attention")


def _decays(s):
    return [1.0 - 2.0 ** (-5 - 3 * h / s["heads"]) for h in range(s["heads"])]


def felolorn_config(s):
    W, D, H = s["width"], s["dim"], s["heads"]
    mixers = {"latent_attention": {"heads": H, "dim": D, "vdim": D, "kv_rank": 256, "q_rank": W // 2, "scale": D ** -0.5},
              "lightning": {"heads": H, "dim": D, "vdim": D, "decay": _decays(s)},
              "hgrn2": {"heads": H, "dim": D, "vdim": D}}
    moe = {"kind": "moe", "expert": {"ff": s["ff"]}, "router": {"experts": s["experts"], "top": s["top"], "groups": {"count": 4, "keep": 2}}}
    return {"architecture": "Felolorn", "vocab": s["vocab"], "width": W, "norm": {"eps": EPS}, "canon": {"taps": TAPS},
            "embedding": {"scale": W ** 0.5}, "logit_softcap": 30.0,
            "layers": [{"type": FELOLORN_KINDS[i % 4], "mixer": mixers[FELOLORN_KINDS[i % 4]], "mlp": moe} for i in range(s["layers"])]}


def _felolorn_weights(case, d):
    s, w = dims(case), {}
    W, H, D, C, Q = s["width"], s["heads"], s["dim"], 256, s["width"] // 2
    routers, table = _routers(d, s, 4, 2, 0.7)
    w["embed"], w["final_norm"] = (table * W ** -0.5).to(d.dtype), d.normal(W, mean=1.0, std=0.05)
    for i in range(s["layers"]):
        p, kind = f"layers.{i}.", FELOLORN_KINDS[i % 4]
        w[p + "norm1"], w[p + "norm2"] = d.normal(W, mean=1.0, std=0.05), d.normal(W, mean=1.0, std=0.05)
        w[p + "conv.weight"] = d.normal(W, TAPS, std=0.2)
        for n in ("out1", "out2"):
            w[p + n + ".gate"], w[p + n + ".gate_b"] = d.mat(W, W), d.normal(W, std=0.3)
            w[p + n + ".weight"] = d.normal(W, mean=0.25, std=0.02)
        m = p + "mix."
        if kind == "latent_attention":
            w[m + "qcg.weight"] = d.mat(Q + C, W)
            w[m + "q_norm"], w[m + "c_norm"] = d.normal(Q, mean=1.0, std=0.05), d.normal(C, mean=1.0, std=0.05)
            w[m + "uq"], w[m + "uk_t"], w[m + "uv"] = d.mat(H * D, Q), d.mat(H, C, D, std=C ** -0.5), d.mat(H, D, C)
            w[m + "sink"] = d.normal(H)
        elif kind == "lightning":
            w[m + "qkvg.weight"], w[m + "norm"] = d.mat(4 * H * D, W), d.normal(H * D, mean=1.0, std=0.05)
        else:
            w[m + "qfv.weight"], w[m + "norm"] = d.mat(3 * H * D, W), d.normal(D, mean=1.0, std=0.05)
            w[m + "f_bias"], w[m + "lower"] = d.normal(H * D, std=0.5), d.uniform(H * D) * 0.9
        w[m + "o"] = d.mat(W, H * D)
        _expert_weights(w, p, d, s, routers[i])
    return w


def inputs(case, seed):
    """(weights, {"ids": the tokens of every sequence, "table": page tables, "slots": state slots, "kv": filled pages})"""
    d = _Draws(seed, torch.float32 if case["weights"] == "f32" else torch.bfloat16)
    s, seqs, block = dims(case), sequences(case), BLOCK[case["model"]]
    w = {"dense": _qwen_weights, "moe": _qwen_weights, "gazutar": _gazutar_weights, "felolorn": _felolorn_weights}[case["model"]](case, d)
    pages = [-(-(a + n) // block) for a, n in seqs]
    total = sum(pages) + 1
    order = torch.randperm(total, device="cuda", generator=d.g).to(torch.int32).cpu()
    table = torch.full((len(seqs), max(pages)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    x = {"table": table.cuda(), "blocks": total,
         "ids": [torch.randint(0, s["vocab"], (a + n,), device="cuda", generator=d.g) for a, n in seqs],
         "slots": torch.randperm(len(seqs), device="cuda", generator=d.g).to(torch.int32)}
    if case["model"] in ("dense", "moe"):
        # keys are normed per head (unit root mean square), values are projections of normed rows; pages behind the step's own
        # rows hold what earlier steps left there
        kv = torch.empty((2, s["layers"], total, s["kv_heads"], block // 16, 16 * s["dim"]), dtype=torch.bfloat16, device="cuda")
        if any(a for a, _ in seqs):
            for i in range(s["layers"]):
                kv[0, i].normal_(0.0, 1.0, generator=d.g)
                kv[1, i].normal_(0.0, 0.6, generator=d.g)
        else:
            kv.zero_()
        x["kv"] = kv
    return w, x


# ---------------------------------------------------------------------------------------------------------------------
# the step
# ---------------------------------------------------------------------------------------------------------------------
def _load(model, w):
    from nanovllm.utils.loader import pack_model_weights

    own = dict(model.named_parameters())
    own.update(model.named_buffers())
    for name, t in w.items():
        assert own[name].shape == t.shape, (name, tuple(own[name].shape), tuple(t.shape))
        own[name].data.copy_(t)
    pack_model_weights(model)


def _capture(body):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        body()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="thread_local"):
        out = body()
    torch.cuda.synchronize()
    return graph, out


def _rows(seqs, x, block, past):
    """Metadata of the step that brings each sequence's new rows (past: the step that brought the rows before them)."""
    ids, pos, slots, cu, kv = [], [], [], [0], []
    table = x["table"].cpu()
    for i, (a, n) in enumerate(seqs):
        lo, hi = (0, a) if past else (a, a + n)
        p = torch.arange(lo, hi)
        ids.append(x["ids"][i][lo:hi])
        pos.append(p)
        slots.append(table[i, p // block].long() * block + p % block)
        cu.append(cu[-1] + hi - lo)
        kv.append(hi)
    i32 = dict(dtype=torch.int32, device="cuda")
    return dict(ids=torch.cat(ids).contiguous(), pos=torch.cat(pos).cuda(), slots=torch.cat(slots).to(**i32),
                cu=torch.tensor(cu, **i32), kv=torch.tensor(kv, **i32),
                max_q=max(b - a for a, b in zip(cu, cu[1:])), max_k=max(kv))


@torch.inference_mode()
def _prepare_qwen(case, w, x):
    from nanovllm.layers.linear import set_weight_quantization
    from nanovllm.models.models_map import model_dict
    from nanovllm.utils.context import reset_context, set_context

    s, seqs, block = dims(case), sequences(case), BLOCK[case["model"]]
    hf = dict(hidden_size=s["width"], num_hidden_layers=s["layers"], num_attention_heads=s["heads"], num_key_value_heads=s["kv_heads"],
              head_dim=s["dim"], intermediate_size=s["ff"], vocab_size=s["vocab"], max_position_embeddings=8192, rms_norm_eps=EPS,
              rope_theta=THETA, tie_word_embeddings=case["model"] == "dense", attention_bias=False, hidden_act="silu")
    if case["model"] == "moe":
        hf.update(intermediate_size=4 * s["width"], num_experts=s["experts"], num_experts_per_tok=s["top"],
                  moe_intermediate_size=s["ff"], decoder_sparse_step=1, mlp_only_layers=[], norm_topk_prob=True)
    set_weight_quantization("fp8" if case["weights"] == "fp8" else None)
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device("cuda"):
            model = model_dict["Qwen3MoeForCausalLM" if case["model"] == "moe" else "Qwen3ForCausalLM"](types.SimpleNamespace(**hf))
        model.eval()
        _load(model, w)
    finally:
        torch.set_default_dtype(torch.float32)
        set_weight_quantization(None)
    for i, layer in enumerate(model.model.layers):
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = x["kv"][0, i], x["kv"][1, i]
    st = {"model": model, "kv": x["kv"], "table": x["table"]}
    r = _rows(seqs, x, block, False)
    st["rows"] = r
    if case["decodes"]:
        n = len(seqs)
        st["slots"] = torch.stack([r["slots"] // block, r["slots"] % block], 1).contiguous()
        st["temps"], st["rng"] = torch.zeros(n, device="cuda"), torch.tensor([7, 1], dtype=torch.int64, device="cuda")
        st["tokens"] = torch.zeros(n, dtype=torch.int64, device="cuda")
        ctx = (False, dict(slot_mapping=st["slots"], context_lens=r["kv"], block_tables=x["table"], is_enforce_eager=False, real_bs=n,
                           block_size=block))

        def body():  # the served decode step: logits and, from the same pass, the greedy tokens (their arg-max)
            return model.lm_head.local_logits_pick(model(r["ids"], r["pos"]), st["temps"], st["rng"], st["tokens"])
    else:
        cu_k = torch.zeros_like(r["cu"])
        cu_k[1:] = torch.cumsum(r["kv"], 0)
        ctx = (True, dict(cu_seqlens_q=r["cu"], cu_seqlens_k=cu_k, max_seqlen_q=r["max_q"], max_seqlen_k=r["max_k"],
                          slot_mapping=r["slots"], block_tables=x["table"], block_size=block, kv_lens=r["kv"]))

        def body():
            return model.compute_logits(model(r["ids"], r["pos"]))
    if case["model"] == "dense" or case["decodes"]:
        set_context(ctx[0], **ctx[1])
        st["graph"], logits = _capture(body)
        reset_context()
        st["out"] = {"logits": logits, "kv": x["kv"]}
    else:
        st["eager"] = (ctx, body)
    return st


@torch.inference_mode()
def _prepare_hybrid(case, w, x):
    from nanovllm.models.felolorn import FelolornConfig, FelolornForCausalLM
    from nanovllm.models.gazutar import GazutarConfig, GazutarForCausalLM
    from nanovllm.utils.context import reset_context, set_context

    s, seqs, block = dims(case), sequences(case), BLOCK[case["model"]]
    dtype = torch.float32 if case["weights"] == "f32" else torch.bfloat16
    torch.set_default_dtype(dtype)
    try:
        with torch.device("cuda"):
            if case["model"] == "gazutar":
                model = GazutarForCausalLM(GazutarConfig(gazutar_config(s)))
            else:
                model = FelolornForCausalLM(FelolornConfig(felolorn_config(s)))
        model.eval()
        _load(model, w)
    finally:
        torch.set_default_dtype(torch.float32)
    model.bind_cache(x["blocks"], block, len(seqs) + 1, dtype, torch.device("cuda"))

    def context(r, table, slots):
        return dict(cu_seqlens_q=r["cu"], kv_lens=r["kv"], slot_mapping=r["slots"], block_tables=table, block_size=block,
                    state_slots=slots, max_seqlen_q=r["max_q"], max_seqlen_k=r["max_k"])

    # what the sequences have already: earlier steps of up to 8192 rows
    group, rows = [], 0
    for i, (a, _) in enumerate(seqs):
        if a:
            group.append(i)
            rows += a
        if group and (rows >= 8192 - 1536 or i + 1 == len(seqs)):
            sub = dict(table=x["table"][group], ids=[x["ids"][j] for j in group])
            r = _rows([seqs[j] for j in group], sub, block, True)
            set_context(True, **context(r, sub["table"].contiguous(), x["slots"][group].contiguous()))
            model(r["ids"])
            reset_context()
            group, rows = [], 0
    r = _rows(seqs, x, block, False)
    last = (r["cu"][1:] - 1).long()
    st = {"model": model, "rows": r, "table": x["table"], "slots": x["slots"], "last": last}
    ctx = (True, context(r, x["table"], x["slots"]))
    kept = []
    for l in model.layers:
        own = [l.conv.state] if case["model"] == "felolorn" else []
        if l.kind == "attention":
            own += [l.mix.k_cache, l.mix.v_cache]
        elif l.kind == "latent_attention":
            own += [l.mix.cache]
        elif l.kind == "channel_delta":
            own += [l.mix.conv_state, l.mix.state]
        else:
            own += [l.mix.state]
        kept.append(own)
    st["kept"] = kept
    if case["prompts"] == 0:
        set_context(ctx[0], **ctx[1])
        state = [t.clone() for own in kept for t in own]
        st["graph"], logits = _capture(lambda: model.compute_logits(model(r["ids"])))
        reset_context()
        for t, was in zip([t for own in kept for t in own], state):  # (the warm-up ran the step once)
            t.copy_(was)
        st["out"] = {"logits": logits, "kept": kept}
    else:
        st["eager"] = (ctx, lambda: model.compute_logits(model(r["ids"]), last))
    return st


def prepare(case, seed):
    w, x = inputs(case, seed)
    return (_prepare_qwen if case["model"] in ("dense", "moe") else _prepare_hybrid)(case, w, x)


@torch.inference_mode()
def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    from nanovllm.utils.context import reset_context, set_context

    (prefill, fields), body = state["eager"]
    set_context(prefill, **fields)
    logits = body()
    reset_context()
    return {"logits": logits, "kv": state["kv"]} if "kv" in state else {"logits": logits, "kept": state["kept"]}


# ---------------------------------------------------------------------------------------------------------------------
# what a step cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def work(case):
    s, seqs = dims(case), sequences(case)
    W, H, G, D, V, L = s["width"], s["heads"], s["kv_heads"], s["dim"], s["vocab"], s["layers"]
    T = sum(n for _, n in seqs)
    item = 4 if case["weights"] == "f32" else 2
    wide = 1 if case["weights"] == "fp8" else item
    def keys(window):  # (query, key) pairs, keys read from the cache, over all sequences
        pairs = sum(min(p + 1, window) for a, n in seqs for p in range(a, a + n))
        read = sum(min(a, window + n) for a, n in seqs)
        return pairs, read
    def experts():
        hit = s["experts"] * (1 - (1 - s["top"] / s["experts"]) ** T)
        return hit * 3 * W * s["ff"] + s["experts"] * W, T * (s["top"] * 3 * W * s["ff"] + s["experts"] * W)
    weights = macs = other = 0.0
    for i in range(L):
        if case["model"] in ("dense", "moe"):
            n = W * (2 * H + 2 * G) * D
            pairs, read = keys(1 << 30)
            macs += T * n + pairs * H * 2 * D
            other += (read + T) * 2 * G * D * 2
            weights += n
            if case["model"] == "dense":
                weights += 3 * W * s["ff"]
                macs += T * 3 * W * s["ff"]
        elif case["model"] == "gazutar":
            if i % 2:
                n = W * (3 * H + 2 * G) * D
                pairs, read = keys(s["window"])
                macs += pairs * H * 2 * D
                other += (read + T) * 2 * G * D * item
            else:
                R = W // 16
                n = W * (2 * H + 2 * G) * D + W * (2 * R + H) + 2 * R * H * D
                macs += T * H * 4 * D * D
                other += len(seqs) * H * D * D * 4 * (1 + (1 if any(a for a, _ in seqs) else 0))
            weights += n
            macs += T * n
        else:
            n = 2 * W * W
            if i % 2:
                C, Q = 256, W // 2
                n += W * (Q + C) + Q * H * D + H * C * 2 * D + H * D * W
                pairs, read = keys(1 << 30)
                macs += pairs * H * 2 * C
                other += (read + T) * C * item
            else:
                n += W * (4 if i % 4 == 0 else 5) * H * D
                macs += T * H * 3 * D * D
                other += len(seqs) * H * D * D * 4 * (1 + (1 if any(a for a, _ in seqs) else 0))
            weights += n
            macs += T * n
        if case["model"] != "dense":
            n, m = experts()
            weights += n
            macs += m
    weights += V * W
    macs += len(seqs) * V * W
    other += len(seqs) * V * (2 if case["model"] in ("dense", "moe") else 4)
    return {"bytes": weights * wide + other, "flops": 2 * macs}


def tolerance(case):
    """About four times what a step is off the 64-bit one: 1e-6 to 2e-6 in 32 bits; 0.003 to 0.006 over four layers of bf16
    products; 0.01 to 0.04 over the dense model's 28 layers, whose residual stream is bf16 too."""
    if case["weights"] == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["model"] == "dense":
        return {"rel": 0.03, "max": 0.9}
    return {"rel": 0.02, "max": 0.6}


# ---------------------------------------------------------------------------------------------------------------------
# the same step in 64 bits, in plain torch
# ---------------------------------------------------------------------------------------------------------------------
def _f8(w):
    """e4m3 with a power-of-two scale per row: a row's largest value lands in [128, 256)"""
    top = w.float().abs().amax(1, keepdim=True)
    e = torch.where(top > 0, torch.frexp(top)[1], torch.zeros_like(top, dtype=torch.int32))
    q = torch.ldexp(w.float(), 8 - e).to(torch.float8_e4m3fn).double()
    return torch.ldexp(q, e - 8)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu(z):
    return z * torch.sigmoid(z)


def _attend(q, k, v, scale, pos0, window=None, slope=None, sink=None):
    """q [n, H, D] at positions pos0.., k [m, G, D], v [m, G, Dv] at 0..m-1 -> [n, H, Dv]"""
    n, H, D = q.shape
    m, G = k.shape[0], k.shape[1]
    out = torch.empty(n, H, v.shape[-1], dtype=torch.float64, device=q.device)
    step = max(1, int(2e8) // max(1, m * H))
    for r in range(0, n, step):
        e = min(n, r + step)
        qq = q[r:e].view(e - r, G, H // G, D).permute(1, 2, 0, 3).reshape(G, -1, D)
        sc = (qq @ k.permute(1, 2, 0)).view(G, H // G, e - r, m).mul_(scale)
        dist = torch.arange(pos0 + r, pos0 + e, device=q.device).view(-1, 1) - torch.arange(m, device=q.device).view(1, -1)
        if slope is not None:
            sc -= slope.view(G, H // G, 1, 1) * dist
        sc.masked_fill_((dist < 0) | (dist >= (window or 1 << 30)), -math.inf)
        if sink is not None:
            sc = torch.cat([sc, sink.view(G, H // G, 1, 1).expand(G, H // G, e - r, 1)], -1)
        p = torch.softmax(sc, -1)[..., :m].reshape(G, -1, m)
        out[r:e] = (p @ v.permute(1, 0, 2)).view(G, H // G, e - r, -1).permute(2, 0, 1, 3).reshape(e - r, H, -1)
    return out


def _tile_maps(D=128):
    t, d = torch.arange(16, device="cuda").view(-1, 1), torch.arange(D, device="cuda").view(1, -1)
    k = (d // 32) * 512 + ((d % 32) // 8 * 16 + t) * 8 + d % 8
    v = (d // 32) * 512 + ((t // 4) * 16 + d % 16) * 8 + (d % 32) // 16 * 4 + t % 4
    return k, v


def _rope(x, pos):
    D = x.shape[-1]
    ang = pos.double().view(-1, 1, 1) / THETA ** (torch.arange(0, D, 2, device=x.device).double() / D)
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _top_experts(h, choice, scores, top, groups, keep, value):
    per = choice.shape[1] // groups
    grouped = choice.view(-1, groups, per)
    best = grouped.max(-1).values if value == "max" else grouped.topk(min(2, per), -1).values.sum(-1)
    kept = torch.zeros_like(best, dtype=torch.bool).scatter_(1, best.topk(keep, -1).indices, True)
    ids = choice.masked_fill(~kept.repeat_interleave(per, 1), -math.inf).topk(top, -1).indices
    return ids, scores.gather(1, ids)


def _mix_experts(h, ids, wts, gate, up, down):
    out = torch.zeros_like(h)
    for e in range(gate.shape[0]):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            x = h[t]
            y = (_silu(x @ gate[e].double().T) * (x @ up[e].double().T)) @ down[e].double().T
            out.index_add_(0, t, y * wts[t, k].unsqueeze(1))
    return out


def _exact_qwen(case, w, x):
    s, seqs, block = dims(case), sequences(case), BLOCK[case["model"]]
    H, G, D = s["heads"], s["kv_heads"], s["dim"]
    full = _f8 if case["weights"] == "fp8" else (lambda t: t.double())
    r = _rows(seqs, x, block, False)
    cu = r["cu"].tolist()
    h = full(w["model.embed_tokens.weight"])[r["ids"]] if case["weights"] == "fp8" else w["model.embed_tokens.weight"][r["ids"]].double()
    km, vm = _tile_maps(D)
    kv = x["kv"].double()
    tile, at = r["slots"].long() // 16, r["slots"].long() % 16
    heads = torch.arange(G, device="cuda").view(1, -1, 1)
    for i in range(s["layers"]):
        p = f"model.layers.{i}."
        f = _rms(h, w[p + "input_layernorm.weight"].double())
        qkv = f @ full(w[p + "self_attn.qkv_proj.weight"]).T
        q = qkv[:, :H * D].view(-1, H, D)
        k = qkv[:, H * D:(H + G) * D].view(-1, G, D)
        v = qkv[:, (H + G) * D:].view(-1, G, D)
        q = _rope(_rms(q, w[p + "self_attn.q_norm.weight"].double()), r["pos"])
        k = _rope(_rms(k, w[p + "self_attn.k_norm.weight"].double()), r["pos"])
        per = block // 16
        blk, sub = (tile // per).view(-1, 1, 1), (tile % per).view(-1, 1, 1)
        kv[0, i][blk, heads, sub, km[at].view(-1, 1, D)] = k
        kv[1, i][blk, heads, sub, vm[at].view(-1, 1, D)] = v
        o = torch.empty(q.shape[0], H, D, dtype=torch.float64, device="cuda")
        for j, (a, n) in enumerate(seqs):
            b = x["table"][j, :-(-(a + n) // block)].long()
            kk = kv[0, i][b][..., km].permute(0, 2, 3, 1, 4).reshape(-1, G, D)[:a + n]
            vv = kv[1, i][b][..., vm].permute(0, 2, 3, 1, 4).reshape(-1, G, D)[:a + n]
            o[cu[j]:cu[j + 1]] = _attend(q[cu[j]:cu[j + 1]], kk, vv, D ** -0.5, a)
        h = h + o.view(-1, H * D) @ full(w[p + "self_attn.o_proj.weight"]).T
        f = _rms(h, w[p + "post_attention_layernorm.weight"].double())
        if case["model"] == "moe":
            pr = torch.softmax(f @ w[p + "mlp.gate.weight"].double().T, -1)
            wts, ids = pr.topk(s["top"], -1)
            gu = w[p + "mlp.gate_up_stacked"]
            h = h + _mix_experts(f, ids, wts / wts.sum(-1, keepdim=True), gu[:, :s["ff"]], gu[:, s["ff"]:], w[p + "mlp.down_stacked"])
        else:
            g, u = (f @ full(w[p + "mlp.gate_up_proj.weight"]).T).chunk(2, -1)
            h = h + (_silu(g) * u) @ full(w[p + "mlp.down_proj.weight"]).T
    h = _rms(h[r["cu"][1:].long() - 1], w["model.norm.weight"].double())
    return {"logits": h @ full(w["lm_head.weight" if case["model"] == "moe" else "model.embed_tokens.weight"]).T, "kv": kv}


class _Ragged:
    """Whole sequences, one after another; recurrences walk them side by side, each to its own end."""

    def __init__(self, lens):
        self.lens, self.n, self.T = lens, len(lens), max(lens)
        self.cu = [0]
        for n in lens:
            self.cu.append(self.cu[-1] + n)

    def pad(self, x):
        out = torch.zeros((self.n, self.T) + x.shape[1:], dtype=x.dtype, device=x.device)
        for j, n in enumerate(self.lens):
            out[j, :n] = x[self.cu[j]:self.cu[j + 1]]
        return out

    def flat(self, x):
        return torch.cat([x[j, :n] for j, n in enumerate(self.lens)])

    def conv(self, x, w):
        """-> (causal convolution of every sequence, its last taps - 1 inputs)"""
        taps, out, tail = w.shape[1], torch.zeros_like(x), []
        for j in range(self.n):
            own = x[self.cu[j]:self.cu[j + 1]]
            padded = torch.cat([torch.zeros(taps - 1, x.shape[1], dtype=x.dtype, device=x.device), own])
            for t in range(taps):
                out[self.cu[j]:self.cu[j + 1]] += padded[t:t + own.shape[0]] * w[:, t]
            tail.append(padded[own.shape[0]:])
        return out, torch.stack(tail)

    def walk(self, S, step):
        """S <- step(S, t) for t = 0.. up to every sequence's end; -> (S, read-outs [rows, ..])"""
        outs, ends = [], torch.tensor(self.lens, device="cuda")
        whole = min(self.lens)
        for t in range(self.T):
            new, o = step(S, t)
            S = new if t < whole else torch.where((t < ends).view((-1,) + (1,) * (S.dim() - 1)), new, S)
            outs.append(o)
        return S, self.flat(torch.stack(outs, 1))


def _pages(case, x, seqs, rows, G, D):
    """rows [all rows, G, D] -> [blocks, G, block, D]"""
    block = BLOCK[case["model"]]
    out = torch.zeros(x["blocks"], G, block, D, dtype=torch.float64, device="cuda")
    at = 0
    for j, (a, n) in enumerate(seqs):
        p = torch.arange(a + n, device="cuda")
        out[x["table"][j, p // block].long(), :, p % block] = rows[at:at + a + n]
        at += a + n
    return out


def _in_slots(x, t):
    out = torch.zeros((t.shape[0] + 1,) + t.shape[1:], dtype=torch.float64, device="cuda")
    out[x["slots"].long()] = t
    return out


def _layer_norm(y, w, b):
    c = y - y.mean(-1, keepdim=True)
    return c * torch.rsqrt((c * c).mean(-1, keepdim=True) + EPS) * w + b


def _exact_gazutar(case, w, x):
    s, seqs = dims(case), sequences(case)
    W, H, G, D = s["width"], s["heads"], s["kv_heads"], s["dim"]
    R, rep = W // 16, H // G
    run_ = _Ragged([a + n for a, n in seqs])
    h = w["embed"][torch.cat(x["ids"])].double()
    kept, v_first = [], None
    slope = 2.0 ** (-8.0 * torch.arange(1, H + 1, device="cuda").double() / H)
    for i in range(s["layers"]):
        p = f"layers.{i}."
        f = {k[len(p):]: t for k, t in w.items() if k.startswith(p) and not k.startswith(p + "mlp")}
        f = {k: t.double() for k, t in f.items()}
        if i % 2:
            y = h @ f["mix.qkvg.weight"].T
            q, k, v, g = y.split([H * D, G * D, G * D, H * D], -1)
            q, k = _rms(q, f["mix.q_norm"]).view(-1, H, D), _rms(k, f["mix.k_norm"]).view(-1, G, D)
            if v_first is None:
                v_first = v
            else:
                v = (1 - f["mix.vmix"]) * v + f["mix.vmix"] * v_first
            v = v.reshape(-1, G, D)
            o = torch.cat([_attend(q[a:b], k[a:b], v[a:b], D ** -0.5, 0, s["window"], slope) for a, b in zip(run_.cu, run_.cu[1:])])
            y = (o.view(-1, H * D) * torch.sigmoid(g)) @ f["mix.o"].T
            kept.append([_pages(case, x, seqs, k, G, D), _pages(case, x, seqs, v, G, D)])
        else:
            c, tail = run_.conv(h @ f["mix.qkv.weight"].T, f["mix.conv.weight"])
            q, k, v = (t.view(-1, t.shape[-1] // D, D) for t in _silu(c).split([G * D, G * D, H * D], -1))
            q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
            k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            a1, g1, b = (h @ f["mix.low.weight"].T).split([R, R, H], -1)
            dt = torch.nn.functional.softplus(a1 @ f["mix.a2"].T + f["mix.dt_bias"]).view(-1, H, D)
            dec = torch.exp(-torch.exp(f["mix.A_log"]).view(1, H, 1) * dt)
            q, k = q.repeat_interleave(rep, 1), k.repeat_interleave(rep, 1)
            pq, pk, pv, pd, pb = (run_.pad(t) for t in (q, k, v, dec, torch.sigmoid(b)))

            def step(S, t):
                S = S * pd[:, t].unsqueeze(-1)
                u = pb[:, t].unsqueeze(-1) * (pv[:, t] - (pk[:, t].unsqueeze(-2) @ S).squeeze(-2))
                S = S + pk[:, t].unsqueeze(-1) * u.unsqueeze(-2)
                return S, (pq[:, t].unsqueeze(-2) @ S).squeeze(-2)

            S, o = run_.walk(torch.zeros(run_.n, H, D, D, dtype=torch.float64, device="cuda"), step)
            o = _rms(o, f["mix.norm"]) * torch.sigmoid(g1 @ f["mix.g2"].T).view(-1, H, D)
            y = o.reshape(-1, H * D) @ f["mix.o"].T
            # the state's own order: [head][32 value channels][key channel / 16][4][value channel][key channel / 4 % 4]
            S = S.view(run_.n, H, D // 16, 4, 4, D // 32, 32).permute(0, 1, 5, 2, 4, 6, 3).reshape(run_.n, -1)
            kept.append([_in_slots(x, tail), _in_slots(x, S)])
        h = h + _layer_norm(y, f["norm1.weight"], f["norm1.bias"])
        sc = torch.softmax(h @ w[p + "mlp.router"].double().T, -1)
        ids, wts = _top_experts(h, sc + w[p + "mlp.correction"].double(), sc, s["top"], 4, 2, "max")
        y = _mix_experts(h, ids, wts, w[p + "mlp.gate"], w[p + "mlp.up"], w[p + "mlp.down"])
        h = h + _layer_norm(y, f["norm2.weight"], f["norm2.bias"])
    last = torch.tensor(run_.cu[1:], device="cuda") - 1
    h = _layer_norm(h[last], w["final_norm.weight"].double(), w["final_norm.bias"].double())
    return {"logits": h @ w["head"].double().T, "kept": kept}


def _exact_felolorn(case, w, x):
    s, seqs = dims(case), sequences(case)
    W, H, D, C, Q = s["width"], s["heads"], s["dim"], 256, s["width"] // 2
    run_ = _Ragged([a + n for a, n in seqs])
    h = w["embed"][torch.cat(x["ids"])].double() * W ** 0.5
    kept = []
    for i in range(s["layers"]):
        p, kind = f"layers.{i}.", FELOLORN_KINDS[i % 4]
        f = {k[len(p):]: t.double() for k, t in w.items() if k.startswith(p) and not k.startswith(p + "mlp")}
        n = _rms(h, f["norm1"])
        gate = torch.sigmoid(n @ f["out1.gate"].T + f["out1.gate_b"])
        c, tail = run_.conv(n, f["conv.weight"])
        u = n + c
        own = [_in_slots(x, tail)]
        if kind == "latent_attention":
            cq, ckv = (u @ f["mix.qcg.weight"].T).split([Q, C], -1)
            q = (_rms(cq, f["mix.q_norm"]) @ f["mix.uq"].T).view(-1, H, D)
            lat = _rms(ckv, f["mix.c_norm"])
            qx = torch.einsum("thd,hcd->thc", q, f["mix.uk_t"])
            o = torch.cat([_attend(qx[a:b], lat[a:b].view(-1, 1, C), lat[a:b].view(-1, 1, C), D ** -0.5, 0, sink=f["mix.sink"])
                           for a, b in zip(run_.cu, run_.cu[1:])])
            y = torch.einsum("thc,hdc->thd", o, f["mix.uv"]).reshape(-1, H * D)
            own.append(_pages(case, x, seqs, lat.view(-1, 1, C), 1, C))
        else:
            if kind == "lightning":
                q, k, v, g = (u @ f["mix.qkvg.weight"].T).split(H * D, -1)
                q, k, v = _silu(q), _silu(k), _silu(v)
                dec = torch.tensor(_decays(s), dtype=torch.float64, device="cuda").view(1, H, 1).expand(q.shape[0], H, D)
            else:
                q, z, v = (u @ f["mix.qfv.weight"].T).split(H * D, -1)
                q = _silu(q)
                low = f["mix.lower"]
                dec = (low + (1 - low) * torch.sigmoid(z + f["mix.f_bias"])).view(-1, H, D)
                k = 1 - dec
            pq, pk, pv, pd = (run_.pad(t.reshape(-1, H, D)) for t in (q, k, v, dec))

            def step(S, t):
                S = S * pd[:, t].unsqueeze(-1) + pk[:, t].unsqueeze(-1) * pv[:, t].unsqueeze(-2)
                return S, (pq[:, t].unsqueeze(-2) @ S).squeeze(-2)

            S, o = run_.walk(torch.zeros(run_.n, H, D, D, dtype=torch.float64, device="cuda"), step)
            if kind == "lightning":
                y = _rms(o.reshape(-1, H * D), f["mix.norm"]) * torch.sigmoid(g)
            else:
                y = _rms(o, f["mix.norm"]).reshape(-1, H * D)
            # the state's own order: [head][32 value channels][key channel / 4][value channel][key channel % 4]
            own.append(_in_slots(x, S.view(run_.n, H, D // 4, 4, D // 32, 32).permute(0, 1, 4, 2, 5, 3).reshape(run_.n, -1)))
        kept.append(own)
        h = h + _rms(gate * (y @ f["mix.o"].T), f["out1.weight"])
        n = _rms(h, f["norm2"])
        gate = torch.sigmoid(n @ f["out2.gate"].T + f["out2.gate_b"])
        sc = torch.sigmoid(n @ w[p + "mlp.router"].double().T)
        ids, wts = _top_experts(n, sc + w[p + "mlp.correction"].double(), sc, s["top"], 4, 2, "top2")
        h = h + _rms(gate * _mix_experts(n, ids, wts, w[p + "mlp.gate"], w[p + "mlp.up"], w[p + "mlp.down"]), f["out2.weight"])
    last = torch.tensor(run_.cu[1:], device="cuda") - 1
    z = _rms(h[last], w["final_norm"].double()) @ w["embed"].double().T
    return {"logits": 30.0 * torch.tanh(z / 30.0), "kept": kept}


@torch.inference_mode()
def exact(case, seed):
    w, x = inputs(case, seed)
    f = {"dense": _exact_qwen, "moe": _exact_qwen, "gazutar": _exact_gazutar, "felolorn": _exact_felolorn}[case["model"]]
    return f(case, w, x)
