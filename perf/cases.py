"""
The serving work that is timed: one pass each of the steps and sublayers that the models of this framework run, at the
widths of their presets and comparison benchmarks, on random weights and inputs.

Kinds of case (``kind``):

* ``llama``     — a whole model step, ``CausalLM.forward`` + ``compute_logits`` + sampling, at the widths of the
                  llama3-8b preset with 4 of its 32 (identical) layers: a prompt batch, or a decode step replayed from the
                  hipGraph that a server keeps for its batch size.
* ``experts``   — the mixture-of-experts half of a layer: routing, experts, weighted sum into the residual with the norm that
                  rides in it. ``style``: mixtral (two of 8 wide experts), scaled, weighted, grouped (the three other mixtures).
* ``attention`` — grouped-query attention over the paged cache in its variants (``style``): over everything, in a window, in
                  chunks, with sigmoid weights, with capped scores and distance slopes, with a learned distance bias.
* ``latent``    — attention over compressed latent cache rows.
* ``recurrent`` — the linear recurrences with fp32 state per sequence (``style``): gated delta rule with a decay per head or per
                  channel, matrix LSTM, state space, linear attention with channel decays, decayed linear attention, scan.

Whole mixture models are not among the cases: at random weights, rounding differences between two correct programs flip routing
decisions, after which their logits can't be compared; the mixtures are measured where their input is given instead. For the
same reason a model step returns the logits and the cache it wrote, not the greedy tokens drawn from them.

``phase`` is prefill (eager, as a server runs prompt steps) or decode (one row per sequence, replayed from a hipGraph that is
captured beforehand, as a server does). ``seqs`` sequences have ``tokens`` new tokens each at most (with ``ragged`` between half of
that and all of it) behind ``past`` cached ones.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

DEV = "cuda"
BF = torch.bfloat16
BS = 16                 # tokens of a cache block
EPS = 1e-5
LLAMA_LAYERS = 4
LLAMA_CONTEXT = 2048    # longest sequence the decode graphs are built for

# width of the experts' model -> expert sizes of each style (experts, identity entries, chosen, expert width, groups, kept groups)
EXPERTS = {
    ("mixtral", 4096): (8, 0, 2, 14336, 1, 1),
    ("scaled", 2048): (8, 0, 2, 2048, 1, 1), ("scaled", 4096): (8, 0, 2, 4096, 1, 1),
    ("weighted", 2048): (8, 2, 2, 2048, 1, 1), ("weighted", 4096): (8, 2, 2, 4096, 1, 1),
    ("grouped", 2048): (16, 0, 4, 1024, 4, 2), ("grouped", 4096): (32, 0, 4, 2048, 8, 4),
}
# style -> heads per 2048 of width, key groups (0: one per head), key size, value size
RECURRENT = {
    "delta": (16, 4, 128, 128), "delta_channel": (16, 4, 128, 128), "lstm": (16, 0, 64, 128), "state_space": (64, 1, 128, 64),
    "linear_channel": (16, 0, 64, 128), "lightning": (16, 0, 128, 128), "scan": (4096, 0, 16, 1),
}


# ------------------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # one user waits for the next token of a short dialogue: the smallest call, bound by latency
        {"name": "llama-decode-1", "kind": "llama", "phase": "decode", "seqs": 1, "tokens": 1, "past": 130, "ragged": False},
        # the serving benchmark's decode step: 32 requests of 512-token prompts, in the middle of their answers
        {"name": "llama-decode-32", "kind": "llama", "phase": "decode", "seqs": 32, "tokens": 1, "past": 576, "ragged": True},
        # the serving benchmark's prompt step: 32 prompts of 512 tokens at once
        {"name": "llama-prefill-32x512", "kind": "llama", "phase": "prefill", "seqs": 32, "tokens": 512, "past": 0, "ragged": False},
        # a prompt step of the Mixtral preset: 8 prompts of 512 tokens through one layer's experts
        {"name": "experts-mixtral-4096", "kind": "experts", "style": "mixtral", "phase": "prefill", "width": 4096, "rows": 4096},
        # an odd number of prompt tokens through 16 small squared-ReLU experts, four chosen out of two of four groups
        {"name": "experts-grouped-8191", "kind": "experts", "style": "grouped", "phase": "prefill", "width": 2048, "rows": 8191},
        # a decode step of 32 requests through clamped gated experts, two of the ten choices being identities
        {"name": "experts-weighted-32", "kind": "experts", "style": "weighted", "phase": "decode", "width": 2048, "rows": 32},
        # ragged prompts of up to 1024 tokens, each key seen for a window of 512
        {"name": "attention-window-16x1024", "kind": "attention", "style": "window", "phase": "prefill", "width": 2048, "vdim": 128,
         "seqs": 16, "tokens": 1024, "past": 0, "ragged": True},
        # a decode step of 32 requests at ragged contexts around 1500, every key visible
        {"name": "attention-decode-32", "kind": "attention", "style": "full", "phase": "decode", "width": 2048, "vdim": 128,
         "seqs": 32, "tokens": 1, "past": 2000, "ragged": True},
        # prompts of 1024 tokens over latent cache rows
        {"name": "latent-16x1024", "kind": "latent", "phase": "prefill", "width": 2048, "window": 0, "seqs": 16, "tokens": 1024,
         "past": 0, "ragged": False},
        # prompts through a state-space layer's recurrence: 64 heads of 128 x 64
        {"name": "state-space-16x1024", "kind": "recurrent", "style": "state_space", "phase": "prefill", "width": 2048,
         "seqs": 16, "tokens": 1024, "past": 0, "ragged": False},
        # ragged prompts through the gated delta rule with a decay per channel
        {"name": "delta-channel-16x1000", "kind": "recurrent", "style": "delta_channel", "phase": "prefill", "width": 2048,
         "seqs": 16, "tokens": 1000, "past": 0, "ragged": True},
        # a decode step of 32 requests through decayed linear attention
        {"name": "lightning-decode-32", "kind": "recurrent", "style": "lightning", "phase": "decode", "width": 2048,
         "seqs": 32, "tokens": 1, "past": 700, "ragged": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, most):
    """Sequences, new tokens, cached tokens and raggedness of a step with at most ``most`` new tokens."""
    if rng.random() < 0.4:
        return {"phase": "decode", "seqs": _log(rng, 1, 64), "tokens": 1, "past": _log(rng, 8, 2000), "ragged": rng.random() < 0.7}
    seqs = _log(rng, 1, 32)
    tokens = _log(rng, 16, max(32, min(1500, most // seqs)))
    return {"phase": "prefill", "seqs": seqs, "tokens": tokens, "past": rng.choice([0, 0, 0, _log(rng, 16, 500)]),
            "ragged": rng.random() < 0.7}


def draw(rng):
    kind = rng.choice(["llama", "llama", "experts", "experts", "experts", "attention", "attention", "latent", "recurrent", "recurrent",
                       "recurrent"])
    if kind == "llama":
        return {"kind": kind, **_batch(rng, 16384)}
    if kind == "experts":
        style, width = rng.choice(sorted(EXPERTS))
        decode = rng.random() < 0.4
        most = 4096 if style == "mixtral" else 16384 if width == 2048 else 8192
        return {"kind": kind, "style": style, "phase": "decode" if decode else "prefill", "width": width,
                "rows": _log(rng, 1, 128) if decode else _log(rng, 129, most)}
    width = rng.choice([2048, 4096])
    most = 16384 if width == 2048 else 8192
    if kind == "attention":
        style = rng.choice(["full", "window", "chunk", "sigmoid", "capped", "bias"])
        return {"kind": kind, "style": style, "width": width, "vdim": rng.choice([128, 128, 256]), **_batch(rng, most)}
    if kind == "latent":
        return {"kind": kind, "width": width, "window": rng.choice([0, 512]), **_batch(rng, most)}
    return {"kind": kind, "style": rng.choice(sorted(RECURRENT)), "width": width, **_batch(rng, most)}


# ------------------------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, mean=0.0, dt=torch.float32):
    t = torch.empty(*shape, dtype=dt, device=DEV)
    return t.normal_(mean, std, generator=g)


def _spans(c):
    """(new tokens, cached tokens) of every sequence."""
    n, t, p = c["seqs"], c["tokens"], c["past"]
    if not c["ragged"]:
        return [(t, p)] * n
    return [(t - (i * 37) % (t // 2 + 1), p - (i * 53) % (p // 2 + 1)) for i in range(n)]


def _step(c, seed):
    """The step's index tensors: positions, row offsets, lengths, scattered cache pages and the slots of the new rows."""
    spans = _spans(c)
    q = torch.tensor([a for a, _ in spans], dtype=torch.int64, device=DEV)
    past = torch.tensor([b for _, b in spans], dtype=torch.int64, device=DEV)
    cu = torch.zeros(len(spans) + 1, dtype=torch.int64, device=DEV)
    cu[1:] = q.cumsum(0)
    T = sum(a for a, _ in spans)
    seq = torch.repeat_interleave(torch.arange(len(spans), device=DEV), q, output_size=T)
    pos = torch.arange(T, device=DEV) - cu[seq] + past[seq]
    pages = max(-(-(a + b) // BS) for a, b in spans)
    perm = torch.randperm(len(spans) * pages, device=DEV, generator=_gen(seed + 7))
    bt = perm.view(len(spans), pages)
    return {"T": T, "S": len(spans), "pos": pos, "seq": seq, "cu": cu.int(), "ctx": (q + past).int(), "bt": bt.int().contiguous(),
            "blocks": len(spans) * pages, "slots": bt[seq, pos // BS] * BS + pos % BS, "max_q": max(a for a, _ in spans),
            "cu_or_none": None if c["phase"] == "decode" else cu.int()}


def _llama_weights(arch, seed):
    g = _gen(seed)
    h, d = arch.hidden_size, arch.head_dim
    w = {"model.embed_tokens.weight": _randn(g, arch.vocab_size, h, dt=BF), "model.norm.weight": torch.ones(h, dtype=BF, device=DEV),
         "lm_head.weight": _randn(g, arch.vocab_size, h, std=0.02, dt=BF)}
    for i in range(arch.num_layers):
        p = f"model.layers.{i}."
        for name, rows, cols, std in (("self_attn.q_proj", arch.num_heads * d, h, 0.02), ("self_attn.k_proj", arch.num_kv_heads * d, h, 0.02),
                                      ("self_attn.v_proj", arch.num_kv_heads * d, h, 0.02), ("self_attn.o_proj", h, arch.num_heads * d, 0.01),
                                      ("mlp.gate_proj", arch.intermediate_size, h, 0.02), ("mlp.up_proj", arch.intermediate_size, h, 0.02),
                                      ("mlp.down_proj", h, arch.intermediate_size, 0.01)):
            w[p + name + ".weight"] = _randn(g, rows, cols, std=std, dt=BF)
        for name in ("input_layernorm", "post_attention_layernorm"):
            w[p + name + ".weight"] = torch.ones(h, dtype=BF, device=DEV)
    return w


def _llama_inputs(c, arch, seed):
    st = _step(c, seed)
    g = _gen(seed + 1)
    ids = torch.randint(3, arch.vocab_size, (st["T"],), device=DEV, generator=g)
    shape = (arch.num_layers, 2, st["blocks"], arch.num_kv_heads, BS, arch.head_dim)
    return st, ids, _randn(g, *shape, dt=BF)


def _expert_inputs(c, seed):
    E, ident, K, ff, groups, keep = EXPERTS[c["style"], c["width"]]
    g, H, T = _gen(seed), c["width"], c["rows"]
    gated = c["style"] != "grouped"
    return {"x": _randn(g, T, H, dt=BF), "resid": _randn(g, T, H), "router": _randn(g, E + ident, H, std=0.03, dt=BF),
            "w13": _randn(g, E, 2 * ff if gated else ff, H, std=0.02, dt=BF), "w2": _randn(g, E, H, ff, std=0.02, dt=BF),
            "norm": _randn(g, H, std=0.1, mean=0.0, dt=BF) if gated else _randn(g, H, std=0.1, mean=1.0),
            "corr": _randn(g, E + ident, std=0.02), "gating": _randn(g, T, E, dt=BF)}


def _attention_inputs(c, seed):
    H = c["width"] // 128
    G, D, V = H // 4, 128, c["vdim"]
    st, g = _step(c, seed), _gen(seed)
    style, kw = c["style"], {}
    if style == "chunk":
        kw.update(seg=512, sink=torch.zeros(H, device=DEV))
    if style == "sigmoid":
        kw.update(sigmoid=True, head_bias=_randn(g, H, std=0.5, mean=-5.0))
    if style == "capped":
        kw.update(softcap=30.0, slopes=torch.exp2(-8.0 * torch.arange(1, H + 1, device=DEV) / H))
    if style == "bias":
        kw.update(bias=_randn(g, 130, H, std=0.5), sink=_randn(g, H))
    window = {"window": 512, "sigmoid": 512, "capped": 1024, "bias": 1024}.get(style, 0)
    q = _randn(g, st["T"], H * D, dt=BF)
    cache = _randn(g, st["blocks"], BS, G * (D + V), dt=BF)
    return st, q, cache, (H, G, D, V, window, D ** -0.5), kw


LATENT = (256, 32, 96)   # latent width, rotated dims, dims of a head before them


def _latent_inputs(c, seed):
    rank, rot, dim = LATENT
    H, st, g = c["width"] // 128, _step(c, seed), _gen(seed)
    freq = (10000.0 ** (-2.0 * torch.arange(rot // 2, dtype=torch.float64) / rot)).float().to(DEV)
    return {"st": st, "H": H, "q_lat": _randn(g, H, st["T"], rank, dt=BF), "q": _randn(g, st["T"], H * (dim + rot), dt=BF),
            "cache": _randn(g, st["blocks"], BS, rank + rot, dt=BF), "sink": _randn(g, H), "freq": freq, "scale": (dim + rot) ** -0.5}


def _recurrent_inputs(c, seed):
    heads, groups, D, V = RECURRENT[c["style"]]
    f = c["width"] // 2048
    H, G = heads * f, groups * f if groups > 1 else groups or heads * f
    st, g, style = _step(c, seed), _gen(seed), c["style"]
    T, S = st["T"], st["S"]
    d = {"st": st, "H": H, "G": G, "D": D, "V": V, "state": _randn(g, S + 1, H, D, V, std=0.3), "slots": torch.randperm(S, device=DEV, generator=g).int()}
    if style in ("delta", "delta_channel"):
        qk = F.normalize(_randn(g, T, 2 * G, D), dim=-1)
        qk[:, :G] *= D ** -0.5
        beta = torch.sigmoid(_randn(g, T, H))
        d["qkv"] = torch.cat([qk.reshape(T, 2 * G * D), F.silu(_randn(g, T, H * V))], 1)
        d["gate"], d["norm"] = _randn(g, T, H * V, dt=BF), _randn(g, V, std=0.1, mean=1.0)
        d["A_log"], d["bg"] = _randn(g, H, std=0.5), beta
        if style == "delta":
            dec = torch.exp(-torch.exp(d["A_log"]) * F.softplus(_randn(g, T, H, std=0.7, mean=-2.5)))
            d["bg"] = torch.cat([beta, dec], 1)
        else:
            d["z"], d["z_bias"] = _randn(g, T, H * D, std=0.5, dt=BF), _randn(g, H * D, std=0.7, mean=-2.5)
    elif style == "scan":
        I, N = H, D
        d["state"] = d["state"].view(S + 1, I, N)
        d["x"], d["dt"], d["z"] = (_randn(g, T, I, dt=BF) for _ in range(3))
        d["dt_bias"], d["bc"] = _randn(g, I, std=0.7, mean=-3.0), _randn(g, T, 2 * N, dt=BF)
        d["A"], d["Dskip"] = -torch.arange(1, N + 1, device=DEV).float().expand(I, N).contiguous(), torch.ones(I, device=DEV)
    else:
        d["x"] = _randn(g, T, 2 * G * D + H * V, dt=BF)
        if style == "lstm":
            d["ab"] = torch.stack([torch.sigmoid(_randn(g, T, H, mean=3.0)), torch.sigmoid(_randn(g, T, H)), torch.ones(T, H, device=DEV)], 2)
            d["n_state"] = _randn(g, S + 1, H, D, std=0.3)
        elif style == "state_space":
            dt = F.softplus(_randn(g, T, H, mean=-3.0))
            d["ab"] = torch.stack([torch.exp(-torch.exp(_randn(g, H, std=0.5)) * dt), dt], 2)
        elif style == "linear_channel":
            d["z"], d["z_bias"] = _randn(g, T, H * D, std=0.5, dt=BF), _randn(g, H * D, mean=1.0)
        else:
            d["decay"] = torch.exp(-torch.exp2(-8.0 * torch.arange(1, H + 1, device=DEV) / H))
    return d


# ----------------------------------------------------------------------------------------------------------------- prepare
def _captured(c, call, mutable):
    """The pass itself: ``call`` for a prompt step; for a decode step the replay of its hipGraph."""
    if c["phase"] != "decode":
        return call
    keep = [t.clone() for t in mutable]
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for t, k in zip(mutable, keep):
        t.copy_(k)

    return _Replay(graph, call, out)


class _Replay:
    """A captured step. It keeps ``call`` with all that the recorded kernels read: a graph holds addresses, not tensors."""

    def __init__(self, graph, call, out):
        self.graph, self.call, self.out = graph, call, out

    def __call__(self):
        self.graph.replay()
        return self.out


def prepare(case, seed):
    with torch.inference_mode():
        return {"llama": _prepare_llama, "experts": _prepare_experts, "attention": _prepare_attention, "latent": _prepare_latent,
                "recurrent": _prepare_recurrent}[case["kind"]](case, seed)


def run(state):
    with torch.inference_mode():
        return state()


def _llama_arch():
    from src.models.presets import get_preset

    return get_preset("llama3-8b", num_layers=LLAMA_LAYERS)


def _prepare_llama(c, seed):
    from src import ops
    from src.models.llama import AttnMetadata, CausalLM
    from src.ops.gemm_table import enable_prefill_gemm_table

    enable_prefill_gemm_table(torch.device(DEV))
    arch = _llama_arch()
    model = CausalLM(arch, DEV, max_position=LLAMA_CONTEXT)
    model.load_state_dict(_llama_weights(arch, seed))
    st, ids, pool = _llama_inputs(c, arch, seed)
    n, f32, i32 = st["S"], torch.float32, torch.int32
    scratch = model.alloc_decode_scratch(max(32, n))
    if c["phase"] == "prefill":
        last = (st["cu"][1:] - 1).long()
        meta = AttnMetadata(is_prefill=True, slot_mapping=st["slots"], block_tables=st["bt"], ctx_lens=st["ctx"], cu_q=st["cu"],
                            max_q_len=st["max_q"], keep_rows=last)

        def call():
            hidden = model.forward(ids, st["pos"], meta, pool)
            if hidden.shape[0] != n:   # a small step keeps every row
                hidden = hidden.index_select(0, last)
            logits = model.compute_logits(hidden)
            ops.sample(logits)
            return {"logits": logits, "cache": pool}

        return call
    parts = ops.decode_partials(LLAMA_CONTEXT)
    amax = torch.zeros(n, model.lm_head_argmax_parts(), 2, dtype=i32, device=DEV)
    samp = (torch.zeros(n * 32, dtype=i32, device=DEV), torch.zeros(n, dtype=i32, device=DEV))
    tables = F.pad(st["bt"], (0, LLAMA_CONTEXT // BS - st["bt"].shape[1]))   # as wide as the longest sequence needs
    meta = AttnMetadata(is_prefill=False, slot_mapping=st["slots"], block_tables=tables, ctx_lens=st["ctx"], max_ctx=LLAMA_CONTEXT,
                        part_o=torch.empty(n * model.hq * parts * 128, dtype=f32, device=DEV),
                        part_ml=torch.empty(n * model.hq * parts * 2, dtype=f32, device=DEV),
                        attn_cnt=torch.zeros(n * model.hkv, dtype=i32, device=DEV), scratch=scratch)
    greedy = torch.zeros(n, dtype=f32, device=DEV)
    zero, ones, zero64 = torch.zeros(n, dtype=i32, device=DEV), torch.ones(n, dtype=f32, device=DEV), torch.zeros(n, dtype=torch.int64, device=DEV)

    def call():
        hidden = model.forward(ids, st["pos"], meta, pool)
        logits = model.compute_logits(hidden, argmax_parts=amax)
        ops.sample(logits, greedy, zero, ones, zero64, zero64, scratch=samp, lm_part=amax)
        return {"logits": logits, "cache": pool}

    return _captured(c, call, ())


def _prepare_experts(c, seed):
    from src import ops
    from src.ops import mix

    E, ident, K, ff, groups, keep = EXPERTS[c["style"], c["width"]]
    d = _expert_inputs(c, seed)
    x, resid, act = d["x"], d["resid"], torch.empty_like(d["x"])
    if c["style"] == "mixtral":
        return _captured(c, lambda: {"out": ops.moe_forward(x, d["w13"], d["w2"], d["gating"], K)}, ())
    if c["style"] == "scaled":
        def call():
            w, ids = mix.route_sigmoid_topk(x, d["router"], K)
            mix.moe_input_scaled(x, d["w13"], d["w2"], w, ids, post_norm=(resid, d["norm"], EPS, True, act))
            return {"resid": resid, "act": act}
    elif c["style"] == "weighted":
        def call():
            w, ids, _ = mix.route_softmax_topk(x, d["router"], K, E + ident, d["corr"])
            mix.moe_output_weighted(x, d["w13"], d["w2"], w, ids, mix.ACT_CLAMPED, 7.0, 1.702, n_route=E + ident,
                                    post_norm=(resid, d["norm"], EPS, True, act, 0.3))
            return {"resid": resid, "act": act}
    else:
        def call():
            w, ids = mix.route_grouped_topk(x, d["router"], K, groups, keep, 2.5)
            mix.moe_output_weighted(x, d["w13"], d["w2"], w, ids, mix.ACT_RELU2, 0.0, 0.0, pre_norm=(resid, d["norm"], EPS, act))
            return {"resid": resid, "act": act}
    return _captured(c, call, (resid,))


def _prepare_attention(c, seed):
    from src.ops import seq

    st, q, cache, (H, G, D, V, window, scale), kw = _attention_inputs(c, seed)
    kw = dict(kw)
    sink, bias = kw.pop("sink", None), kw.pop("bias", None)
    return _captured(c, lambda: {"out": seq.sink_attn(q, cache, st["bt"], st["cu_or_none"], st["ctx"], st["pos"], sink, bias, st["max_q"],
                                                      H, G, D, V, window, scale, **kw)}, ())


def _prepare_latent(c, seed):
    from src.ops import mix

    d, (rank, rot, dim) = _latent_inputs(c, seed), LATENT
    st = d["st"]
    return _captured(c, lambda: {"out": mix.latent_attn(d["q_lat"], d["q"], dim, d["cache"], st["bt"], st["cu_or_none"], st["ctx"], st["pos"],
                                                        d["sink"], st["max_q"], c["window"], d["scale"], rot, d["freq"])}, ())


def _prepare_recurrent(c, seed):
    from src.ops import lin, rec, seq

    d, style = _recurrent_inputs(c, seed), c["style"]
    st, H, G, D, V, state = d["st"], d["H"], d["G"], d["D"], d["V"], d["state"]
    rag = seq.Ragged(st["pos"], st["cu_or_none"], d["slots"])
    mutable = [state]
    if style in ("delta", "delta_channel"):
        chan = {k: d[k] for k in ("z", "z_bias", "A_log")} if style == "delta_channel" else {}

        def call():
            return {"out": seq.gated_delta(d["qkv"], d["bg"], d["gate"], d["norm"], EPS, state, H, G, D, V, rag, **chan), "state": state}
    elif style == "scan":
        def call():
            return {"out": rec.selective_scan(d["x"], d["dt"], d["dt_bias"], d["bc"], 0, D, d["A"], d["Dskip"], d["z"], state, rag), "state": state}
    elif style == "lightning":
        def call():
            return {"out": lin.lightning_attn(d["x"], 0, H * D, 2 * H * D, d["decay"], state, H, D, V, rag), "state": state}
    else:
        n_state = d.get("n_state")
        if n_state is not None:
            mutable.append(n_state)

        def call():
            o, nq = rec.gated_linear_attn(d["x"], 0, G * D, 2 * G * D, d.get("ab"), state, n_state, H, G, D, V, D ** -0.5, rag,
                                          z=d.get("z"), z_bias=d.get("z_bias"), tau=16.0)
            return {"out": o, "nq": nq, "state": state, "n_state": n_state}
    return _captured(c, call, mutable)


# -------------------------------------------------------------------------------------------------------------------- work
def _pairs(c, window=0, seg=0):
    """Visible (query, key) pairs, and cached rows that some query of the step sees."""
    pairs = rows = 0
    for a, b in _spans(c):
        lo = [max(max(0, p - window + 1) if window else 0, p // seg * seg if seg else 0) for p in range(b, b + a)]
        pairs += sum(p - first + 1 for p, first in zip(range(b, b + a), lo))
        rows += a + b - lo[0]
    return pairs, rows


def work(case):
    c = case
    if c["kind"] == "experts":
        E, _, K, ff, _, _ = EXPERTS[c["style"], c["width"]]
        T, H, mats = c["rows"], c["width"], 2 if c["style"] == "grouped" else 3
        io = T * H * (4 if c["style"] == "mixtral" else 12)
        return {"bytes": min(E, T * K) * mats * H * ff * 2 + io, "flops": 2 * T * K * mats * H * ff}
    T = sum(a for a, _ in _spans(c))
    if c["kind"] == "llama":
        arch = _llama_arch()
        h, d = arch.hidden_size, arch.head_dim
        layer = h * (2 * arch.num_heads + 2 * arch.num_kv_heads) * d + 3 * h * arch.intermediate_size
        pairs, rows = _pairs(c)
        flops = arch.num_layers * (2 * layer * T + 4 * pairs * arch.num_heads * d) + 2 * c["seqs"] * h * arch.vocab_size
        return {"bytes": 2 * (arch.num_layers * layer + arch.vocab_size * h) + rows * arch.num_layers * 4 * arch.num_kv_heads * d
                + 2 * T * h + 2 * c["seqs"] * arch.vocab_size, "flops": flops}
    H = c["width"] // 128
    if c["kind"] == "attention":
        style, V = c["style"], c["vdim"]
        window = {"window": 512, "sigmoid": 512, "capped": 1024, "bias": 1024}.get(style, 0)
        pairs, rows = _pairs(c, window, 512 if style == "chunk" else 0)
        return {"bytes": 2 * (rows * (H // 4) * (128 + V) + T * H * (128 + V)), "flops": 2 * pairs * H * (128 + V)}
    if c["kind"] == "latent":
        rank, rot, dim = LATENT
        pairs, rows = _pairs(c, c["window"])
        return {"bytes": 2 * (rows * (rank + rot) + T * H * (2 * rank + rot)), "flops": 2 * pairs * H * (2 * rank + rot)}
    heads, groups, D, V = RECURRENT[c["style"]]
    f = c["width"] // 2048
    H, G = heads * f, groups * f if groups > 1 else groups or heads * f
    state = 4 * c["seqs"] * H * D * V * (2 if c["past"] else 1)
    if c["style"] in ("delta", "delta_channel"):
        io = T * (4 * (2 * G * D + H * V) + 4 * H * V + (2 * H * D if c["style"] == "delta_channel" else 4 * H))
        return {"bytes": io + state, "flops": 7 * T * H * D * V}
    if c["style"] == "scan":
        return {"bytes": T * 8 * H + state, "flops": 6 * T * H * D}
    io = T * (2 * (2 * G * D + H * V) + 4 * H * V + {"lstm": 12 * H, "state_space": 8 * H, "linear_channel": 2 * H * D}.get(c["style"], 0))
    return {"bytes": io + state, "flops": 4 * T * H * D * V}


def tolerance(case):
    """About four times the measured distance from :func:`exact`: bf16 results of one sublayer are 0.002 - 0.004 off, those of the four
    layers of a model step 0.009; the recurrences with fp32 results are 1e-7 off (sums in another order: 1e-6)."""
    if case["kind"] == "llama":
        return {"rel": 3e-2}
    if case["kind"] == "recurrent" and case["style"] in ("lstm", "state_space", "linear_channel"):
        return {"rel": 1e-5}
    return {"rel": 1.5e-2 if case["kind"] == "experts" else 1e-2}


# ------------------------------------------------------------------------------------------------------------------- exact
def exact(case, seed):
    with torch.inference_mode():
        return {"llama": _exact_llama, "experts": _exact_experts, "attention": _exact_attention, "latent": _exact_latent,
                "recurrent": _exact_recurrent}[case["kind"]](case, seed)


def _norm(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w


def _exact_llama(c, seed):
    arch = _llama_arch()
    w = _llama_weights(arch, seed)
    st, ids, pool = _llama_inputs(c, arch, seed)
    pool, pos, T = pool.double(), st["pos"], st["T"]
    hq, hkv, d = arch.num_heads, arch.num_kv_heads, arch.head_dim
    ang = pos.double()[:, None] * (arch.rope_theta ** (-torch.arange(d // 2, dtype=torch.float64, device=DEV) / (d // 2)))
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def turn(x):
        a, b = x[..., : d // 2], x[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def proj(x, name):
        return x @ w[name + ".weight"].double().t()

    x = w["model.embed_tokens.weight"][ids].double()
    for i in range(arch.num_layers):
        p = f"model.layers.{i}."
        h = _norm(x)
        q = turn(proj(h, p + "self_attn.q_proj").view(T, hq, d))
        k, v = turn(proj(h, p + "self_attn.k_proj").view(T, hkv, d)), proj(h, p + "self_attn.v_proj").view(T, hkv, d)
        pool[i, 0, st["slots"] // BS, :, st["slots"] % BS] = k
        pool[i, 1, st["slots"] // BS, :, st["slots"] % BS] = v
        o = torch.empty(T, hq, d, dtype=torch.float64, device=DEV)
        for s in range(st["S"]):
            a, b, n = int(st["cu"][s]), int(st["cu"][s + 1]), int(st["ctx"][s])
            rows = pool[i][:, st["bt"][s].long()].permute(0, 2, 1, 3, 4).reshape(2, hkv, -1, d)[:, :, :n].repeat_interleave(hq // hkv, 1)
            sc = torch.matmul(q[a:b].transpose(0, 1), rows[0].transpose(1, 2).contiguous()) * d ** -0.5
            sc.masked_fill_(torch.arange(n, device=DEV)[None, None] > pos[a:b][None, :, None], -math.inf)
            o[a:b] = torch.matmul(torch.softmax(sc, -1), rows[1]).transpose(0, 1)
        x = x + proj(o.reshape(T, hq * d), p + "self_attn.o_proj")
        h = _norm(x)
        x = x + proj(F.silu(proj(h, p + "mlp.gate_proj")) * proj(h, p + "mlp.up_proj"), p + "mlp.down_proj")
    last = (st["cu"][1:] - 1).long()
    return {"logits": proj(_norm(x[last]), "lm_head"), "cache": pool}


def _exact_experts(c, seed):
    E, ident, K, ff, groups, keep = EXPERTS[c["style"], c["width"]]
    d, style = _expert_inputs(c, seed), c["style"]
    x, T = d["x"].double(), c["rows"]

    def best(s, k):   # the k largest, the lowest index first among equals
        return torch.sort(s, dim=-1, descending=True, stable=True)[1][:, :k]

    if style == "mixtral":
        p = torch.softmax(d["gating"].double(), -1)
        ids = best(p, K)
        w = p.gather(1, ids)
        w = w / w.sum(-1, keepdim=True)
    else:
        z = x @ d["router"].double().t()
        if style == "scaled":
            p = torch.sigmoid(z)
            ids = best(p, K)
            w = p.gather(1, ids)
        elif style == "weighted":
            p = torch.softmax(z, -1)
            ids = best(p + d["corr"].double(), K)
            w = p.gather(1, ids)
            w = w / (w.sum(-1, keepdim=True) + 1e-20)
        else:
            p = torch.softmax(z, -1)
            top = best(p.view(T, groups, E // groups).amax(-1), keep)
            is_open = torch.zeros(T, groups, dtype=torch.bool, device=DEV).scatter_(1, top, True).repeat_interleave(E // groups, 1)
            ids = best(p.masked_fill(~is_open, -1.0), K)
            w = 2.5 * p.gather(1, ids)
    y = torch.zeros_like(x)
    for e in range(E + ident):
        t, j = (ids == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        we, xe = w[t, j][:, None], x[t]
        if e >= E:
            y.index_add_(0, t, we * xe)
            continue
        w13, w2 = d["w13"][e].double().t(), d["w2"][e].double().t()
        if style == "scaled":
            xe, we = we * xe, 1.0
        u = xe @ w13
        if style == "grouped":
            u = torch.relu(u) ** 2
        elif style == "weighted":
            a = u[:, :ff].clamp(max=7.0)
            u = a * torch.sigmoid(1.702 * a) * (u[:, ff:].clamp(-7.0, 7.0) + 1.0)
        else:
            u = F.silu(u[:, :ff]) * u[:, ff:]
        y.index_add_(0, t, we * (u @ w2))
    if style == "mixtral":
        return {"out": y}
    resid = d["resid"].double()
    if style == "grouped":
        resid = resid + y
        return {"resid": resid, "act": _norm(resid, d["norm"].double())}
    resid = resid + (0.3 if style == "weighted" else 1.0) * _norm(y, 1.0 + d["norm"].double())
    return {"resid": resid, "act": resid}


def _exact_attention(c, seed):
    st, q, cache, (H, G, D, V, window, scale), kw = _attention_inputs(c, seed)
    out = torch.empty(st["T"], H, V, dtype=torch.float64, device=DEV)
    for s in range(st["S"]):
        a, b, n = int(st["cu"][s]), int(st["cu"][s + 1]), int(st["ctx"][s])
        rows = cache.view(-1, G, BS, D + V)[st["bt"][s].long()].permute(1, 0, 2, 3).reshape(G, -1, D + V)[:, :n].double()
        rows = rows.repeat_interleave(H // G, 0)
        sc = torch.matmul(q[a:b].double().view(-1, H, D).transpose(0, 1), rows[..., :D].transpose(1, 2).contiguous()) * scale
        p, j = st["pos"][a:b][:, None], torch.arange(n, device=DEV)[None, :]
        seen = (j <= p) & ((p - j < window) if window else (j >= 0))
        if "seg" in kw:
            seen &= j // kw["seg"] == p // kw["seg"]
        if "softcap" in kw:
            sc = kw["softcap"] * torch.tanh(sc / kw["softcap"]) - kw["slopes"].double()[:, None, None] * (p - j)[None]
        if "bias" in kw:
            sc = sc + kw["bias"].double()[(p - j).clamp(0, kw["bias"].shape[0] - 1)].permute(2, 0, 1)
        if "sigmoid" in kw:
            wgt = torch.sigmoid(sc + kw["head_bias"].double()[:, None, None]).masked_fill(~seen[None], 0.0)
        else:
            sc = sc.masked_fill(~seen[None], -math.inf)
            if "sink" in kw:
                sc = torch.cat([sc, kw["sink"].double()[:, None, None].expand(H, b - a, 1)], -1)
            wgt = torch.softmax(sc, -1)[..., :n]
        out[a:b] = torch.matmul(wgt, rows[..., D:].contiguous()).transpose(0, 1)
    return {"out": out.reshape(st["T"], H * V)}


def _exact_latent(c, seed):
    d, (rank, rot, dim) = _latent_inputs(c, seed), LATENT
    st, H = d["st"], d["H"]
    ang = st["pos"].double()[:, None] * d["freq"].double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    qr = d["q"].double().view(st["T"], H, dim + rot)[..., dim:]
    qr = torch.stack([qr[..., 0::2] * cos - qr[..., 1::2] * sin, qr[..., 1::2] * cos + qr[..., 0::2] * sin], -1).flatten(-2).transpose(0, 1)
    q = torch.cat([d["q_lat"].double(), qr], -1)
    out = torch.empty(H, st["T"], rank, dtype=torch.float64, device=DEV)
    for s in range(st["S"]):
        a, b, n = int(st["cu"][s]), int(st["cu"][s + 1]), int(st["ctx"][s])
        rows = d["cache"][st["bt"][s].long()].reshape(-1, rank + rot)[:n].double()
        p, j = st["pos"][a:b][:, None], torch.arange(n, device=DEV)[None, :]
        seen = (j <= p) & ((p - j < c["window"]) if c["window"] else (j >= 0))
        sc = (torch.matmul(q[:, a:b], rows.t().contiguous()) * d["scale"]).masked_fill(~seen[None], -math.inf)
        sc = torch.cat([sc, d["sink"].double()[:, None, None].expand(H, b - a, 1)], -1)
        out[:, a:b] = torch.matmul(torch.softmax(sc, -1)[..., :n], rows[:, :rank].contiguous())
    return {"out": out}


def _exact_recurrent(c, seed):
    d, style = _recurrent_inputs(c, seed), c["style"]
    st, H, G, D, V = d["st"], d["H"], d["G"], d["D"], d["V"]
    T, S, rep = st["T"], st["S"], H // G
    rows = d["state"].double()
    cu, slots = st["cu"].tolist(), d["slots"].long()
    order = sorted(range(S), key=lambda s: cu[s] - cu[s + 1])         # the longest first: the live ones stay a prefix
    first = torch.tensor([cu[s] for s in order], device=DEV)
    slot = slots[torch.tensor(order, device=DEV)]
    fresh = st["pos"][first] == 0
    live = rows[slot].masked_fill(fresh.view(-1, *[1] * (rows.dim() - 1)), 0.0)
    nrm = d["n_state"].double() if "n_state" in d else None
    live_n = nrm[slot].masked_fill(fresh[:, None, None], 0.0) if nrm is not None else None
    if style == "scan":
        dt = F.softplus(d["dt"].double() + d["dt_bias"].double())
        x, B, C, A = d["x"].double(), d["bc"][:, :D].double(), d["bc"][:, D:].double(), d["A"].double()
        out = torch.empty(T, H, dtype=torch.float64, device=DEV)
    else:
        src = d["qkv"].double() if "qkv" in d else d["x"].double()
        if style == "lightning":
            src = F.silu(src)
        q, k = (src[:, i * G * D: (i + 1) * G * D].view(T, G, D) for i in (0, 1))
        v = src[:, 2 * G * D:].view(T, H, V)
        beta = torch.ones(T, H, dtype=torch.float64, device=DEV)
        if style in ("delta", "delta_channel"):
            beta = d["bg"][:, :H].double()
        elif "ab" in d:
            beta = d["ab"][..., 1].double()
        if style == "delta":
            dec = d["bg"][:, H:].double()[..., None]
        elif style == "delta_channel":
            dec = torch.exp(-torch.exp(d["A_log"].double())[:, None] * F.softplus(d["z"].double() + d["z_bias"].double()).view(T, H, D))
        elif style == "linear_channel":
            dec = torch.exp(F.logsigmoid(d["z"].double() + d["z_bias"].double()) / 16.0).view(T, H, D)
        elif style == "lightning":
            dec = d["decay"].double().expand(T, H)[..., None]
        else:
            dec = d["ab"][..., 0].double()[..., None]
        if style not in ("delta", "delta_channel", "lightning"):
            q = q * D ** -0.5
        out = torch.empty(T, H, V, dtype=torch.float64, device=DEV)
        nq = torch.empty(T, H, dtype=torch.float64, device=DEV) if nrm is not None else None
    for i in range(st["max_q"]):
        n = sum(1 for s in order if cu[s + 1] - cu[s] > i)
        t = first[:n] + i
        if style == "scan":
            live[:n] = torch.exp(dt[t][..., None] * A) * live[:n] + (dt[t] * x[t])[..., None] * B[t][:, None, :]
            out[t] = (live[:n] * C[t][:, None, :]).sum(-1)
            continue
        kt, qt = k[t].repeat_interleave(rep, 1), q[t].repeat_interleave(rep, 1)
        live[:n] *= dec[t][..., None]
        u = v[t]
        if "qkv" in d:
            u = u - (live[:n] * kt[..., None]).sum(2)
        live[:n] += kt[..., None] * (beta[t][..., None] * u)[:, :, None, :]
        out[t] = (live[:n] * qt[..., None]).sum(2)
        if nrm is not None:
            live_n[:n] = dec[t] * live_n[:n] + beta[t][..., None] * kt
            nq[t] = (live_n[:n] * qt).sum(-1)
    rows[slot] = live
    if style == "scan":
        return {"out": (out + d["Dskip"].double() * x) * F.silu(d["z"].double()), "state": rows}
    if "qkv" in d:
        gate = d["gate"].double().view(T, H, V)
        out = _norm(out, d["norm"].double()) * F.silu(gate)
    out = out.reshape(T, H * V)
    if "qkv" in d or style == "lightning":
        return {"out": out, "state": rows}
    if nrm is not None:
        nrm[slot] = live_n
    return {"out": out, "nq": nq, "state": rows, "n_state": nrm}
