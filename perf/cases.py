"""Performance cases of the gated-delta verify path and the hybrid target.

Each case is one call (or short call sequence) that a program using this
package makes: the gated-delta scan and chunked prefill ops, the layer body,
the LM head with its greedy accept, a draft block through the target, the
device-driven verify step and the prompt pass.  Sizes are the package's own
configurations (Qwen3.5-4B shapes: hidden 2560, 16 key / 32 value heads of
128, MLP 9216, vocabulary 151936) and generic ones around them.  Models have
at most one period of four layers (three gated-delta, one attention): rounding
differences grow with depth, and a period holds every kernel of the full
depth.  Weights are random, at the scale of the package's random init.

``listed`` / ``draw`` give cases, ``prepare`` what a program holds before the
call, ``run`` one pass, ``work`` the bytes and operations it cannot do
without, ``tolerance`` the spread of correct implementations and ``exact`` the
same outputs in fp64 from plain torch.
"""
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "dflash-mlx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

BF, F32, F64, I32 = torch.bfloat16, torch.float32, torch.float64, torch.int32
HIDDEN, MLP, VOCAB = 2560, 9216, 151936
HK, HV, D, CONV_K = 16, 32, 128, 4        # gated-delta heads
HQ, HKV, ROT, THETA = 16, 4, 32, 100000.0  # attention heads
CONV = 2 * HK * D + HV * D
EPS = 1e-6


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # a block of 16 drafts through one small layer: launch latency
        {"name": "scan-small", "kind": "scan", "B": 1, "T": 16, "Hk": 4, "Hv": 4, "D": 64},
        # the scans of a 24-layer target's block, stacked: the state tape's bytes
        {"name": "scan-24-layers", "kind": "scan", "B": 24, "T": 16, "Hk": 16, "Hv": 32, "D": 128},
        # the gated-delta layer body between its projections, four sequences
        {"name": "layer-b4", "kind": "layer", "B": 4, "T": 16},
        # the linear-attention scan of a long prompt, and of a few short ragged ones
        {"name": "prefill-8k", "kind": "prefill", "B": 1, "T": 8192, "Hk": 16, "Hv": 32},
        {"name": "prefill-b3-ragged", "kind": "prefill", "B": 3, "T": 777, "Hk": 16, "Hv": 32},
        # verification by logits: head over a block, then the greedy accept
        {"name": "head-logits-16", "kind": "head", "B": 1, "N": 16, "V": VOCAB, "fused": False},
        # verification without logits, four sequences' blocks
        {"name": "head-fused-64", "kind": "head", "B": 4, "N": 16, "V": VOCAB, "fused": True},
        # a draft block through the target (logits, hidden states, rollback) after a long prompt
        {"name": "verify-block", "kind": "verify", "T": 16, "past": 4096},
        # the graph-replayed serving step for four sequences of different lengths
        {"name": "step-b4", "kind": "step", "B": 4, "T": 16, "past": 3000},
        # a short chat turn's prompt, and a document's
        {"name": "prompt-short", "kind": "prompt", "P": 120, "past": 0, "attn": False},
        {"name": "prompt-4k", "kind": "prompt", "P": 4096, "past": 0, "attn": False},
        # an attention layer of a prompt that goes on after a long cached prefix
        {"name": "attn-long", "kind": "prompt", "P": 2048, "past": 14336, "attn": True},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["scan", "layer", "prefill", "head", "verify", "step", "prompt", "attn"])
    if kind == "scan":
        hk, hv = rng.choice([(4, 4), (4, 8), (8, 16), (16, 16), (16, 32)])
        d = rng.choice([64, 96, 128, 128])
        return {"kind": kind, "B": _log(rng, 1, 24), "T": rng.randint(1, 16), "Hk": hk, "Hv": hv, "D": d}
    if kind == "layer":
        return {"kind": kind, "B": _log(rng, 1, 16), "T": rng.randint(2, 16)}
    if kind == "prefill":
        b = rng.randint(1, 4)
        hk, hv = rng.choice([(4, 8), (8, 16), (16, 32)])
        return {"kind": kind, "B": b, "T": _log(rng, 65, 8192 // b), "Hk": hk, "Hv": hv}
    if kind == "head":
        return {"kind": kind, "B": rng.randint(1, 4), "N": rng.randint(1, 16),
                "V": 16 * _log(rng, 2000, VOCAB // 16), "fused": rng.random() < 0.5}
    if kind == "verify":
        return {"kind": kind, "T": rng.randint(1, 16), "past": _log(rng, 17, 8192)}
    if kind == "step":
        return {"kind": kind, "B": rng.randint(1, 4), "T": rng.randint(2, 16), "past": _log(rng, 64, 8192)}
    if kind == "prompt":
        return {"kind": "prompt", "P": _log(rng, 17, 4096), "past": rng.choice([0, _log(rng, 17, 2048)]),
                "attn": False}
    return {"kind": "prompt", "P": _log(rng, 256, 2048), "past": _log(rng, 64, 14336), "attn": True}


# ------------------------------------------------------------------ the inputs

def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + salt)


def _rand(gen, *shape, std=1.0, dtype=BF):
    return (torch.randn(*shape, generator=gen, device="cuda", dtype=F32) * std).to(dtype)


def _unit(x):
    return (x / torch.linalg.vector_norm(x, dim=-1, keepdim=True).clamp_min(1e-12)).to(BF)


def _scan_inputs(seed, B, T, Hk, Hv, Dh):
    """Normalised q and k rows, values, decays and gates of a trained layer's
    ranges, and a state of earlier tokens."""
    g = _gen(seed)
    q = _unit(_rand(g, B, T, Hk, Dh, dtype=F32))
    k = _unit(_rand(g, B, T, Hk, Dh, dtype=F32))
    v = _rand(g, B, T, Hv, Dh)
    decay = torch.exp(-torch.nn.functional.softplus(_rand(g, B, T, Hv, dtype=F32)))
    beta = torch.sigmoid(_rand(g, B, T, Hv, dtype=F32))
    state = _rand(g, B, Hv, Dh, Dh, std=0.05, dtype=F32)
    return [q, k, v, decay, beta, state]


def _linear_params(g):
    return {"conv_w": _rand(g, CONV, CONV_K, std=0.5),
            "A_log": torch.log((torch.rand(HV, generator=g, device="cuda") * 16).clamp_min(1e-4)),
            "dt_bias": torch.ones(HV, dtype=BF, device="cuda"),
            "norm": torch.ones(D, dtype=BF, device="cuda")}


def _layer_inputs(case, seed):
    g = _gen(seed, 1)
    B, T = case["B"], case["T"]
    return {"qkv": _rand(g, B, T, CONV), "z": _rand(g, B, T, HV * D), "a": _rand(g, B, T, HV),
            "b": _rand(g, B, T, HV), "conv": _rand(g, B, CONV_K - 1, CONV),
            "state": _rand(g, B, HV, D, D, std=0.05, dtype=F32), "p": _linear_params(g)}


def _head_inputs(case, seed):
    """Hidden rows whose next token stands out, as a trained head's does, and
    drafts that agree with it for a while."""
    g = _gen(seed, 2)
    B, N, V = case["B"], case["N"], case["V"]
    weight = _rand(g, V, HIDDEN, std=0.02)
    toks = torch.randint(0, V, (B, N), generator=g, device="cuda")
    hidden = (_rand(g, B, N, HIDDEN, dtype=F32) + 8.0 * weight[toks].float()).to(BF)
    agree = torch.randint(0, N + 1, (B, 1), generator=g, device="cuda")
    pos = torch.arange(N, device="cuda")[None]
    draft = torch.where(pos < agree, toks, (toks + 1) % V)[:, :max(N - 1, 1)].to(I32)
    return weight, hidden, draft


def _model_weights(seed, attn_only):
    """Raw weights of one period (three gated-delta layers and an attention
    layer), or of a single attention layer."""
    g = _gen(seed, 3)
    ones = lambda n: torch.ones(n, dtype=BF, device="cuda")  # noqa: E731
    layers = []
    for linear in ([False] if attn_only else [True, True, True, False]):
        lw = {"ln_in": ones(HIDDEN), "ln_post": ones(HIDDEN),
              "w_gu": _rand(g, 2 * MLP, HIDDEN, std=0.02), "w_down": _rand(g, HIDDEN, MLP, std=0.02)}
        if linear:
            lw["w_in"] = _rand(g, CONV + HV * D + 2 * HV, HIDDEN, std=0.02)
            lw["w_out"] = _rand(g, HIDDEN, HV * D, std=0.02)
            lw["p"] = _linear_params(g)
        else:
            lw["w_qkv"] = _rand(g, (2 * HQ + 2 * HKV) * D, HIDDEN, std=0.02)
            lw["w_o"] = _rand(g, HIDDEN, HQ * D, std=0.02)
            lw["q_norm"], lw["k_norm"] = ones(D), ones(D)
        layers.append(lw)
    vocab = 8192 if attn_only else VOCAB
    return {"embed": _rand(g, vocab, HIDDEN, std=0.02), "final": ones(HIDDEN),
            "lm_head": _rand(g, vocab, HIDDEN, std=0.02), "layers": layers}


def _tokens(seed, n, vocab):
    g = _gen(seed, 4)
    return torch.randint(0, vocab, (n,), generator=g, device="cuda", dtype=I32)


def _step_caches(case, seed):
    """Cache contents of ragged sequences: lengths, conv windows, states, keys, values."""
    g = _gen(seed, 5)
    B, past = case["B"], case["past"]
    lens = [max(1, past - (past * b) // 7) for b in range(B)]
    conv = [_rand(g, B, CONV_K - 1, CONV) for _ in range(3)]
    rec = [_rand(g, B, HV, D, D, std=0.05, dtype=F32) for _ in range(3)]
    keys, vals = _rand(g, B, HKV, past, D), _rand(g, B, HKV, past, D)
    toks = torch.randint(0, VOCAB, (B, case["T"]), generator=g, device="cuda", dtype=I32)
    return lens, conv, rec, keys, vals, toks


def _config(attn_only, vocab):
    from dflash_mlx.hybrid_model import HybridConfig

    if attn_only:
        return HybridConfig(num_hidden_layers=1, full_attention_interval=1, vocab_size=vocab)
    return HybridConfig(num_hidden_layers=4, vocab_size=vocab)


def _hybrid_weights(w):
    from dflash_mlx.gdn_layer import GatedDeltaWeights
    from dflash_mlx.hybrid_model import HybridWeights

    layers = []
    for lw in w["layers"]:
        d = {k: v for k, v in lw.items() if k != "p"}
        if "p" in lw:
            p = lw["p"]
            d["gdn"] = GatedDeltaWeights(conv_weight=p["conv_w"], A_log=p["A_log"],
                                         dt_bias=p["dt_bias"], norm_weight=p["norm"])
        layers.append(d)
    return HybridWeights(embed=w["embed"], final_norm=w["final"], lm_head=w["lm_head"], layers=layers)


# ------------------------------------------------------------------ the calls

def prepare(case, seed):
    import dflash_mlx

    kind = case["kind"]
    if kind == "scan":
        return {"kind": kind, "x": _scan_inputs(seed, case["B"], case["T"], case["Hk"], case["Hv"], case["D"])}
    if kind == "prefill":
        x = _scan_inputs(seed, case["B"], case["T"], case["Hk"], case["Hv"], D)
        need = dflash_mlx.chunked_prefill_workspace_bytes(case["B"], case["T"], case["Hv"])
        return {"kind": kind, "x": x, "ws": torch.empty(need, dtype=torch.uint8, device="cuda")}
    if kind == "layer":
        from dflash_mlx.gdn_layer import GatedDeltaConfig, GatedDeltaWeights

        x = _layer_inputs(case, seed)
        p = x.pop("p")
        return {"kind": kind, "x": x, "cfg": GatedDeltaConfig(),
                "w": GatedDeltaWeights(conv_weight=p["conv_w"], A_log=p["A_log"], dt_bias=p["dt_bias"],
                                       norm_weight=p["norm"])}
    if kind == "head":
        from dflash_mlx.hybrid_model import HybridConfig, HybridWeights
        from dflash_mlx.target import HybridTargetModel

        weight, hidden, draft = _head_inputs(case, seed)
        w = HybridWeights(embed=weight, final_norm=torch.ones(HIDDEN, dtype=BF, device="cuda"),
                          lm_head=weight, layers=[], lm_head_tiled=dflash_mlx.tile_weight(weight))
        model = HybridTargetModel(HybridConfig(vocab_size=case["V"]), w, torch.device("cuda", 0))
        return {"kind": kind, "fused": case["fused"], "model": model, "hidden": hidden, "draft": draft}
    if kind == "step":
        from dflash_mlx.hybrid_model import HybridVerifyRunner

        w = _model_weights(seed, False)
        lens, conv, rec, keys, vals, toks = _step_caches(case, seed)
        smax = -(-(case["past"] + 2 * case["T"]) // 64) * 64
        run_ = HybridVerifyRunner(_config(False, VOCAB), _hybrid_weights(w), case["B"], case["T"], smax,
                                  torch.device("cuda", 0))
        run_.set_state(lens=lens, conv=conv, rec=rec, k=[keys], v=[vals])
        run_.capture_step()
        return {"kind": kind, "run": run_, "toks": toks, "lens": run_.lens.clone(),
                "conv": run_.conv_all.clone()}
    # verify / prompt: the target behind its model interface, a prefix in its caches
    from dflash_mlx.adapters import LoadedTargetModel
    from dflash_mlx.target import HybridTargetModel

    attn = kind == "prompt" and case["attn"]
    n = case["T"] if kind == "verify" else case["P"]
    past = case["past"]
    w = _model_weights(seed, attn)
    vocab = w["embed"].shape[0]
    model = HybridTargetModel(_config(attn, vocab), _hybrid_weights(w), torch.device("cuda", 0),
                              max_seq_len=past + n)
    target = LoadedTargetModel(model=model)
    cache = target.make_cache()
    toks = _tokens(seed, past + n, vocab)
    ids = [0] if attn else [1, 3]
    if past:
        model.forward_dflash(toks[None, :past], cache, ids)
    snap = target.snapshot_linear_caches(cache)
    return {"kind": kind, "target": target, "cache": cache, "toks": toks[None, past:].contiguous(),
            "ids": ids, "past": past, "snap": snap}


def _appended(cache, past):
    """Keys and values that the call added to the attention layers."""
    return [t for i in cache.attn_idx for t in (cache[i].keys[:, :, past:], cache[i].values[:, :, past:])]


def run(state):
    import dflash_mlx

    kind = state["kind"]
    if kind == "scan":
        return dflash_mlx.gated_delta_verify(*state["x"])
    if kind == "prefill":
        return dflash_mlx.gated_delta_prefill(*state["x"], workspace=state["ws"])
    if kind == "layer":
        from dflash_mlx.gdn_layer import gdn_layer_verify

        x = state["x"]
        y, conv, final, tape, _ = gdn_layer_verify(x["qkv"], x["z"], x["a"], x["b"], x["conv"], x["state"],
                                                   state["w"], state["cfg"])
        return [y, conv, final, tape]
    if kind == "head":
        model = state["model"]
        if state["fused"]:
            return list(dflash_mlx.lm_head_greedy_accept(
                state["hidden"], model.weights.lm_head, state["draft"],
                weight_tiled=model.weights.lm_head_tiled))
        logits = model.lm_head_logits(state["hidden"])
        return [logits, *dflash_mlx.greedy_accept(logits, state["draft"])]
    if kind == "step":
        # the block again from the same caches: lengths, windows and keep counts put back
        r = state["run"]
        r.lens.copy_(state["lens"])
        r.conv_all.copy_(state["conv"])
        r.keep.zero_()
        r.tokens.copy_(state["toks"])
        r.replay()
        return [r.xn, *r.tape]
    target, cache, toks, past = state["target"], state["cache"], state["toks"], state["past"]
    if kind == "verify":
        # a block of drafts, all of them refused, so that the caches stand as before
        logits, hidden, records = target.forward_with_hidden_states(
            toks, cache, state["ids"], return_rollback_records=True)
        outs = [logits, hidden, *[records[i]["state_tape"] for i in cache.linear_idx], *_appended(cache, past)]
        target.rewind_kv_caches(cache, toks.shape[1])
        target.rollback_linear_caches(cache, records, 0)
        return outs
    # a prompt on the cached prefix; then the caches go back to the prefix
    logits, hidden = target.forward_accept_all_block(toks, cache, state["ids"])
    outs = [logits, hidden, *[cache[i][1] for i in cache.linear_idx], *_appended(cache, past)]
    target.rewind_kv_caches(cache, toks.shape[1])
    target.restore_linear_caches(cache, state["snap"])
    return outs


# ------------------------------------------------------------------ the work

def _layer_params(linear):
    mixer = (CONV + HV * D + 2 * HV + HV * D) if linear else ((2 * HQ + 2 * HKV) * D + HQ * D)
    return HIDDEN * (mixer + 3 * MLP)


def work(case):
    kind = case["kind"]
    state = 4 * HV * D * D  # one sequence's fp32 state
    if kind in ("scan", "prefill"):
        B, T, hk, hv, d = case["B"], case["T"], case["Hk"], case["Hv"], case.get("D", D)
        io = 2 * B * T * (2 * hk * d + 2 * hv * d) + 8 * B * T * hv
        slabs = T + 2 if kind == "scan" else 2
        return {"bytes": io + 4 * B * hv * d * d * slabs, "flops": 8 * B * T * hv * d * d}
    if kind == "layer":
        B, T = case["B"], case["T"]
        return {"bytes": 2 * B * T * (CONV + 2 * HV * D + 2 * HV) + 8 * B * (CONV_K - 1) * CONV // 2
                + B * state * (T + 2), "flops": 8 * B * T * HV * D * D}
    if kind == "head":
        rows, V = case["B"] * case["N"], case["V"]
        return {"bytes": 2 * V * HIDDEN + 2 * rows * HIDDEN + (0 if case["fused"] else 2 * rows * V),
                "flops": 2 * rows * V * HIDDEN}
    if kind == "step":
        B, T, past = case["B"], case["T"], case["past"]
    else:
        B, T, past = 1, case["T"] if kind == "verify" else case["P"], case["past"]
    attn = kind == "prompt" and case["attn"]
    n_lin = 0 if attn else 3
    params = n_lin * _layer_params(True) + _layer_params(False)
    vocab = 8192 if attn else VOCAB
    head_rows = 1 if kind == "prompt" else B * T
    live = sum(max(1, past - (past * b) // 7) for b in range(B)) if kind == "step" else past
    kv = 2 * 2 * HKV * D * (live + B * T)
    tape = n_lin * B * state * (2 if kind == "prompt" else T + 1)
    flops = 2 * B * T * params + 2 * head_rows * vocab * HIDDEN
    flops += n_lin * 8 * B * T * HV * D * D + 4 * HQ * D * (live * T + B * T * T // 2)
    act = 2 * B * T * HIDDEN * (2 if attn else 3) + (0 if kind == "step" else 2 * head_rows * vocab)
    return {"bytes": 2 * params + 2 * vocab * HIDDEN + kv + tape + act, "flops": flops}


def tolerance(case):
    """About four times the difference measured between the package's own
    formulations: the chunked and the sequential scan (rel 2.5e-4), row-major
    and tiled weights, norms fused or launched (models: rel 8e-3 for a block),
    a prompt in one pass or in 16-token blocks (rel 1.7e-2, one attention
    layer 6.4e-3), the head against a library product (rel 2.4e-5).  A single
    bf16 rounding moves one value by 8e-3 of itself."""
    kind = case["kind"]
    if kind in ("scan", "prefill"):
        return {"rel": 1e-3, "max": 3.2e-2}
    if kind == "layer":
        return {"rel": 4e-3, "max": 6.4e-2}
    if kind == "head":
        return {"rel": 1e-3, "max": 3.2e-2}
    if kind == "prompt" and case["attn"]:
        return {"rel": 2.5e-2, "max": 1.1e-1}
    return {"rel": 3e-2, "max": 8e-1}


# ------------------------------------------------------------------ fp64

def _gated_delta64(q, k, v, g, beta, S, tape):
    """The gated delta rule token by token: q, k [B,T,Hk,D], v [B,T,Hv,D]."""
    rep = v.shape[2] // k.shape[2]
    q, k = (t.double().repeat_interleave(rep, dim=2) for t in (q, k))
    v, g, beta, S = v.double(), g.double(), beta.double(), S.double()
    outs, slabs = [], []
    for t in range(v.shape[1]):
        kt = k[:, t, :, None, :]
        S = S * g[:, t, :, None, None]
        delta = (v[:, t] - (S * kt).sum(-1)) * beta[:, t, :, None]
        S = S + delta[..., None] * kt
        outs.append((S * q[:, t, :, None, :]).sum(-1))
        if tape:
            slabs.append(S)
    return torch.stack(outs, 1), S, torch.stack(slabs) if tape else None


def _rms64(x, w=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _silu64(x):
    return x * torch.sigmoid(x)


def _linear64(qkv, z, a, b, conv, S, p, tape):
    """The gated-delta layer body: (y, last conv rows, final state, tape)."""
    B, T = qkv.shape[:2]
    x = torch.cat([conv.double(), qkv.double()], 1)
    w = p["conv_w"].double()
    act = _silu64(sum(w[:, j] * x[:, j:j + T] for j in range(CONV_K)))
    kd = HK * D
    q = _rms64(act[..., :kd].reshape(B, T, HK, D)) / D
    k = _rms64(act[..., kd:2 * kd].reshape(B, T, HK, D)) * D ** -0.5
    v = act[..., 2 * kd:].reshape(B, T, HV, D)
    g = torch.exp(-torch.exp(p["A_log"].double())
                  * torch.nn.functional.softplus(a.double() + p["dt_bias"].double()))
    out, final, slabs = _gated_delta64(q, k, v, g, torch.sigmoid(b.double()), S, tape)
    y = _rms64(out, p["norm"]) * _silu64(z.double().reshape(B, T, HV, D))
    return y.reshape(B, T, HV * D), x[:, T:], final, slabs


def _rope64(x, pos):
    half = ROT // 2
    ang = pos.double()[:, None, None] * THETA ** (-2.0 * torch.arange(half, device=x.device).double() / ROT)
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., :half], x[..., half:ROT]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., ROT:]], -1)


def _attention64(x, lw, past, keys, vals):
    """One sequence's attention: x [T, H]; keys, vals [Hkv, past, D] or None."""
    T = x.shape[0]
    proj = x @ lw["w_qkv"].double().t()
    qg = proj[:, :2 * HQ * D].reshape(T, HQ, 2 * D)
    q, gate = qg[..., :D], qg[..., D:]
    k, v = proj[:, 2 * HQ * D:].reshape(T, 2, HKV, D).unbind(1)
    pos = torch.arange(past, past + T, device=x.device)
    q, k = _rope64(_rms64(q, lw["q_norm"]), pos), _rope64(_rms64(k, lw["k_norm"]), pos)
    kn, vn = k.transpose(0, 1), v.transpose(0, 1)
    ka = kn if keys is None else torch.cat([keys[:, :past].double(), kn], 1)
    va = vn if vals is None else torch.cat([vals[:, :past].double(), vn], 1)
    seen = torch.arange(past + T, device=x.device)[None, :]
    o = torch.empty(T, HQ, D, dtype=F64, device=x.device)
    for h in range(HQ):
        for t0 in range(0, T, 2048):
            s = q[t0:t0 + 2048, h] @ ka[h // (HQ // HKV)].t() * D ** -0.5
            s.masked_fill_(seen > pos[t0:t0 + 2048, None], float("-inf"))
            o[t0:t0 + 2048, h] = torch.softmax(s, -1) @ va[h // (HQ // HKV)]
            del s
    o = (o * torch.sigmoid(gate)).reshape(T, HQ * D)
    return o @ lw["w_o"].double().t(), kn, vn


def _model64(w, toks, lens, conv, rec, keys, vals, tape):
    """The model over toks [B, T] from its caches (None: empty ones)."""
    B, T = toks.shape
    h = w["embed"][toks.long()].double()
    res = {"layers": [], "state": [], "tape": [], "kv": []}
    gi = 0
    for lw in w["layers"]:
        x = _rms64(h, lw["ln_in"])
        if "w_in" in lw:
            proj = x @ lw["w_in"].double().t()
            qkv, z = proj[..., :CONV], proj[..., CONV:CONV + HV * D]
            b, a = proj[..., CONV + HV * D:].split(HV, -1)
            c0 = torch.zeros(B, CONV_K - 1, CONV, device=h.device) if conv is None else conv[gi]
            s0 = torch.zeros(B, HV, D, D, device=h.device) if rec is None else rec[gi]
            y, _, final, slabs = _linear64(qkv, z, a, b, c0, s0, lw["p"], tape)
            r = y @ lw["w_out"].double().t()
            res["state"].append(final)
            res["tape"].append(slabs)
            gi += 1
        else:
            per = [_attention64(x[i], lw, lens[i], None if keys is None else keys[i],
                                None if vals is None else vals[i]) for i in range(B)]
            r = torch.stack([o for o, _, _ in per])
            res["kv"] += [torch.stack([k for _, k, _ in per]), torch.stack([v for _, _, v in per])]
        h = h + r
        x = _rms64(h, lw["ln_post"])
        gu = x @ lw["w_gu"].double().t()
        h = h + (_silu64(gu[..., :MLP]) * gu[..., MLP:]) @ lw["w_down"].double().t()
        res["layers"].append(h)
    res["norm"] = _rms64(h, w["final"])
    return res


def exact(case, seed):
    kind = case["kind"]
    if kind in ("scan", "prefill"):
        x = _scan_inputs(seed, case["B"], case["T"], case["Hk"], case["Hv"], case.get("D", D))
        out, final, slabs = _gated_delta64(*x, tape=kind == "scan")
        return (out, final, slabs) if kind == "scan" else (out, final)
    if kind == "layer":
        x = _layer_inputs(case, seed)
        return list(_linear64(x["qkv"], x["z"], x["a"], x["b"], x["conv"], x["state"], x["p"], True))
    if kind == "head":
        weight, hidden, _ = _head_inputs(case, seed)
        if case["fused"]:
            return None
        rows = hidden.reshape(-1, HIDDEN).double()
        logits = torch.cat([rows @ w.double().t() for w in weight.split(16384)], 1)
        return [logits.reshape(case["B"], case["N"], -1), None, None, None]
    if kind == "step":
        lens, conv, rec, keys, vals, toks = _step_caches(case, seed)
        r = _model64(_model_weights(seed, False), toks, lens, conv, rec, keys, vals, True)
        return [r["norm"].reshape(-1, HIDDEN), *r["tape"]]
    attn = kind == "prompt" and case["attn"]
    n = case["T"] if kind == "verify" else case["P"]
    past = case["past"]
    w = _model_weights(seed, attn)
    toks = _tokens(seed, past + n, w["embed"].shape[0])[None]
    r = _model64(w, toks, [0], None, None, None, None, False)
    ids = [0] if attn else [1, 3]
    hidden = torch.cat([r["layers"][i][:, past:] for i in ids], -1)
    rows = r["norm"][0, past:] if kind == "verify" else r["norm"][0, -1:]
    logits = torch.cat([rows @ p.double().t() for p in w["lm_head"].split(16384)], 1)[None]
    states = [None] * len(r["state"]) if kind == "verify" else r["state"]
    return [logits, hidden, *states, *[t[:, :, past:] for t in r["kv"]]]
