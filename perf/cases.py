"""The work that a user of this framework has it do, as cases with their inputs, outputs, needed work and 64-bit results.

  look    photos and a question in, the first token's logits and the filled key / value cache out (PaliGemma-3B)
  reply   one graph-replayed step of a reply, for one conversation or several in lock step (PaliGemma-3B)
  read    prompts of unequal lengths in one packed step (layered decoders: Tuvodra, Raritar), bf16 or fp32
  write   one graph-replayed step of every sequence (layered decoders), each at its own position, bf16 or fp32
  sample  top-p draws over a vocabulary

Layer sizes are those of this repository's configurations and benchmark.  Weights are random with the scales of an
ordinary initialisation, so that the layers keep the residual's size; inputs come from the seed.
"""
import math
import os
import sys

import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "multimodal-financial-analysis-tool-using-paligemma_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

DEV = "cuda"
REPLY = 256  # tokens of a reply before the next one starts from its prompt again
IMAGE_TOKEN = 257152


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: the next token of one chat, drawn from logits that the caller already has
        {"name": "draw one token", "what": "sample", "rows": 1, "vocab": 257216, "temperature": 0.8, "top_p": 0.9},
        # one photo and a question, until the first token of the answer can be picked
        {"name": "photo", "what": "look", "images": 1, "side": 224, "text": 32},
        # the same at the larger checkpoint's resolution
        {"name": "large photo", "what": "look", "images": 1, "side": 448, "text": 32},
        # eight photos answered as one batch: the largest
        {"name": "eight photos", "what": "look", "images": 8, "side": 224, "text": 32},
        # a chat's reply, token by token
        {"name": "reply", "what": "reply", "rows": 1, "kept": 288},
        # two chats about large photos
        {"name": "two replies", "what": "reply", "rows": 2, "kept": 1056},
        # the eight photos' replies in lock step
        {"name": "eight replies", "what": "reply", "rows": 8, "kept": 288},
        # a few prompts that arrived together
        {"name": "prompts", "what": "read", "design": "Tuvodra", "size": "2b", "dtype": "bfloat16", "lens": "1024,387,129"},
        # a small model's reply, where launches and latency count
        {"name": "small model's step", "what": "write", "design": "Tuvodra", "size": "1b", "dtype": "bfloat16", "lens": "1000"},
        # prompts through a mixture of experts
        {"name": "mixture prompts", "what": "read", "design": "Raritar", "size": "2b", "dtype": "bfloat16", "lens": "511,2,1300,235"},
        # a server's step: eight conversations of unequal lengths
        {"name": "mixture step", "what": "write", "design": "Raritar", "size": "2b", "dtype": "bfloat16",
         "lens": "1020,33,700,1411,256,90,510,64"},
        # a prompt in the 32-bit mode, which a checkpoint's results are compared in
        {"name": "32-bit prompt", "what": "read", "design": "Tuvodra", "size": "1b", "dtype": "float32", "lens": "500"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["sample", "look", "look", "reply", "reply", "read", "read", "write", "write"])
    if what == "sample":
        return {"what": what, "rows": rng.randint(1, 8), "vocab": rng.choice([257216, 65536, 32768, _log(rng, 1000, 250000)]),
                "temperature": round(rng.uniform(0.6, 1.2), 3), "top_p": round(rng.uniform(0.8, 0.98), 3)}
    if what == "look":
        if rng.random() < 0.25:
            return {"what": what, "images": 1, "side": 448, "text": rng.randint(8, 128)}
        text = rng.randint(8, 64)
        return {"what": what, "images": rng.randint(1, 2304 // (256 + text)), "side": 224, "text": text}
    if what == "reply":
        return {"what": what, "rows": rng.randint(1, 8), "kept": _log(rng, 200, 1400)}
    dtype = "float32" if rng.random() < 0.25 else "bfloat16"
    case = {"what": what, "design": rng.choice(["Tuvodra", "Raritar"]), "size": "1b" if dtype == "float32" else rng.choice(["1b", "2b"]),
            "dtype": dtype}
    if what == "read":
        total, n = _log(rng, 32, 1024 if dtype == "float32" else 4096), rng.randint(1, 8)
        cuts = sorted(rng.sample(range(1, total), n - 1))
        lens = [b - a for a, b in zip([0] + cuts, cuts + [total])]
    else:
        rows = _log(rng, 1, 32)
        lens = [_log(rng, 32, min(2048, 16384 // rows)) for _ in range(rows)]
    return dict(case, lens=",".join(map(str, lens)))


def _lens(case):
    return [int(n) for n in case["lens"].split(",")]


# ---------------------------------------------------------------- PaliGemma-3B: sizes and weights
VIS, TXT = "vision_tower.vision_model.", "language_model.model."
V = {"width": 1152, "ff": 4304, "layers": 27, "heads": 16, "patch": 14}
T = {"width": 2048, "ff": 16384, "layers": 18, "heads": 8, "dim": 256, "vocab": 257216}


def _pali_config(side):
    return {"vision_config": {"hidden_size": V["width"], "intermediate_size": V["ff"], "num_hidden_layers": V["layers"],
                              "num_attention_heads": V["heads"], "num_channels": 3, "image_size": side, "patch_size": V["patch"],
                              "layer_norm_eps": 1e-6, "projection_dim": T["width"]},
            "text_config": {"vocab_size": T["vocab"], "hidden_size": T["width"], "intermediate_size": T["ff"],
                            "num_hidden_layers": T["layers"], "num_attention_heads": T["heads"], "num_key_value_heads": 1,
                            "head_dim": T["dim"], "max_position_embeddings": 8192, "rms_norm_eps": 1e-6, "rope_theta": 10000.0},
            "image_token_index": IMAGE_TOKEN, "vocab_size": T["vocab"], "projection_dim": T["width"], "hidden_size": T["width"],
            "pad_token_id": 0, "bos_token_id": 2, "eos_token_id": 1}


def _patches(side):
    return (side // V["patch"]) ** 2


def _pali_specs(side):
    """name -> (shape, standard deviation, mean)"""
    w, f, out = V["width"], V["ff"], {}

    def lin(name, n, k, gain=1.0):
        out[name + ".weight"] = ((n, k), gain / math.sqrt(k), 0.0)

    def biased(name, n, k, gain=1.0):
        lin(name, n, k, gain)
        out[name + ".bias"] = ((n,), 0.02, 0.0)

    out[VIS + "embeddings.patch_embedding.weight"] = ((w, 3, V["patch"], V["patch"]), 1.0 / math.sqrt(3 * V["patch"] ** 2), 0.0)
    out[VIS + "embeddings.patch_embedding.bias"] = ((w,), 0.02, 0.0)
    out[VIS + "embeddings.position_embedding.weight"] = ((_patches(side), w), 0.5, 0.0)
    res = 1.0 / math.sqrt(V["layers"])
    for i in range(V["layers"]):
        p = VIS + "encoder.layers.%d." % i
        for n in ("q_proj", "k_proj", "v_proj"):
            biased(p + "self_attn." + n, w, w)
        biased(p + "self_attn.out_proj", w, w, res)
        biased(p + "mlp.fc1", f, w)
        biased(p + "mlp.fc2", w, f, res)
        for n in ("layer_norm1", "layer_norm2"):
            out[p + n + ".weight"], out[p + n + ".bias"] = ((w,), 0.1, 1.0), ((w,), 0.05, 0.0)
    out[VIS + "post_layernorm.weight"], out[VIS + "post_layernorm.bias"] = ((w,), 0.1, 1.0), ((w,), 0.05, 0.0)
    biased("multi_modal_projector.linear", T["width"], w)
    w, f, res = T["width"], T["ff"], 1.0 / math.sqrt(T["layers"])
    out[TXT + "embed_tokens.weight"] = ((T["vocab"], w), 1.0 / math.sqrt(w), 0.0)
    for i in range(T["layers"]):
        p = TXT + "layers.%d." % i
        lin(p + "self_attn.q_proj", T["heads"] * T["dim"], w)
        lin(p + "self_attn.k_proj", T["dim"], w)
        lin(p + "self_attn.v_proj", T["dim"], w)
        lin(p + "self_attn.o_proj", w, T["heads"] * T["dim"], res)
        lin(p + "mlp.gate_proj", f, w)
        lin(p + "mlp.up_proj", f, w)
        lin(p + "mlp.down_proj", w, f, res)
        out[p + "input_layernorm.weight"] = out[p + "post_attention_layernorm.weight"] = ((w,), 0.1, 0.0)
    out[TXT + "norm.weight"] = ((w,), 0.1, 0.0)
    return out


def _random(specs):
    """bf16 tensors of these shapes and scales; a model's weights are the same for every input."""
    g = torch.Generator(DEV).manual_seed(2024)
    out = {}
    for name, (shape, std, mean) in specs.items():
        r = torch.randn(shape, device=DEV, generator=g)
        out[name] = r.mul_(std).add_(mean).to(torch.bfloat16)
    return out


# ---------------------------------------------------------------- layered decoders: sizes and weights
KINDS = 64  # tokens fall into kinds, by which the mixtures' routers choose


def _decoder_config(design, size):
    w = {"1b": 1024, "2b": 2048}[size]
    heads, kv, ff, vocab = {"1b": (8, 2, 4096, 32768), "2b": (16, 2, 16384, 257216)}[size]
    if design == "Raritar":
        experts, expert_ff, shared_ff = {"1b": (28, 512, 1024), "2b": (60, 1024, 4096)}[size]
        moe = {"kind": "moe", "expert": {"ff": expert_ff}, "shared": {"ff": shared_ff},
               "router": {"experts": experts, "identity": 4, "top": 6, "groups": {"count": 4, "keep": 2}}}
        layers = []
        for i in range(8):
            m = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 50.0,
                 "mask": {"size": 1024, "keep_first": 16},
                 "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}
            if i > 4:
                m["kv_from"] = 4
            layers.append({"type": "attention", "mixer": m, "mlp": moe})
        return {"architecture": design, "vocab": vocab, "width": w, "canon": {"taps": 4}, "norm": {"eps": 1e-5},
                "embedding": {"bigram": {"buckets": 65521, "mul_prev": 4099, "mul_cur": 257}}, "residual_mult": 0.5, "layers": layers}
    mamba = {"type": "mamba1", "mixer": {"inner": 2 * w, "state": 16, "dt_rank": w // 16, "conv": 4}, "mlp": None}
    gru = {"type": "mingru", "mixer": {"width": w}, "mlp": None}
    attn = {"type": "attention", "mixer": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                                           "mask": {"size": 1024}}, "mlp": {"kind": "dense", "ff": ff}}
    return {"architecture": design, "vocab": vocab, "width": w, "streams": 2, "norm": {"groups": 4, "eps": 1e-5},
            "embedding": {"scale": 32.0}, "layers": [mamba, gru, mamba, attn] * 4}


def _decoder_specs(cfg):
    """name -> (shape, standard deviation, mean)"""
    D, raritar, out = cfg["width"], cfg["architecture"] == "Raritar", {}
    res = 1.0 if raritar else 0.5

    def lin(name, n, k, gain=1.0):
        out[name] = ((n, k), gain / math.sqrt(k), 0.0)

    if raritar:
        out["embed"], out["bigram"] = ((cfg["vocab"], D), 1.0, 0.0), ((cfg["embedding"]["bigram"]["buckets"] + 1, D), 0.3, 0.0)
        out["head"] = ((cfg["vocab"], D), 1.0 / math.sqrt(D), 0.0)
    else:
        out["embed"] = ((cfg["vocab"], D), 1.0 / 32.0, 0.0)
    norm, eye = (() if raritar else (D,)), cfg.get("streams", 1)
    for i, layer in enumerate(cfg["layers"]):
        p, x, m, mlp = "l%d." % i, "l%d.mix." % i, layer["mixer"], layer["mlp"]
        for q in ("1", "2") if mlp else ("1",):
            out[p + "norm" + q] = (norm, 0.1, 1.0)
            if not raritar:
                out[p + "hc%s.in" % q], out[p + "hc%s.out" % q] = ((eye,), 0.05, 1.0 / eye), ((eye,), 0.1, 1.0)
                out[p + "hc%s.mix" % q] = ((eye, eye), 0.02, 0.0)  # and the identity, below
        if raritar:
            out[p + "canon1"] = ((D, cfg["canon"]["taps"]), 0.3, 0.0)
        if layer["type"] == "mamba1":
            C, N, R = m["inner"], m["state"], m["dt_rank"]
            lin(x + "in", 2 * C, D)
            out[x + "conv"], out[x + "conv.b"] = ((C, m["conv"]), 0.5, 0.0), ((C,), 0.1, 0.0)
            lin(x + "x", R + 2 * N, C)
            lin(x + "dt", C, R)
            out[x + "dt.b"], out[x + "A_log"], out[x + "D"] = ((C,), 1.0, -3.0), ((C, N), 0.8, 0.5), ((C,), 0.3, 1.0)
            lin(x + "o", D, C, res)
        elif layer["type"] == "mingru":
            C = m["width"]
            for n in "zxg":
                lin(x + n, C, D)
            out[x + "z.b"], out[x + "x.b"] = ((C,), 1.0, -2.0), ((C,), 0.1, 0.0)
            lin(x + "o", D, C, res)
        else:
            H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            sizes = [("q", H * d)] + ([] if m.get("kv_from") is not None else [("k", G * d), ("v", G * e)])
            for n, rows in sizes:
                lin(x + n, rows, D)
                if not raritar:
                    out[x + n + ".b"] = ((rows,), 0.1, 0.0)
            if not raritar:
                out[x + "r1"] = out[x + "r2"] = ((H,), 0.1, 0.5)
            lin(x + "o", D, H * e, res)
        if mlp and mlp["kind"] == "dense":
            lin(p + "mlp.gate", mlp["ff"], D)
            lin(p + "mlp.up", mlp["ff"], D)
            lin(p + "mlp.down", D, mlp["ff"], res)
        elif mlp:
            r = mlp["router"]
            parts = [("e%d." % e, mlp["expert"]["ff"]) for e in range(r["experts"])] + [("shared.", mlp["shared"]["ff"])]
            for n, ff in parts:
                lin(p + "mlp." + n + "gate", ff, D)
                lin(p + "mlp." + n + "up", ff, D)
                lin(p + "mlp." + n + "down", D, ff, 2.0)
            out[p + "mlp.router"], out[p + "mlp.correction"] = ((r["experts"] + r["identity"], D), 0.0, 0.0), ((r["experts"] + r["identity"],), 0.0, 0.0)
            lin(p + "mlp.shared.sg", 1, D)
    out["final.norm"] = (norm, 0.1, 1.0)
    return out


def _decoder_weights(cfg):
    """Random weights.  A trained router decides clearly; a random one over a random residual has close calls, which rounding
    turns.  So the last KINDS coordinates of Raritar's residual hold the token's kind, which no layer writes and which alone
    the routers read: for every kind a layer's router has its own chosen experts, in its own chosen groups."""
    W = _random(_decoder_specs(cfg))
    D = cfg["width"]
    g = torch.Generator().manual_seed(7)
    for name, w in W.items():
        leaf = name.split(".", 1)[-1]
        if leaf.startswith("hc") and leaf.endswith(".mix"):
            w += torch.eye(w.shape[0], dtype=w.dtype, device=DEV)
        if cfg["architecture"] != "Raritar":
            continue
        if name in ("embed", "bigram"):
            w[:, D - KINDS:] = 0.0
            if name == "embed":
                at = torch.arange(w.shape[0], device=DEV)
                w[at, D - KINDS + at % KINDS] = 8.0
        elif leaf.endswith(".down") or leaf == "mix.o":
            w[D - KINDS:] = 0.0
        elif leaf == "canon1":
            w[D - KINDS:] = 0.0
        elif leaf == "mlp.router":
            r = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            n, count, keep, top = w.shape[0], r["groups"]["count"], r["groups"]["keep"], r["top"]
            z = torch.rand((n, KINDS), generator=g) * 0.5 - 0.4  # left: up to 0.1; chosen: 0.5 to 1
            for k in range(KINDS):
                groups = torch.randperm(count, generator=g)[:keep]
                members = torch.cat([torch.arange(n // count) + int(q) * (n // count) for q in groups])
                heads = torch.stack([int(q) * (n // count) + torch.randint(n // count, (1,), generator=g)[0] for q in groups])
                rest = members[~torch.isin(members, heads)]
                chosen = torch.cat([heads, rest[torch.randperm(len(rest), generator=g)[:top - keep]]])
                z[chosen, k] = torch.rand(top, generator=g) * 0.5 + 0.5
            w[:, D - KINDS:] = z.to(w)
    return W


# ---------------------------------------------------------------- inputs
def _inputs(case, seed):
    g = torch.Generator(DEV).manual_seed(seed)

    def ids(n, vocab):
        return torch.randint(3, vocab, (n,), device=DEV, generator=g)

    if case["what"] == "sample":
        # a language model's logits: a broad body, and a head that falls off with the rank
        R, n = case["rows"], case["vocab"]
        x = torch.randn((R, n), device=DEV, generator=g) * 1.5
        k = min(1000, n // 8)
        top = torch.rand((R, n), device=DEV, generator=g).topk(k, 1).indices
        x.scatter_add_(1, top, (15.5 - 1.2 * torch.log(torch.arange(1, k + 1, device=DEV).float()))[None].expand(R, k))
        return {"logits": x, "u": torch.rand(R, device=DEV, generator=g)}
    if case["what"] == "look":
        B, n = case["images"], _patches(case["side"])
        # photos: neighbouring pixels are alike; values in [-1, 1]
        low = torch.randn((B, 3, case["side"] // 8, case["side"] // 8), device=DEV, generator=g)
        px = torch.nn.functional.interpolate(low, size=(case["side"], case["side"]), mode="bilinear")
        px = (px + 0.2 * torch.randn(px.shape, device=DEV, generator=g)).tanh()
        text = ids(B * case["text"], 256000).view(B, -1)
        return {"pixels": px, "ids": torch.cat([torch.full((B, n), IMAGE_TOKEN, device=DEV), text], 1)}
    if case["what"] == "reply":
        kv = torch.randn((T["layers"], 2, case["rows"], case["kept"], T["dim"]), device=DEV, generator=g).to(torch.bfloat16)
        return {"kv": kv, "ids": ids(case["rows"], 256000)}
    lens, vocab = _lens(case), _decoder_config(case["design"], case["size"])["vocab"]
    return {"prompts": [ids(n, vocab) for n in lens], "ids": ids(len(lens), vocab)}


def _pali_engine(side, max_batch, max_seq):
    from pgmi import Engine
    eng = Engine(_pali_config(side), device=DEV, max_batch=max_batch, max_seq=max_seq)
    eng.load_state_dict(_random(_pali_specs(side)))
    eng.prepare()
    return eng


def _decoder_engine(case):
    from pgmi import DecoderEngine, registry
    cfg = _decoder_config(case["design"], case["size"])
    eng = DecoderEngine(registry.decoder_config(cfg), device=DEV, dtype=case["dtype"])
    eng.load_state_dict(_decoder_weights(cfg))
    eng.prepare()
    return eng


def prepare(case, seed):
    x = _inputs(case, seed)
    what = case["what"]
    if what == "sample":
        return dict(x, case=case, engine=_decoder_engine({"design": "Tuvodra", "size": "1b", "dtype": "bfloat16"}))
    if what == "look":
        B, L = x["ids"].shape
        eng = _pali_engine(case["side"], B, L)
        return dict(x, case=case, engine=eng, kv=eng.new_kv(B, L).zero_(), positions=torch.arange(L).expand(B, L))
    if what == "reply":
        B, n = case["rows"], case["kept"]
        eng = _pali_engine(224, B, 64)
        kv = eng.new_kv(B, n + REPLY).zero_()
        kv[:, :, :, :n] = x["kv"]
        return {"case": case, "engine": eng, "kv": kv, "ids": x["ids"], "next": torch.empty_like(x["ids"]), "at": 0,
                "logits": torch.empty((B, T["vocab"]), device=DEV)}
    eng, lens = _decoder_engine(case), _lens(case)
    cache = eng.new_cache(len(lens), max(lens) + (REPLY if what == "write" else 0))
    slots = [cache.alloc() for _ in lens]
    tokens = torch.cat(x["prompts"])
    state = {"case": case, "engine": eng, "cache": cache, "slots": slots, "lens": lens, "tokens": tokens}
    if what == "write":
        eng.forward(cache, slots, tokens, lens)
        state.update(ids=x["ids"], next=torch.empty_like(x["ids"]), at=0,
                     logits=torch.empty((len(lens), eng.vocab), device=DEV))
    return state


def run(s):
    eng, what = s["engine"], s["case"]["what"]
    if what == "sample":
        return eng.sample_top_p(s["logits"], s["case"]["top_p"], s["case"]["temperature"], u=s["u"], return_kept_mass=True)
    if what == "look":
        feats = eng.project(eng.vision(s["pixels"]))
        return eng.lm_forward(s["kv"], 0, s["positions"], ids=s["ids"], image_feats=feats, logits_rows=2), s["kv"]
    if what == "reply":
        at = s["case"]["kept"] + s["at"]
        s["at"] = (s["at"] + 1) % REPLY
        return eng.decode(s["ids"], s["kv"], at, at + 1, logits=s["logits"], next_ids=s["next"], graph=True), s["kv"]
    cache, slots, lens = s["cache"], s["slots"], s["lens"]
    if what == "read":
        for slot in slots:  # a sequence of no tokens yet
            cache.length[slot] = 0
        return eng.forward(cache, slots, s["tokens"], lens)
    if s["at"] == REPLY:  # the next reply
        s["at"] = 0
        for slot, n in zip(slots, lens):
            cache.length[slot] = n
    s["at"] += 1
    return eng.decode(cache, slots, s["ids"], logits=s["logits"], next_ids=s["next"], graph=True)


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    what = case["what"]
    if what == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n, "flops": 8 * n}
    vis = V["layers"] * (4 * V["width"] ** 2 + 2 * V["width"] * V["ff"]) + T["width"] * V["width"] + V["width"] * 3 * V["patch"] ** 2
    txt = T["layers"] * (2 * T["width"] * T["heads"] * T["dim"] + 2 * T["width"] * T["dim"] + 3 * T["width"] * T["ff"])
    head, kv = T["width"] * T["vocab"], T["layers"] * 2 * T["dim"]
    if what == "look":
        B, n = case["images"], _patches(case["side"])
        L = n + case["text"]
        flops = 2 * B * (n * vis + L * txt + head + V["layers"] * 2 * n * n * V["width"] + T["layers"] * 2 * L * L * T["heads"] * T["dim"])
        return {"bytes": 2 * (vis + txt + head) + B * (12 * case["side"] ** 2 + 2 * L * kv + 4 * T["vocab"]), "flops": flops}
    if what == "reply":
        B, n = case["rows"], case["kept"]
        return {"bytes": 2 * (txt + head) + B * (2 * n * kv + 4 * T["vocab"]),
                "flops": 2 * B * (txt + head + T["layers"] * 2 * n * T["heads"] * T["dim"])}
    cfg, lens = _decoder_config(case["design"], case["size"]), _lens(case)
    rows, one = (sum(lens) if what == "read" else len(lens)), 4 if case["dtype"] == "float32" else 2
    bytes_ = flops = 0.0
    for name, (shape, _, _) in _decoder_specs(cfg).items():
        n = math.prod(shape)
        if name == "bigram" or (name == "embed" and cfg["architecture"] == "Raritar"):
            continue  # a few rows of a table
        times, used = rows, 1.0
        if ".mlp.e" in name:  # on average
            r = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            share = r["top"] / (r["experts"] + r["identity"])
            times, used = rows * share, 1.0 - (1.0 - share) ** min(rows, KINDS)
        bytes_ += 2 * n * used
        flops += 2 * n * (len(lens) if name in ("embed", "head") else times)
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "attention":
            per = m["kv_heads"] * (m["dim"] + m["vdim"]) * one
            for n in lens:
                seen = min(n, m["mask"]["size"] + m["mask"].get("keep_first", 0))
                pairs = seen if what == "write" else n * (n + 1) / 2 - max(0, n - seen) * (n - seen + 1) / 2
                flops += 2 * pairs * m["heads"] * (m["dim"] + m["vdim"])
                bytes_ += per * (seen if what == "write" else n if m.get("kv_from") is None else 0)
        else:
            state = m["inner"] * m["state"] if layer["type"] == "mamba1" else m["width"]
            flops += 6 * rows * state
            bytes_ += 4 * len(lens) * state * (2 if what == "write" else 1)
    return {"bytes": bytes_ + 4 * len(lens) * cfg["vocab"], "flops": flops}


def tolerance(case):
    # measured against exact(): PaliGemma 1.2e-2 (45 layers of bf16 activations) and 1.5e-2 (the cache), the layered
    # decoders 4e-3 in bf16 and 1.4e-6 in fp32; two correct implementations differ by up to the sum of their errors
    if case["what"] == "sample":
        return {"rel": 1e-5, "differ": 0.0}
    if case.get("dtype") == "float32":
        return {"rel": 6e-6}
    return {"rel": 2.5e-2 if case["what"] in ("look", "reply") else 1.6e-2}


# ---------------------------------------------------------------- the same results in 64 bits
class _Doubles:
    """Weights in 64 bits, one at a time."""

    def __init__(self, weights):
        self.w = weights

    def __getitem__(self, name):
        return self.w[name].double()


def exact(case, seed):
    x = _inputs(case, seed)
    with torch.no_grad():
        if case["what"] == "sample":
            return [None, _kept_mass(x["logits"].double() / case["temperature"], case["top_p"])]
        if case["what"] == "look":
            return _look(case, x)
        if case["what"] == "reply":
            return _reply(case, x)
        cfg = _decoder_config(case["design"], case["size"])
        W = _Doubles(_decoder_weights(cfg))
        seqs = x["prompts"]
        if case["what"] == "write":
            seqs = [torch.cat([p, t[None]]) for p, t in zip(seqs, x["ids"])]
        return (_raritar if case["design"] == "Raritar" else _tuvodra)(cfg, W, seqs)


def _kept_mass(z, top_p):
    p = torch.softmax(z, -1).sort(-1, descending=True).values
    before = p.cumsum(-1) - p
    return (p * (before <= top_p)).sum(-1)


def _linear(x, W, name, bias=True):
    y = x @ W[name + ".weight"].t()
    return y + W[name + ".bias"] if bias else y


def _layer_norm(x, W, name):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], W[name + ".weight"], W[name + ".bias"], 1e-6)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale):
    """q (B, H, n, d), k and v (B, H or 1, m, d)"""
    return torch.softmax(q @ k.transpose(-1, -2).contiguous() * scale, -1) @ v


def _look(case, x):
    W = _Doubles(_random(_pali_specs(case["side"])))
    B, n, w, p = case["images"], _patches(case["side"]), V["width"], V["patch"]
    g = case["side"] // p
    px = x["pixels"].to(torch.bfloat16).double()
    rows = px.view(B, 3, g, p, g, p).permute(0, 2, 4, 1, 3, 5).reshape(B, n, 3 * p * p)
    h = rows @ W[VIS + "embeddings.patch_embedding.weight"].view(w, -1).t() + W[VIS + "embeddings.patch_embedding.bias"]
    h = h + W[VIS + "embeddings.position_embedding.weight"]

    def heads(y):
        return y.view(B, n, V["heads"], -1).transpose(1, 2).contiguous()

    for i in range(V["layers"]):
        q = VIS + "encoder.layers.%d." % i
        y = _layer_norm(h, W, q + "layer_norm1")
        o = _attend(*(heads(_linear(y, W, q + "self_attn." + m)) for m in ("q_proj", "k_proj", "v_proj")), (w // V["heads"]) ** -0.5)
        h = h + _linear(o.transpose(1, 2).reshape(B, n, w), W, q + "self_attn.out_proj")
        y = torch.nn.functional.gelu(_linear(_layer_norm(h, W, q + "layer_norm2"), W, q + "mlp.fc1"), approximate="tanh")
        h = h + _linear(y, W, q + "mlp.fc2")
    feats = _linear(_layer_norm(h, W, VIS + "post_layernorm"), W, "multi_modal_projector.linear")
    e = W.w[TXT + "embed_tokens.weight"][x["ids"]].double()
    e[:, :n] = feats / math.sqrt(T["width"])
    L = e.shape[1]
    kv = torch.zeros((T["layers"], 2, B, L, T["dim"]), dtype=torch.float64, device=DEV)
    h = _gemma(W, e, torch.arange(L, device=DEV), kv, 0)
    return _pali_head(W, h[:, -1:]), kv


def _reply(case, x):
    W = _Doubles(_random(_pali_specs(224)))
    n = case["kept"]
    kv = torch.zeros((T["layers"], 2, case["rows"], n + REPLY, T["dim"]), dtype=torch.float64, device=DEV)
    kv[:, :, :, :n] = x["kv"].double()
    e = W.w[TXT + "embed_tokens.weight"][x["ids"]].double()[:, None]
    h = _gemma(W, e, torch.tensor([n + 1], device=DEV), kv, n)
    return _pali_head(W, h)[:, 0], kv


def _gemma(W, e, positions, kv, start):
    """The text layers over rows at `positions`, whose keys and values go to rows start .. of kv."""
    B, L, w = e.shape
    d, H = T["dim"], T["heads"]
    angle = positions.double()[:, None] * 10000.0 ** (-torch.arange(0, d, 2, device=DEV).double() / d)
    cos, sin = torch.cat([angle, angle], 1).cos(), torch.cat([angle, angle], 1).sin()

    def turned(y):
        return y * cos + torch.cat([-y[..., d // 2:], y[..., :d // 2]], -1) * sin

    h = e * 45.25  # the square root of the width, as the model holds it
    for i in range(T["layers"]):
        p = TXT + "layers.%d." % i
        y = _rms(h, 1e-6) * (1.0 + W[p + "input_layernorm.weight"])
        q = turned(_linear(y, W, p + "self_attn.q_proj", False).view(B, L, H, d).transpose(1, 2))
        kv[i, 0, :, start:start + L] = turned(_linear(y, W, p + "self_attn.k_proj", False))
        kv[i, 1, :, start:start + L] = _linear(y, W, p + "self_attn.v_proj", False)
        k, v = kv[i, 0, :, None, :start + L], kv[i, 1, :, None, :start + L]
        o = _attend(q, k, v, d ** -0.5).transpose(1, 2).reshape(B, L, H * d)
        h = h + _linear(o, W, p + "self_attn.o_proj", False)
        y = _rms(h, 1e-6) * (1.0 + W[p + "post_attention_layernorm.weight"])
        y = torch.nn.functional.gelu(_linear(y, W, p + "mlp.gate_proj", False), approximate="tanh") * _linear(y, W, p + "mlp.up_proj", False)
        h = h + _linear(y, W, p + "mlp.down_proj", False)
    return h


def _pali_head(W, h):
    return (_rms(h, 1e-6) * (1.0 + W[TXT + "norm.weight"])) @ W[TXT + "embed_tokens.weight"].t()


def _gated(h, W, p):
    return (torch.nn.functional.silu(h @ W[p + "gate"].t()) * (h @ W[p + "up"].t())) @ W[p + "down"].t()


def _seen(n, mask):
    at = torch.arange(n, device=DEV)
    gap = at[:, None] - at[None]
    return gap, (gap >= 0) & ((gap < mask["size"]) | (at[None] < mask.get("keep_first", 0)))


def _heads(y, n):
    return y.view(y.shape[0], n, -1).transpose(0, 1).contiguous()


def _repeated(y, H):
    return y.repeat_interleave(H // y.shape[0], 0)


def _shifted_sum(x, w):
    """A causal convolution per channel: x (n, C), w (C, taps), its last column the current row's."""
    n, taps = x.shape[0], w.shape[1]
    past = torch.cat([x.new_zeros((taps - 1, x.shape[1])), x])
    return sum(past[k:k + n] * w[:, k] for k in range(taps))


def _tuvodra(cfg, W, seqs):
    eps, groups, last = cfg["norm"]["eps"], cfg["norm"]["groups"], []

    def norm(x, name):
        return _rms(x.view(x.shape[0], groups, -1), eps).reshape(x.shape) * W[name]

    for ids in seqs:
        n = len(ids)
        X = (W.w["embed"][ids].double() * cfg["embedding"]["scale"])[None].repeat(cfg["streams"], 1, 1)
        for i, layer in enumerate(cfg["layers"]):
            p, x, m = "l%d." % i, "l%d.mix." % i, layer["mixer"]

            def sub(q, fn, X):
                h = norm((W[p + "hc%d.in" % q][:, None, None] * X).sum(0), p + "norm%d" % q)
                return torch.einsum("st,snd->tnd", W[p + "hc%d.mix" % q], X) + W[p + "hc%d.out" % q][:, None, None] * fn(h)

            def mamba(h):
                C, N, R = m["inner"], m["state"], m["dt_rank"]
                u, z = (h @ W[x + "in"].t()).split(C, 1)
                u = torch.nn.functional.silu(_shifted_sum(u, W[x + "conv"]) + W[x + "conv.b"])
                q = u @ W[x + "x"].t()
                dt = torch.nn.functional.softplus(q[:, :R] @ W[x + "dt"].t() + W[x + "dt.b"])
                A, S, y = -W[x + "A_log"].exp(), u.new_zeros((C, N)), torch.empty_like(u)
                for a in range(0, n, 512):
                    b = min(n, a + 512)
                    keep = (dt[a:b, :, None] * A).exp()
                    all_S = (dt[a:b] * u[a:b])[:, :, None] * q[a:b, None, R:R + N]
                    for t in range(b - a):
                        S = all_S[t].addcmul_(keep[t], S)
                    y[a:b] = (all_S * q[a:b, None, R + N:]).sum(-1)
                return ((y + W[x + "D"] * u) * torch.nn.functional.silu(z)) @ W[x + "o"].t()

            def gru(h):
                z = torch.sigmoid(h @ W[x + "z"].t() + W[x + "z.b"])
                u = h @ W[x + "x"].t() + W[x + "x.b"]
                S, all_S = u.new_zeros(u.shape[1]), z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
                for t in range(n):
                    S = all_S[t].addcmul_(1.0 - z[t], S)
                return (all_S * torch.nn.functional.silu(h @ W[x + "g"].t())) @ W[x + "o"].t()

            def attention(h):
                H, G = m["heads"], m["kv_heads"]
                q, k, v = (_heads(h @ W[x + c].t() + W[x + c + ".b"], c_n) for c, c_n in (("q", H), ("k", G), ("v", G)))
                q, k = _rms(q, eps), _repeated(_rms(k, eps), H)
                gap, seen = _seen(n, m["mask"])
                s = q @ k.transpose(1, 2).contiguous() * m["scale"]
                s = s - W[x + "r1"][:, None, None] * torch.log1p(W[x + "r2"][:, None, None] * gap.clamp(min=0))
                o = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ _repeated(v, H)
                return o.transpose(0, 1).reshape(n, -1) @ W[x + "o"].t()

            X = sub(1, {"mamba1": mamba, "mingru": gru, "attention": attention}[layer["type"]], X)
            if layer["mlp"]:
                X = sub(2, lambda h: _gated(h, W, p + "mlp."), X)
        last.append(X.sum(0)[-1])
    return norm(torch.stack(last), "final.norm") @ W["embed"].t()


def _frequencies(rot):
    f = rot["base"] ** (-torch.arange(0, rot["dims"], 2, device=DEV).double() / rot["dims"])
    sc, wave = rot["scaling"], 2.0 * math.pi / f
    s = ((sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
    return (1.0 - s) * f / sc["factor"] + s * f


def _raritar(cfg, W, seqs):
    eps, mult, mul = cfg["norm"]["eps"], cfg["residual_mult"], cfg["embedding"]["bigram"]
    n_all, sizes = sum(len(s) for s in seqs), [len(s) for s in seqs]
    rows = []
    for ids in seqs:
        pair = (ids[:-1] * mul["mul_prev"] + ids[1:] * mul["mul_cur"]) % mul["buckets"]
        pair = torch.cat([torch.tensor([mul["buckets"]], device=DEV), pair])
        rows.append(W.w["embed"][ids].double() + W.w["bigram"][pair].double())
    x = torch.cat(rows)
    kept = {}
    for i, layer in enumerate(cfg["layers"]):
        p, q_, m, mlp = "l%d." % i, "l%d.mix." % i, layer["mixer"], layer["mlp"]
        H, G, rot = m["heads"], m["kv_heads"], m["rot"]
        h = _rms(x, eps) * W[p + "norm1"]
        h = torch.cat([y + _shifted_sum(y, W[p + "canon1"]) for y in h.split(sizes)])
        q, out, f = h @ W[q_ + "q"].t(), [], _frequencies(rot)
        k, v = (None, None) if m.get("kv_from") is not None else (h @ W[q_ + "k"].t(), h @ W[q_ + "v"].t())

        def turned(y):
            a = torch.arange(y.shape[1], device=DEV).double()[:, None] * f
            u, w, d = y[..., 0:rot["dims"]:2], y[..., 1:rot["dims"]:2], rot["dims"]
            t = torch.stack([u * a.cos() - w * a.sin(), w * a.cos() + u * a.sin()], -1).flatten(-2)
            return torch.cat([t, y[..., d:]], -1)

        own = [] if k is not None else kept[m["kv_from"]]
        for b, qb in enumerate(q.split(sizes)):
            if k is not None:
                own.append((turned(_heads(k.split(sizes)[b], G)), _rms(_heads(v.split(sizes)[b], G), eps)))
            s = turned(_heads(qb, H)) @ _repeated(own[b][0], H).transpose(1, 2).contiguous() * m["scale"]
            s = m["softcap"] * torch.tanh(s / m["softcap"])
            s = s.masked_fill(~_seen(len(qb), m["mask"])[1], -math.inf)
            out.append((torch.softmax(s, -1) @ _repeated(own[b][1], H)).transpose(0, 1).reshape(len(qb), -1))
        kept[i] = own
        x = x + mult * (torch.cat(out) @ W[q_ + "o"].t())
        h, r = _rms(x, eps) * W[p + "norm2"], mlp["router"]
        s = torch.softmax(h @ W[p + "mlp.router"].t(), -1)
        choice = (s + W[p + "mlp.correction"]).view(n_all, r["groups"]["count"], -1)
        groups = choice.amax(-1).topk(r["groups"]["keep"], 1).indices
        allowed = torch.full_like(choice, -math.inf)
        allowed.scatter_(1, groups[..., None].expand(-1, -1, choice.shape[2]), choice.gather(1, groups[..., None].expand(-1, -1, choice.shape[2])))
        chosen = allowed.view(n_all, -1).topk(r["top"], 1).indices
        weight = torch.zeros_like(s).scatter_(1, chosen, s.gather(1, chosen))
        y = weight[:, r["experts"]:].sum(1, keepdim=True) * h  # those that return their input
        y += torch.sigmoid(h @ W[p + "mlp.shared.sg"].t()) * _gated(h, W, p + "mlp.shared.")
        for e in range(r["experts"]):
            at = weight[:, e].nonzero()[:, 0]
            if len(at):
                y[at] += weight[at, e, None] * _gated(h[at], W, p + "mlp.e%d." % e)
        x = x + mult * y
    last = x[torch.tensor(sizes, device=DEV).cumsum(0) - 1]
    return (_rms(last, eps) * W["final.norm"]) @ W["head"].t()
