"""Shared test helpers (no reference code: restatements of its preprocessing arithmetic)."""
import json
import os

import numpy as np

# SURVEY.md sec.8c model-level rule: per-step logits rel-L2 <= 2e-2 against the reference bf16.
REL_L2_RULE = 2e-2


# Products for which the cost rule (csrc/plan.h) picks each of its forms in turn, whole and in K slices, with K tails and rows and
# columns past the last tile: test_cpu_plan.py holds the list to that, test_gpu_ops.py runs it.
PLANNED = [
    (17, 2560, 2048, "store"), (33, 200, 72, "bias"), (257, 1152, 1152, "bias_res"), (289, 1001, 2048, "store"),
    (304, 2048, 4096, "res"), (512, 4304, 1152, "bias_gelu"), (577, 1152, 4304, "bias_res"), (640, 1024, 2048, "geglu"),
    (783, 2048, 1160, "res"), (1281, 3456, 1152, "bias"), (1540, 520, 2048, "geglu"), (2049, 1152, 1152, "bias_res"),
    # the forms that those leave out
    (33, 3456, 8192, "geglu"), (193, 8200, 72, "geglu"), (601, 2560, 72, "geglu"), (1563, 2560, 2048, "bias_gelu"),
    (416, 8200, 128, "geglu"), (416, 8200, 512, "geglu"), (601, 8200, 128, "geglu"), (675, 8200, 128, "geglu"),
    # K slices
    (17, 200, 4096, "store"), (289, 200, 4304, "bias_res"), (65, 2560, 4304, "res"), (97, 8200, 4096, "bias_gelu"),
    (161, 8200, 4096, "bias"),
]


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def logit_stats(label, ours, ref_bf16, ref_fp32=None):
    """Per-step rel-L2 of our logits (steps x sampled vocabulary) against the reference bf16
    (the SURVEY sec.8c quantity), and -- when the fp32 truth is given -- the reference bf16's own
    rel-L2 against it (the floor: two bf16 implementations that each sit that far from the truth
    cannot be expected much closer to each other) and ours against it.

    The record is printed and, when PGMI_PARITY_LOG names a file, appended to it as one JSON line
    (tools/probes/parity_table.py collects them into DESIGN.md sec.5's table)."""
    ours, ref_bf16 = np.atleast_2d(ours), np.atleast_2d(ref_bf16)
    per = np.array([rel_l2(ours[t], ref_bf16[t]) for t in range(len(ours))])
    st = {"label": label, "steps": int(len(per)), "rel_vs_ref_bf16_mean": float(per.mean()),
          "rel_vs_ref_bf16_max": float(per.max()), "worst_step": int(per.argmax()),
          "steps_over_2e-2": int((per > REL_L2_RULE).sum())}
    if ref_fp32 is not None:
        ref_fp32 = np.atleast_2d(ref_fp32)
        floor = np.array([rel_l2(ref_bf16[t], ref_fp32[t]) for t in range(len(ours))])
        ofp = np.array([rel_l2(ours[t], ref_fp32[t]) for t in range(len(ours))])
        st.update({"ref_bf16_vs_fp32_mean": float(floor.mean()), "ref_bf16_vs_fp32_max": float(floor.max()),
                   "ours_vs_fp32_mean": float(ofp.mean()), "ours_vs_fp32_max": float(ofp.max()),
                   "per_step_ratio_max": float((per / np.maximum(floor, 1e-30)).max())})
        over = per > REL_L2_RULE  # the steps the floor rule governs (the rest pass on the 2e-2 bound)
        st["floor_ratio_max_over_2e-2"] = float((per[over] / np.maximum(floor[over], 1e-30)).max()) if over.any() else 0.0
        st["_per"], st["_floor"] = per, floor
    print("parity " + json.dumps({k: v for k, v in st.items() if not k.startswith("_")}))
    path = os.environ.get("PGMI_PARITY_LOG")
    if path:
        with open(path, "a") as f:
            f.write(json.dumps({k: v for k, v in st.items() if not k.startswith("_")}) + "\n")
    return st


STEP_FLOOR_FACTOR = 1.45  # per step: rel-L2 vs reference bf16 <= max(2e-2, 1.45 x the reference's own error)
MEAN_FLOOR_FACTOR = 1.25  # over the steps: mean <= max(2e-2, 1.25 x the reference's mean error)
# module-level chains (assert_within_floor: one layer or block against the oracle, base 1e-2) keep the
# earlier factor: their floors are a single module's rounding noise, not a whole model's
MODULE_FLOOR_FACTOR = 1.6


def assert_step_rule(st, step_factor=STEP_FLOOR_FACTOR, mean_factor=MEAN_FLOOR_FACTOR):
    """The SURVEY sec.8c rule as asserted here: every step's rel-L2 against the reference bf16 is
    <= 2e-2, or -- where the reference bf16 is itself further than that from its fp32 truth at
    that step -- <= step_factor x that step's reference error, and the mean over the steps
    <= max(2e-2, mean_factor x the reference's mean error).  DESIGN.md sec.5 has the measured
    table: the reference's own bf16 error vs fp32 is 1.7e-2 .. 2.9e-2 on average on the full-size
    fixtures (3.4e-2 on smoke's), our error vs fp32 is at or below it, and two independent bf16
    implementations that each sit that far from the truth land 2.2e-2 .. 2.7e-2 apart."""
    per = st["_per"]
    if "_floor" in st:
        floor = st["_floor"]
        bound = np.maximum(REL_L2_RULE, step_factor * floor)
        mean_bound = max(REL_L2_RULE, mean_factor * float(floor.mean()))
    else:
        bound, mean_bound = np.full_like(per, REL_L2_RULE), REL_L2_RULE
    bad = np.nonzero(per > bound)[0]
    assert len(bad) == 0, (st["label"], [(int(t), float(per[t]), float(bound[t])) for t in bad[:8]])
    assert float(per.mean()) <= mean_bound, (st["label"], float(per.mean()), mean_bound)


def check_model_parity(label, ours, ref_bf16, ref_fp32=None):
    """logit_stats + assert_step_rule; with the fp32 truth also the rule that our error against it
    is <= 1.5x the reference bf16's own (averaged over the steps)."""
    st = logit_stats(label, ours, ref_bf16, ref_fp32)
    assert_step_rule(st)
    if ref_fp32 is not None:
        assert st["ours_vs_fp32_mean"] <= 1.5 * st["ref_bf16_vs_fp32_mean"], (label, st["ours_vs_fp32_mean"],
                                                                            st["ref_bf16_vs_fp32_mean"])
    return st


def pixels_from_u8(u8):
    """processing_paligemma.py:20-29,47-49 on the resized uint8 image: x/255 (float64 -> float32),
    (x - 0.5)/0.5 in float32, HWC -> CHW."""
    px = (u8 * (1 / 255.0)).astype(np.float32)
    return ((px - np.float32(0.5)) / np.float32(0.5)).transpose(2, 0, 1)


# ---- the ablation harness's two monkey-patches (ablation_study_fixed.py:99-142, 144-166), restated.
# load_model_simple (:335-342) installs them on the model instance / every layer's rotary module;
# tests install these on the drop-in model to drive it the way the paper's benchmark does.

def ablation_merge(self, image_features, inputs_embeds, input_ids, attention_mask, kv_cache=None):
    """Merge semantics of ablation_study_fixed.py:99-142: the reference merge with no q_len == 1
    assertion, kv_len = cached + q_len for a filled cache, the single position
    cumsum(mask)[:, -1:] for EVERY query row of a filled cache, and positions 0..L-1 (clamped to
    max_position_embeddings - 1) otherwise."""
    import torch
    B, L = input_ids.shape
    D = image_features.shape[-1]
    dt, dev = inputs_embeds.dtype, inputs_embeds.device
    img_id, pad_id = self.config.image_token_index, self.pad_token_id
    out = torch.zeros(B, L, D, dtype=dt, device=dev)
    is_img = input_ids == img_id
    is_pad = input_ids == pad_id
    is_txt = ~is_img & ~is_pad
    out = torch.where(is_txt[..., None].expand(-1, -1, D), inputs_embeds, out)
    out = out.masked_scatter(is_img[..., None].expand(-1, -1, D), image_features / (self.config.hidden_size ** 0.5))
    out = torch.where(is_pad[..., None].expand(-1, -1, D), torch.zeros_like(out), out)
    filled = kv_cache is not None and kv_cache.num_items() > 0
    kv_len = kv_cache.num_items() + L if filled else L
    mask = torch.zeros((B, L, kv_len), dtype=dt, device=dev).unsqueeze(1)
    if filled:
        pos = attention_mask.cumsum(-1)[:, -1:]
        if pos.dim() == 1:
            pos = pos.unsqueeze(0)
    else:
        n = attention_mask.shape[1]
        pos = torch.arange(n, device=dev, dtype=torch.long).unsqueeze(0).expand(B, -1)
        pos = pos.masked_fill(attention_mask == 0, 0)
        pos = torch.clamp(pos, 0, self.config.text_config.max_position_embeddings - 1)
    return out, mask, pos


def ablation_rotary(self, x, position_ids, seq_len=None):
    """Rotary semantics of ablation_study_fixed.py:144-166: positions clamped to
    max_position_embeddings - 1, fp32 angles, cos/sin cast to x's dtype."""
    import torch
    if position_ids.dim() == 1:
        position_ids = position_ids.unsqueeze(0)
    position_ids = torch.clamp(position_ids, 0, self.max_position_embeddings - 1)
    inv = self.inv_freq.to(x.device)[None, :, None].float().expand(position_ids.shape[0], -1, 1)
    ang = (inv @ position_ids[:, None, :].float()).transpose(1, 2)
    ang = torch.cat((ang, ang), dim=-1)
    return ang.cos().to(x.dtype), ang.sin().to(x.dtype)


def install_ablation_patches(model):
    import types
    model._merge_input_ids_with_image_features = types.MethodType(ablation_merge, model)
    for layer in model.language_model.model.layers:
        layer.self_attn.rotary_emb.forward = types.MethodType(ablation_rotary, layer.self_attn.rotary_emb)


def remove_ablation_patches(model):
    model.__dict__.pop("_merge_input_ids_with_image_features", None)
    for layer in model.language_model.model.layers:
        layer.self_attn.rotary_emb.__dict__.pop("forward", None)


def assert_within_floor(label, got, ref_bf16, ref_fp32, base=1e-2, factor=MODULE_FLOOR_FACTOR):
    """Module-level form of the floor rule: rel-L2 of our output vs the oracle bf16
    <= max(base, factor x the oracle bf16's own rel-L2 vs its fp32 truth) -- for module chains whose
    bf16 rounding noise alone approaches the kernel-level 1e-2 bound (a Gemma attention: 0.96e-2, a
    whole decoder layer + final norm: 1.22e-2 on the module tests' inputs)."""
    r = rel_l2(got, ref_bf16)
    floor = rel_l2(ref_bf16, ref_fp32)
    bound = max(base, factor * floor)
    print("module-parity " + json.dumps({"label": label, "rel_vs_oracle_bf16": r, "oracle_bf16_vs_fp32": floor,
                                           "bound": bound}))
    assert r <= bound, (label, r, bound, floor)
