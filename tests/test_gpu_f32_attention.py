"""fp32 prompts' attention on the matrix units: tiles of 16 (position, head) pairs and 16 keys at their edges, windows and kept
keys across them, head sizes up to each padded width, and values that are not finite behind the mask."""
import numpy as np
import pytest
import torch

import decoder_cases as C
import raritar_cases as R
from decoder_helpers import build, close, oracle, tokens

pytestmark = pytest.mark.gpu

CASES = {
    "bias_64": C.model([C.attn(6, 2, 52, 64, 47)], width=60, streams=2, groups=3),
    "bias_128": C.model([C.attn(3, 1, 128, 72, 500)], width=60, streams=1, groups=1),
    "bias_256": C.model([C.attn(5, 1, 136, 256, 33)], width=60, streams=2, groups=3),
    "cap_keep_64": R.model([R.layer(4, 4, 64, 20, 31, keep=17, rot=8)]),
    "cap_keep_128": R.model([R.layer(8, 2, 128, 128, 64, keep=3, rot=64, cap=50.0)]),
    "plain_256": R.model([R.layer(20, 1, 256, 130, 1000, keep=16, rot=20, cap=None, scale=0.06)]),
    "past_256": R.model([R.layer(2, 1, 260, 260, 40, rot=4)]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_prompts_and_a_second_part(name):
    cfg = CASES[name]
    eng, W = build(cfg, "float32")
    lens = [1, 15, 16, 17, 65, 150]
    seqs = [tokens(cfg, n + 37, 5 + n) for n in lens]
    want = [oracle(cfg).run(cfg, W, s) for s in seqs]
    cache = eng.new_cache(len(seqs), 256)
    slots = [cache.alloc() for _ in seqs]
    for a, part in ((0, lens), (None, [37] * len(lens))):
        at = [0 if a == 0 else n for n in lens]
        lg = eng.step(cache, slots, [s[b:b + n] for s, b, n in zip(seqs, at, part)], want=list(range(sum(part))))
        close(lg, np.concatenate([w[b:b + n] for w, b, n in zip(want, at, part)]), "float32")


@pytest.mark.parametrize("name", ["bias_64", "cap_keep_128", "plain_256"])
def test_what_is_not_finite_stays_behind_the_mask(name):
    """A token whose embedding is infinite: the positions before it are as without it."""
    cfg = CASES[name]
    W = oracle(cfg).random_weights(cfg, 3)
    for k in W:
        if "embed" in k and W[k].ndim == 2 and W[k].shape[0] == cfg["vocab"]:
            W[k] = W[k].copy()
            W[k][7] = np.inf
    eng, P = build(cfg, "float32", weights=W)
    toks = [t if t != 7 else 8 for t in tokens(cfg, 60, 2)]
    cols = [c for c in range(cfg["vocab"]) if c != 7]  # the embedding is the output matrix too
    with np.errstate(invalid="ignore"):
        clean = oracle(cfg).run(cfg, P, toks)[:, cols]
    for at in (21, 44):
        cache = eng.new_cache(1, 64)
        lg = eng.step(cache, [cache.alloc()], [toks[:at] + [7] + toks[at + 1:]], want=list(range(60)))[:, cols]
        close(lg[:at], clean[:at], "float32")
        assert not torch.isfinite(lg[at]).all()
