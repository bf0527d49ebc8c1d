"""The recurrences' run lengths (rows one workgroup walks) follow the step's size: sequences read together, in steps large enough
for each run length, against the same sequences alone, whose runs are the shortest."""
import numpy as np
import pytest
import torch

import decoder_cases as C
from decoder_helpers import build, tokens

pytestmark = pytest.mark.gpu


# (sequences, tokens each): run lengths from 64 rows down to 16 at these models' widths, and past 16,384 rows of 256
@pytest.mark.parametrize("n,length", [(36, 450), (30, 400), (20, 450), (3, 97), (40, 430)])
@pytest.mark.parametrize("name", sorted(C.MIXED))
def test_together_as_alone(name, n, length):
    cfg = C.MIXED[name]
    eng, _ = build(cfg, "float32", max_batch=64)
    lens = [length - 7 * (r % 5) for r in range(n)]
    seqs = [tokens(cfg, k + 1, 200 + r) for r, k in enumerate(lens)]
    cache = eng.new_cache(n + 1, length + 8)
    slots = [cache.alloc() for _ in seqs]
    together = eng.forward(cache, slots, [t for s, k in zip(seqs, lens) for t in s[:k]], lens)
    after = eng.step(cache, slots, [[s[k]] for s, k in zip(seqs, lens)])  # from the states that were left
    one = cache.alloc()
    for r in range(0, n, max(1, n // 4)):
        cache.length[one] = 0
        alone = eng.forward(cache, [one], seqs[r][:lens[r]], [lens[r]])
        nxt = eng.step(cache, [one], [[seqs[r][lens[r]]]])
        for got, want in ((together[r], alone[0]), (after[r], nxt[0])):
            rms = want.double().square().mean().sqrt()
            assert torch.isfinite(got).all() and (got - want).double().abs().max() <= 2e-4 * rms
