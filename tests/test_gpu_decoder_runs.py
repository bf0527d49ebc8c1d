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


def test_time_goes_by_the_states():
    """1,540 rows of 2,048 channels: 256 states are twice the work of 128, in the same kernel."""
    times = []
    for states in (128, 256):
        eng, _ = build(C.model([C.mamba(2048, states, 8, 4)] * 4, width=64, vocab=64, streams=1, groups=1), "bfloat16")
        cache = eng.new_cache(1, 2048)
        slot, toks = cache.alloc(), torch.arange(1540, device="cuda") % 64
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(9)]
        for e in ev:
            cache.length[slot] = 0
            eng.forward(cache, [slot], toks, [1540])
            e.record()
        torch.cuda.synchronize()
        times.append(min(a.elapsed_time(b) for a, b in zip(ev, ev[1:])))
    assert times[1] <= 2.5 * times[0]
