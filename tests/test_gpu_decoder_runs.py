"""The recurrences' run lengths (rows one workgroup walks) follow the step's size: sequences read together, in steps large enough
for each run length, against the same sequences alone, whose runs are the shortest or which are walked whole."""
import numpy as np
import pytest
import torch

import decoder_cases as C
from decoder_helpers import build, tokens

pytestmark = pytest.mark.gpu


# The scans of MIXED have 9 to 16 states, and these steps walk their sequences whole, as they do minGRU's; those of other numbers of states
# go in runs.
MODELS = {**C.MIXED, "runs": C.model([C.mamba(72, 8, 6, 3), C.gru(44), C.attn(6, 3, 24, 36, 40, ff=100), C.mamba(40, 20, 3, 5, ff=28)],
                                     width=84, streams=2, groups=3, vocab=211)}


# (sequences, tokens each): runs of the scan of 64, 50, 36, 32, 30, 22, 18 and 16 rows at these models' widths, and past 16,384 rows of
# 256
@pytest.mark.parametrize("n,length", [(36, 450), (30, 400), (20, 450), (3, 97), (40, 430), (36, 448), (16, 450), (12, 450), (10, 450)])
@pytest.mark.parametrize("name", sorted(MODELS))
def test_together_as_alone(name, n, length):
    cfg = MODELS[name]
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


@pytest.mark.parametrize("states", [8, 16])
def test_a_shorter_step_of_more_runs_allocates_nothing(states):
    """9,081 rows of 4,096 channels of 8 states go in 142 runs, 8,942 in 160: the workspace of the first holds the second.  (Of 16 states
    both are walked whole and carry nothing.)"""
    eng, _ = build(C.model([C.mamba(4096, states, 8, 4)], width=64, vocab=64, streams=1, groups=1), "bfloat16")
    cache = eng.new_cache(1, 9200)
    slot, toks = cache.alloc(), torch.arange(9081, device="cuda") % 64
    free = []
    for n in (9081, 8942):
        cache.length[slot] = 0
        eng.forward(cache, [slot], toks[:n], [n])
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
    assert free[0] == free[1]


@pytest.mark.parametrize("name", ["a", "runs"])
def test_captured_steps_outlive_more_runs(name):
    """A decode graph, then a packed step of as many rows in more runs (of "a", walked whole), then the graph again: as eager steps."""
    cfg = MODELS[name]
    eng, _ = build(cfg, "bfloat16", max_batch=64)
    out = []
    for graph in (True, False):
        cache = eng.new_cache(41, 64)
        one, logits = cache.alloc(), torch.empty((1, eng.vocab), device="cuda")
        ids = torch.empty(1, dtype=torch.int64, device="cuda")
        eng.forward(cache, [one], tokens(cfg, 40, 1), [40])
        for k in range(6):  # the first eager, the second captured
            ids.fill_(3 + k)
            out.append(eng.decode(cache, [one], ids, logits=logits, graph=graph).clone())
            if k == 2:
                eng.forward(cache, [cache.alloc() for _ in range(40)], tokens(cfg, 40, 2), [1] * 40)
    for a, b in zip(out[:6], out[6:]):
        assert torch.isfinite(a).all() and torch.equal(a, b)
