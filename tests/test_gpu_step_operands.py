"""Steps whose operands are asked for ahead of the sums, past what is held: more taps than 4, states and rank past a lane's first two,
1, 2, 3 and 8 streams, rows on both sides of the forms' borders, several slots out of order."""
import numpy as np
import pytest
import torch

import decoder_cases as C
from decoder_helpers import build, close, oracle, tokens

pytestmark = pytest.mark.gpu

CASES = {
    "rank_200_state_33_taps_6": C.model([C.mamba(512, 33, 200, 6)], width=512, streams=2, groups=1),
    "rank_128_state_16_taps_4": C.model([C.mamba(512, 16, 128, 4), C.mamba(1024, 17, 129, 5)], width=512, streams=1, groups=2),
    "three_streams": C.model([C.gru(24, ff=40), C.mamba(64, 5, 3, 3)], width=1024, streams=3, groups=4),
    "eight_streams": C.model([C.gru(24, ff=40), C.mamba(64, 5, 3, 1), C.attn(4, 2, 32, 32, 20)], width=72, streams=8, groups=3),
}


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("B", [1, 2, 9, 17])
@pytest.mark.parametrize("name", list(CASES))
def test_steps(name, B, dtype):
    cfg = CASES[name]
    eng, W = build(cfg, dtype)
    seqs = [tokens(cfg, 8, 90 + r) for r in range(B)]
    some = sorted({0, B // 2, B - 1})
    want = [oracle(cfg).run(cfg, W, seqs[r]) for r in some]
    cache = eng.new_cache(B + 2, 12)
    cache.slab.fill_(0x7F)  # a fresh slot's state is not read
    slots = [cache.alloc() for _ in range(B + 2)][::-1][:B]
    for t in range(8):
        lg = eng.decode(cache, slots, torch.tensor([s[t] for s in seqs], device="cuda")).clone()
        close(lg[some], np.stack([w[t] for w in want]), dtype, 0.5)
