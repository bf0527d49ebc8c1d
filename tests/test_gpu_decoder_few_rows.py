"""Two to sixteen sequences in bf16 where one workgroup walks several groups of outputs (more than 512 of them: the output
matrix, gate|up), at group edges, widths below and at the held 2,048, one input past them, on both sides of the 512 from which it
does, and with every number of steps, whole and not."""
import numpy as np
import pytest
import torch

import decoder_cases as C
from decoder_helpers import build, close, oracle, tokens

pytestmark = pytest.mark.gpu

CASES = {
    "8208_outputs": C.model([C.gru(40, ff=8208)], width=72, vocab=8209, streams=2, groups=3),
    "16400_outputs": C.model([C.gru(24, ff=8193)], width=1000, vocab=16400, streams=1, groups=1),
    "held_2048": C.model([C.gru(16)], width=2048, vocab=9001, streams=2, groups=4),
    "past_2048": C.model([C.gru(16)], width=2056, vocab=8200, streams=2, groups=4),
}
CASES.update({f"width_{w}": C.model([C.gru(24, ff=8200)], width=w, vocab=8201, streams=1, groups=1)
              for w in (504, 512, 520, 768, 1032, 1280, 1400, 1536, 1672, 1792, 2040)})


@pytest.mark.parametrize("B", [2, 7, 16])
@pytest.mark.parametrize("name", list(CASES))
def test_steps(name, B):
    cfg = CASES[name]
    eng, W = build(cfg, "bfloat16")
    seqs = [tokens(cfg, 3, 70 + r) for r in range(B)]
    some = [0, B // 2, B - 1]
    want = [oracle(cfg).run(cfg, W, seqs[r]) for r in some]
    cache = eng.new_cache(B, 8)
    slots = [cache.alloc() for _ in seqs]
    nxt = torch.empty(B, dtype=torch.int64, device="cuda")
    for t in range(3):
        lg = eng.decode(cache, slots, torch.tensor([s[t] for s in seqs], device="cuda"), next_ids=nxt).clone()
        close(lg[some], np.stack([w[t] for w in want]), "bfloat16", 0.5)
        assert torch.equal(nxt, lg.argmax(-1))
