"""One sequence in bf16 at widths that are whole multiples of 512 (the register-held projections of a step): stream counts, norm
groups below, at and above a 512-wide piece, every layer kind, odd output counts, argmax, against the plain oracle."""
import numpy as np
import pytest
import torch

import decoder_cases as C
import raritar_cases as R
from decoder_helpers import build, close, oracle, tokens

pytestmark = pytest.mark.gpu


def tuvodra(width, streams, groups, conv=4, vocab=211):
    return C.model([C.mamba(512, 16, 32, conv), C.gru(509), C.attn(6, 2, 64, 64, 20, ff=331), C.mamba(1024, 8, 16, conv, ff=512)],
                   width=width, streams=streams, groups=groups, vocab=vocab)


CASES = {
    "512_one_stream": tuvodra(512, 1, 1, vocab=3001),
    "1024_groups_256": tuvodra(1024, 2, 4),
    "1024_groups_16_three_streams": tuvodra(1024, 3, 64, conv=2),
    "1536_groups_512": tuvodra(1536, 2, 3, conv=1),
    "2048_groups_1024": tuvodra(2048, 2, 2, conv=3, vocab=1027),
    "long_rows": C.model([C.mamba(4096, 4, 8, 4), C.gru(512, ff=8192), C.gru(512, ff=16384)], width=512, streams=2, groups=1),
    "raritar_512": R.model([R.layer(4, 2, 64, 128, 17, keep=3, rot=32, mlp=R.moe(6, 64, 2, 96, identity=1))], width=512),
}


@pytest.mark.parametrize("name", list(CASES))
def test_token_by_token(name):
    cfg = CASES[name]
    eng, W = build(cfg, "bfloat16")
    toks = tokens(cfg, 24, 4)
    want = oracle(cfg).run(cfg, W, toks)
    cache = eng.new_cache(3, 40)
    cache.slab.fill_(0x7F)
    slots = [cache.alloc() for _ in range(3)]
    got, nxt = [], torch.empty(1, dtype=torch.int64, device="cuda")
    for t, tok in enumerate(toks):
        ids = torch.tensor([tok], device="cuda")
        lg = eng.decode(cache, [slots[1]], ids, next_ids=nxt, graph=t % 2 == 1).clone()
        assert int(nxt) == int(lg.argmax())
        got.append(lg[0])
    close(torch.stack(got), np.stack(want), "bfloat16", 0.5)
