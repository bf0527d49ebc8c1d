"""Steps of a few rows in the forms that read weights by whole lines or by dot products, at sizes where their launch rules take
them (bf16; a matrix of 2^21 elements or more whose K is whole turns of the waves), outputs off the tiles of 16 where the layer lets
them be."""
import numpy as np
import pytest
import torch

import decoder_cases as C
import raritar_cases as R
from decoder_helpers import build, close, oracle, tokens

pytestmark = pytest.mark.gpu

# K of 64 times 4 waves times 2, 4 or 8 steps: an input projection with its convolution, a minGRU's three matrices, q|k|v and a gate|up
# of width K; an output projection in 8 slices of K.  (Several matrices go 4 steps at most; of 2,048 and more the one input matrix is left.)
LINES = {
    "turns_of_2": C.model([C.mamba(2050, 5, 9, 4), C.gru(1370), C.attn(16, 8, 128, 128, 20, ff=2052)], width=512, streams=2, groups=2),
    "turns_of_4": C.model([C.mamba(1026, 5, 9, 3), C.gru(700), C.attn(2, 1, 16, 24, 20, ff=1030)], width=1024, streams=1, groups=4),
    "turns_of_8": C.model([C.mamba(516, 5, 9, 5)], width=2048, streams=3, groups=4),
    "slices_of_2": C.model([C.gru(4096)], width=1000, streams=2, groups=1),
    "slices_of_4": C.model([C.gru(8192)], width=512, streams=2, groups=1),
    "slices_of_8": C.model([C.gru(40, ff=16384)], width=512, streams=2, groups=1),
}


@pytest.mark.parametrize("B", [1, 2, 3, 8])
@pytest.mark.parametrize("name", list(LINES))
def test_whole_lines(name, B):
    cfg = LINES[name]
    eng, W = build(cfg, "bfloat16")
    seqs = [tokens(cfg, 5, 30 + r) for r in range(B)]
    want = [oracle(cfg).run(cfg, W, s) for s in seqs]
    cache = eng.new_cache(B + 1, 8)
    slots = [cache.alloc() for _ in range(B + 1)][::-1][:B]
    for t in range(5):
        lg = eng.decode(cache, slots, torch.tensor([s[t] for s in seqs], device="cuda"))
        close(lg, np.stack([w[t] for w in want]), "bfloat16", 0.5)


# gate|up over pieces of 512 of the width, down over those of an expert's ff; the shared expert's gate|up with them where it has whole
# turns of outputs (1,023: not)
@pytest.mark.parametrize("rows", [1, 3, 4, 8])
@pytest.mark.parametrize("width,ff,shared", [(4096, 512, 1024), (1024, 4096, 1024), (2048, 1024, 2048), (1024, 2048, 1023)])
def test_experts_by_dot_products(width, ff, shared, rows):
    cfg = R.model([R.layer(2, 1, 32, 32, 40, rot=16, mlp=R.moe(5, ff, 2, shared, identity=1, groups=(2, 1)))], width=width, vocab=101)
    eng, W = build(cfg, "bfloat16")
    seqs = [tokens(cfg, 4, 50 + r) for r in range(rows)]
    want = [oracle(cfg).run(cfg, W, s) for s in seqs]
    cache = eng.new_cache(rows, 8)
    slots = [cache.alloc() for _ in seqs]
    for t in range(4):
        lg = eng.decode(cache, slots, torch.tensor([s[t] for s in seqs], device="cuda"))
        close(lg, np.stack([w[t] for w in want]), "bfloat16")
