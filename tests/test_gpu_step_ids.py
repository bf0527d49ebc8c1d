"""Replayed decode steps whose token ids come from a tensor of their own at every step, or fed back in place, against eager steps:
the launch that reads them stands in front of the graph, or in it."""
import pytest
import torch

import decoder_cases as C
import raritar_cases as R
from decoder_helpers import build
from oracle import weights as W

pytestmark = pytest.mark.gpu
STEPS = 6
DECODERS = {
    "streams": C.MIXED["a"],
    "plain": R.model([R.layer(4, 2, 64, 128, 17, keep=3, rot=32, mlp=R.moe(6, 64, 2, 96, identity=1))], width=512),
}


@pytest.mark.parametrize("rows", [1, 3, 17])
@pytest.mark.parametrize("name", list(DECODERS))
def test_decoder(name, rows):
    cfg = DECODERS[name]
    eng, _ = build(cfg, "bfloat16")
    g = torch.Generator("cuda").manual_seed(rows)
    ids = [torch.randint(0, cfg["vocab"], (rows,), device="cuda", generator=g) for _ in range(STEPS)]
    out = {}
    for graph in (False, True):
        cache = eng.new_cache(rows, 32)
        slots = [cache.alloc() for _ in range(rows)]
        lg, nxt, got = torch.empty((rows, cfg["vocab"]), device="cuda"), torch.empty_like(ids[0]), []
        for t in ids:
            eng.decode(cache, slots, t, logits=lg, next_ids=nxt, graph=graph)
            got += [lg.clone(), nxt.clone()]
        for t in ids[:3]:  # two steps a call: the second reads what the first picked
            eng.decode(cache, slots, t, n_steps=2, logits=lg, next_ids=nxt, graph=graph)
            got += [lg.clone(), nxt.clone()]
        for _ in range(4):  # in place
            eng.decode(cache, slots, nxt, logits=lg, next_ids=nxt, graph=graph)
            got += [lg.clone(), nxt.clone()]
        out[graph] = got
    assert all(torch.equal(a, b) for a, b in zip(out[False], out[True]))


@pytest.mark.parametrize("rows", [1, 2, 3])
def test_text_model(rows):
    from pgmi import Engine
    cfg = W.small_config(vision_layers=1, text_layers=2, vocab=2048)
    eng = Engine(cfg, max_batch=3, max_seq=64, max_kv=128)
    eng.fill_synthetic(11, W.init_policy)
    eng.prepare()
    g = torch.Generator("cuda").manual_seed(rows)
    ids = [torch.randint(3, 1900, (rows,), device="cuda", generator=g) for _ in range(STEPS)]
    out = {}
    for graph in (False, True):
        kv = eng.new_kv(rows, 128).zero_()
        lg, nxt, got, at = torch.empty((rows, 2048), device="cuda"), torch.empty_like(ids[0]), [], 0
        for t in ids:
            eng.decode(t, kv, at, at + 1, logits=lg, next_ids=nxt, graph=graph)
            at += 1
            got += [lg.clone(), nxt.clone()]
        for _ in range(4):
            eng.decode(nxt, kv, at, at + 1, logits=lg, next_ids=nxt, graph=graph)
            at += 1
            got += [lg.clone(), nxt.clone()]
        out[graph] = got + [kv]
    # (eager steps size their attention by the keys there are, replayed ones by the cache: its partials may join in another order)
    for a, b in zip(out[False], out[True]):
        if a.dtype is torch.int64:
            assert torch.equal(a, b)
        else:
            assert float((a.float() - b.float()).norm() / b.float().norm()) < 1e-2
