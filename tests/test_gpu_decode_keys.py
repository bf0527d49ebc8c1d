"""Decode steps over random caches at the edges of the attention combine's passes (12 and 48 chunks of 64 keys), against the
numpy oracle with the same cache."""
import numpy as np
import pytest
import torch

from oracle import paligemma_np as O
from oracle import weights as W

pytestmark = pytest.mark.gpu
SEED, CAP = 1234, 3200


@pytest.fixture(scope="module")
def model():
    from pgmi import Engine
    cfg = W.small_config(vision_layers=1, text_layers=2, vocab=4096)
    eng = Engine(cfg, max_batch=3, max_seq=64, max_kv=CAP)
    eng.fill_synthetic(SEED, W.init_policy)
    eng.prepare()
    P = {n: v for n, v in W.synthetic_state_dict_f32(cfg, SEED).items() if n.startswith("language_model")}
    return cfg, eng, P


@pytest.mark.parametrize("B", [1, 2, 3])
@pytest.mark.parametrize("kept", [1, 63, 767, 768, 800, 1535, 1536, 3071, 3072])
def test_step_over_a_random_cache(model, B, kept):
    cfg, eng, P = model
    rng = np.random.default_rng(kept)
    kv = eng.new_kv(B, CAP).zero_()
    rows = O.bf16(rng.standard_normal((2, 2, B, kept, 256)).astype(np.float32))
    kv[:, :, :, :kept] = torch.from_numpy(rows).cuda().bfloat16()
    okv = O.KV()
    okv.k, okv.v = [rows[i, 0][:, None] for i in range(2)], [rows[i, 1][:, None] for i in range(2)]
    ids = rng.integers(3, 4000, size=B).astype(np.int64)
    got = eng.decode(torch.from_numpy(ids).cuda(), kv, kept, kept + 1)
    ref = O.paligemma_decode(P, cfg, ids, okv, kept + 1)[:, -1]
    g = got.cpu().numpy()
    # two bf16 runs of a two-layer model: 1.2e-2 .. 1.7e-2 apart (rounding of q, k, the weights and every activation)
    assert (np.linalg.norm(g - ref, axis=1) / np.linalg.norm(ref, axis=1)).max() < 2.5e-2
    for i in range(2):
        new = kv[i, :, :, kept].float().cpu().numpy()
        want = np.stack([okv.k[i][:, 0, kept], okv.v[i][:, 0, kept]])
        assert np.linalg.norm(new - want) / np.linalg.norm(want) < 2e-2
