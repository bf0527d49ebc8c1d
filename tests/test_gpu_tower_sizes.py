"""The vision tower at widths of the feed-forward that are whole k-tiles of 64 and that are not (fc1's output rows are further apart
than they are long), several batches, and once more after the weights changed."""
import numpy as np
import pytest
import torch

from oracle import paligemma_np as O
from oracle import weights as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ff", [64, 72, 120, 4296, 4352])
def test_tower_feed_forward_widths(ff):
    from pgmi import Engine
    cfg = W.small_config(vision_layers=2, text_layers=1, vocab=1024)
    cfg["vision_config"]["intermediate_size"] = ff
    eng = Engine(cfg, max_batch=2, max_seq=320, max_kv=320)
    rng = np.random.default_rng(ff)
    px = O.bf16(rng.uniform(-1, 1, (2, 3, 224, 224)).astype(np.float32))
    for seed in (5, 6):  # the second load must reach fc2
        eng.fill_synthetic(seed, W.init_policy)
        eng.prepare()
        want = O.siglip_vision(W.synthetic_state_dict_f32(cfg, seed), cfg, px)
        for rows in (2, 1):
            got = eng.vision(torch.from_numpy(px[:rows]).cuda()).float().cpu().numpy()
            # two layers of bf16 activations: the bound of test_vision_tower
            err = np.linalg.norm(got - want[:rows]) / np.linalg.norm(want[:rows])
            assert err < 1e-2, (ff, seed, rows, err)
