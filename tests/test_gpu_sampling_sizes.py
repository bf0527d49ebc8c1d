"""Top-p draws where the selects change form or meet their edges: vocabularies around a block's slice, candidate counts around
those held in registers, ties, mass on one token, nothing to draw from."""
import numpy as np
import pytest
import torch

from oracle import sampling_np as S
from oracle import weights as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from pgmi import Engine
    e = Engine(W.small_config(vision_layers=1, text_layers=1, vocab=1024), max_batch=1, max_seq=64, max_kv=64)
    e.prepare()
    return e


def check(eng, p, top_p, n_u=24):
    us = np.concatenate([np.random.default_rng(len(p)).random(n_u), [0.0, 0.5, 1 - 2 ** -24]]).astype(np.float32)
    x = torch.from_numpy(np.broadcast_to(p, (len(us), len(p))).copy()).cuda()
    tok, kept = eng.sample_top_p(x, top_p, u=torch.from_numpy(us).cuda(), return_kept_mass=True)
    tok, kept = tok.cpu().numpy(), kept.cpu().numpy()
    for i, u in enumerate(us):
        ref, Z, margin = S.sample_top_p(p, top_p, float(u))
        assert abs(kept[i] - Z) <= 2e-6 * Z
        assert tok[i] == ref or margin <= 1e-6 * max(1.0, Z), (i, tok[i], ref)


@pytest.mark.parametrize("top_p", [0.0, 0.3, 0.9, 1.0])
@pytest.mark.parametrize("V", [1, 2, 255, 2047, 2048, 2049, 4097, 300000])
def test_vocabularies(eng, V, top_p):
    p = np.random.default_rng(V).random(V).astype(np.float32) ** 6
    check(eng, (p / p.sum(dtype=np.float64)).astype(np.float32), top_p)


# equal probabilities: every token a candidate, ties resolved by index; up to 256 are ranked, 2,048 stay in LDS
@pytest.mark.parametrize("n", [1, 7, 255, 256, 257, 2047, 2048, 2049, 5000])
def test_ties(eng, n):
    p = np.zeros(6000, np.float32)
    p[np.random.default_rng(n).permutation(6000)[:n]] = np.float32(1.0 / n)
    check(eng, p, 0.7)


def test_mass_at_the_cut_off(eng):
    """Sums of exact binary fractions that reach p itself, where fp32 decides which token is the last."""
    p = np.array([0.5, 0.25, 0.125, 0.0625, 0.0625] + [0.0] * 11, np.float32)
    for top_p in (0.5, 0.75, 0.875, 0.9375, 1.0, 0.50000006):
        check(eng, p, top_p)


def test_the_cut_off_where_sums_of_doubles_round(eng):
    """Masses whose sum passes p by 1.25 half-units of a double: the token that passes it is past p by the sum of all up to it, and
    not past it by the rounded sum of those before it plus its own."""
    rng = np.random.default_rng(4)
    unit = 2 ** 56  # every mass is a whole number of 2^-56
    half, target = unit // 2, unit // 2 + 5
    masses, total = [half - unit // 2 ** 25], half - unit // 2 ** 25
    while target - total >= 2 ** 23:  # of 2^-33 to 2^-32
        masses.append(int(rng.integers(2 ** 23, 2 ** 24)))
        total += masses[-1]
    last = target - total
    assert 2 ** 22 <= last < 2 ** 23 and len(masses) < 250
    before = float(np.float64(total) * 2.0 ** -56)
    assert before + last * 2.0 ** -56 <= 0.5 < float(np.float64(target) * 2.0 ** -56)
    p = np.full(1 << 20, 2.0 ** -35, np.float32)  # and a tail of 3e-5
    p[0] = 0.0
    at = rng.permutation(np.arange(1, 1 << 20))[:len(masses) + 2]
    p[at] = (np.array(masses + [last, 2 ** 22], np.float64) * 2.0 ** -56).astype(np.float32)
    us = torch.tensor([0.0, 0.3, 1 - 2 ** -24], device="cuda")
    tok, kept = eng.sample_top_p(torch.from_numpy(p).cuda().expand(3, -1).contiguous(), 0.5, u=us, return_kept_mass=True)
    assert ((kept.double() - 0.5).abs() < 1e-7).all()
    assert tok[0] == at[0] and tok[1] == at[0] and int(tok[2]) in set(at.tolist())


def test_nothing_and_not_a_number(eng):
    u = torch.tensor([0.3, 0.3, 0.3], device="cuda")
    x = torch.zeros((3, 5000), device="cuda")
    x[1, 4321], x[2, 17], x[2, 18] = float("nan"), -1.0, 0.25
    tok, kept = eng.sample_top_p(x, 0.9, u=u, return_kept_mass=True)
    assert tok.tolist() == [0, 0, 18] and kept.tolist() == [0.0, 0.0, 0.25]
