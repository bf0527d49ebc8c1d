"""Layered decoders on the MI355X against the plain float64 oracle (oracle/decoder_np.py): each mechanism alone, whole
prompts, portions, single tokens, batches of unequal sequences, reused slots, window edges, long decoding, greedy
generation through the engine's own entry point, and the trace runner."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import decoder_cases as C
from decoder_helpers import DTYPES, REPO, TOL, build, close, feed, oracle, rel, save, tokens
from oracle import decoder_np as O

pytestmark = pytest.mark.gpu
ALL = {**C.MECHANISMS, **{"mixed_" + k: v for k, v in C.MIXED.items()}}


# ---------------------------------------------------------------- products
@pytest.mark.parametrize("M,N,K", [(1, 80, 16), (5, 33, 8), (70, 203, 104), (300, 515, 264), (130, 4096, 1024),
                                   (1100, 2304, 1088), (2048, 6144, 2048), (64, 160, 4096)])
@pytest.mark.parametrize("act", [0, 2])
def test_matmul_any_shape(M, N, K, act):
    import ctypes

    from pgmi import _native as N_
    if act == 2:  # the fp32 form has one tile shape: smaller sizes say as much
        M, N = min(M, 200), min(N, 600)
    eng, _ = build(C.MECHANISMS["gru"], "float32")
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn((M, K + 8), generator=g, device="cuda")
    A = A.bfloat16() if act == 0 else A
    W = torch.randn((2 * N, K), generator=g, device="cuda").bfloat16()
    bias = torch.randn(N, generator=g, device="cuda").bfloat16()
    ref = A[:, :K].float() @ W.float().t()
    tol = 2e-5 * K ** 0.5
    ldo = (N + 7) // 8 * 8
    dt = torch.bfloat16 if act == 0 else torch.float32
    scratch = torch.empty((M, 2 * N), device="cuda")
    s = N_.stream_handle(eng.device)

    def call(mode, out, ld, b=None):
        sp = ctypes.c_int()
        N_.check(eng.lib.pgmi_op_matmul(eng.ctx, A.data_ptr(), K + 8, W.data_ptr(), K, M, N, K, act, mode, N_.ptr(b),
                                        out.data_ptr(), ld, out.numel() * out.element_size(), scratch.data_ptr(),
                                        ctypes.byref(sp), s))
        return sp.value

    out = torch.full((M, ldo), float("nan"), dtype=dt, device="cuda")
    call(0, out, ldo, bias)
    want = ref[:, :N] + bias.float()
    assert ((out[:, :N].float() - want).abs() <= (8e-3 * want.abs() + 1e-2 if act == 0 else tol)).all()
    assert (out[:, N:] == 0).all()
    out = torch.full((M, N), float("nan"), device="cuda")
    call(1, out, N)
    assert (out - ref[:, :N]).abs().max() <= tol
    slabs = torch.full((8, M, N), float("nan"), device="cuda")
    sp = call(2, slabs, N)
    assert 1 <= sp <= 8 and (slabs[:sp].sum(0) - ref[:, :N]).abs().max() <= tol
    out = torch.full((M, ldo), float("nan"), dtype=dt, device="cuda")
    call(3, out, ldo)
    want = torch.nn.functional.silu(ref[:, :N]) * ref[:, N:]
    assert ((out[:, :N].float() - want).abs() <= (8e-3 * want.abs() + 1e-2 if act == 0 else 4 * tol * (1 + want.abs()))).all()
    assert (out[:, N:] == 0).all()


@pytest.mark.parametrize("M,N,K", [(40, 2048, 4096), (500, 2561, 2048), (1000, 8190, 1088), (1540, 4096, 128), (1540, 6146, 2048),
                                   (1537, 8192, 2048), (3000, 4095, 1024), (3000, 2048, 4096), (257, 8192, 2056)])
def test_matmul_forms(M, N, K):
    """Sizes at which the least predicted time is each form's in turn (32 and 96 x 64, 128 x 128, 128 to 256 x 256), whole or in
    K slices, with rows, columns and k past the last tile.  (K <= 4096: K / 32 roundings of a sum of size sqrt(K) add up to
    about 2^-24 K / sqrt(32), 5 sigma of it over the outputs 2e-7 K on either side; 2e-5 sqrt(K) covers both up to K = 2500
    and, as partial sums are smaller than the last, 4096.  At 16384, 3.5e-3 stood against 2.6e-3.)"""
    test_matmul_any_shape(M, N, K, 0)


# ---------------------------------------------------------------- mechanisms and whole models
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(ALL))
def test_layers_and_logits_of_a_prompt(name, dtype):
    cfg = ALL[name]
    eng, W = build(cfg, dtype)
    toks = tokens(cfg, 150)
    taps = []
    want = O.run(cfg, W, toks, taps=taps)
    cache = eng.new_cache(2, 200)
    got = torch.zeros((len(cfg["layers"]), len(toks), cfg["width"]), device="cuda")
    lg = eng.forward(cache, [cache.alloc()], toks, [len(toks)], want=range(len(toks)), taps=got)
    for i, t in enumerate(np.stack(taps, 1)):
        close(got[i], t, dtype)
    close(lg, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inner,dt_rank,rows", [(1032, 24, 600), (2048, 64, 1301)])
def test_steps_and_scan_of_many_rows(inner, dt_rank, rows, dtype):
    """The step sizes' product on the tiles that many rows take (one with columns past the last tile), and their scan."""
    cfg = C.model([C.mamba(inner, 16, dt_rank, 4)], width=64, streams=1, groups=1)
    eng, W = build(cfg, dtype)
    toks = tokens(cfg, rows, 5)
    cache = eng.new_cache(1, rows)
    close(eng.step(cache, [cache.alloc()], [toks], want=range(rows)), O.run(cfg, W, toks), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inner,states", [(16, 16), (48, 9), (64, 12), (72, 16), (40, 13)])
def test_scan_of_sequences_walked_whole(inner, states, dtype):
    """Sequences that end just before, on and just after a block of 16 and a stage of 64 rows, of channels that are and are not whole
    vectors and workgroups, then the next portions from the states that were left."""
    cfg = C.model([C.mamba(inner, states, 8, 4)], width=64, streams=1, groups=1)
    eng, W = build(cfg, dtype)
    first, then = [1, 15, 16, 17, 63, 64, 65, 129, 190], [65, 1, 128, 16, 2, 64, 63, 17, 3]
    seqs = [tokens(cfg, a + b, 40 + r) for r, (a, b) in enumerate(zip(first, then))]
    cache = eng.new_cache(len(seqs), 256)
    slots = [cache.alloc() for _ in seqs]
    a = eng.forward(cache, slots, [t for s, n in zip(seqs, first) for t in s[:n]], first, want=range(sum(first))).clone()
    b = eng.forward(cache, slots, [t for s, n in zip(seqs, first) for t in s[n:]], then, want=range(sum(then))).clone()
    for r, s in enumerate(seqs):
        i, j = sum(first[:r]), sum(then[:r])
        close(torch.cat([a[i:i + first[r]], b[j:j + then[r]]]), O.run(cfg, W, s), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("states", [9, 16])
def test_scan_of_states_that_do_not_last(states, dtype):
    """A_log = 90, whose decay per step of 1 is not finite in fp32: such a state keeps its last input alone, whether or not the
    sequence ends with a block of 16 or a stage of 64 rows, and the next portions and single tokens go on from it."""
    cfg = C.model([C.mamba(48, states, 8, 4)], width=64, streams=1, groups=1)
    weights = oracle(cfg).random_weights(cfg, 3)
    name = next(n for n in weights if n.endswith("mix.A_log"))
    weights[name] = weights[name].copy()
    weights[name][::3, ::2] = 90.0
    eng, W = build(cfg, dtype, weights=weights)
    first, then = [1, 15, 16, 17, 63, 64, 65, 130], [20, 1, 16, 3, 64, 65, 2, 15]
    seqs = [tokens(cfg, a + b + 2, 90 + r) for r, (a, b) in enumerate(zip(first, then))]
    cache = eng.new_cache(len(seqs), 256)
    slots = [cache.alloc() for _ in seqs]
    a = eng.forward(cache, slots, [t for s, n in zip(seqs, first) for t in s[:n]], first, want=range(sum(first))).clone()
    b = eng.forward(cache, slots, [t for s, n, m in zip(seqs, first, then) for t in s[n:n + m]], then, want=range(sum(then))).clone()
    c = [eng.step(cache, slots, [[s[k]] for s in seqs]).clone() for k in (-2, -1)]
    for r, s in enumerate(seqs):
        i, j = sum(first[:r]), sum(then[:r])
        close(torch.cat([a[i:i + first[r]], b[j:j + then[r]], c[0][r:r + 1], c[1][r:r + 1]]), O.run(cfg, W, s), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mixer", ["mamba", "gru"])
def test_walked_sequences_beside_one_that_is_not_finite(mixer, dtype):
    """A token whose embedding is not a number, last or in the middle of its sequence: what comes before it and the other sequences
    are what they are without it, what comes after it is no number."""
    cfg = C.model([C.mamba(48, 16, 8, 4) if mixer == "mamba" else C.gru(48)], width=64, streams=1, groups=1)
    weights = oracle(cfg).random_weights(cfg, 3)
    weights["embed"] = weights["embed"].copy()
    weights["embed"][5] = np.nan
    eng, _ = build(cfg, dtype, weights=weights)
    lens, bad = [33, 70, 129, 20], {1: 69, 3: 7}
    seqs = [[t + 1 if t == 5 else t for t in tokens(cfg, n + 9, 95 + r)] for r, n in enumerate(lens)]
    got = []
    for planted in (False, True):
        cache = eng.new_cache(len(lens), 160)
        slots = [cache.alloc() for _ in lens]
        now = [[5 if planted and bad.get(r) == i else t for i, t in enumerate(s)] for r, s in enumerate(seqs)]
        a = eng.forward(cache, slots, [t for s, n in zip(now, lens) for t in s[:n]], lens, want=range(sum(lens))).clone()
        b = eng.forward(cache, slots, [t for s, n in zip(now, lens) for t in s[n:]], [9] * len(lens), want=range(9 * len(lens))).clone()
        got.append([torch.cat([a[sum(lens[:r]):sum(lens[:r + 1])], b[9 * r:9 * r + 9]]) for r in range(len(lens))])
    for r in range(len(lens)):
        sound = bad.get(r, lens[r] + 9)
        finite = torch.isfinite(got[0][r]).all(0)  # (the tied output matrix has the token's row too)
        assert int(finite.sum()) == cfg["vocab"] - 1
        assert torch.equal(got[0][r][:sound, finite], got[1][r][:sound, finite])
        assert torch.isnan(got[1][r][sound:]).all()


@pytest.mark.parametrize("mixer,width,rows,seed,most", [("mamba", 512, 700, 3, 5.5e-7), ("gru", 512, 900, 4, 1.3e-6)])
def test_walked_states_that_last(mixer, width, rows, seed, most):
    """fp32 states that last for hundreds of rows, whose roundings add up: the error of the last 100 rows' logits, rms, mean over the
    rows.  Scan: 3.6e-7 in runs and as it is walked, of which 3.4e-7 are the products around it; 7.8e-7 step by step.  minGRU: 8.5e-7 as
    it is walked, 1.7e-6 row by row.  The bounds lie half way."""
    cfg = C.model([C.mamba(width, 16, 8, 4) if mixer == "mamba" else C.gru(width)], width=64, streams=1, groups=1)
    weights = oracle(cfg).random_weights(cfg, seed)
    for name in weights:
        leaf = name.split(".", 1)[-1]
        if leaf in ("mix.A_log", "mix.z.b", "mix.dt.b"):
            weights[name] = np.full_like(weights[name], -2.0 if leaf == "mix.dt.b" else -6.0)
        elif leaf in ("mix.z", "mix.D"):
            weights[name] = np.zeros_like(weights[name])
    eng, W = build(cfg, "float32", weights=weights)
    toks = tokens(cfg, rows, seed)
    cache = eng.new_cache(1, rows)
    got = eng.forward(cache, [cache.alloc()], toks, [rows], want=range(rows))
    assert rel(got, O.run(cfg, W, toks))[-100:].mean() <= most


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inner", [64, 1032])
def test_scan_in_runs_as_walked(inner, dtype):
    """2,300 rows of few channels go in runs, with whole and broken blocks of rows; in portions of 230 they are walked."""
    cfg = C.model([C.mamba(inner, 16, 8, 4)], width=64, streams=1, groups=1)
    eng, _ = build(cfg, dtype)
    toks = tokens(cfg, 2300, 9)
    cache = eng.new_cache(2, 2304)
    whole = eng.forward(cache, [cache.alloc()], toks, [len(toks)], want=range(len(toks))).clone()
    close(feed(eng, cache, cache.alloc(), toks, [230]), whole.double().cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [16, 48, 56, 13])
def test_gru_of_sequences_walked_whole(width, dtype):
    """Sequences that end just before, on and just after a wave's 16 rows, the walker's 32 and a stage's 128, of one to four stages,
    of channels that are and are not whole vectors and workgroups, then the next portions from the states that were left."""
    cfg = C.model([C.gru(width)], width=64, streams=1, groups=1)
    eng, W = build(cfg, dtype)
    first, then = [1, 15, 17, 32, 33, 127, 128, 129, 256, 257, 400], [129, 1, 128, 16, 31, 64, 33, 17, 3, 270, 2]
    seqs = [tokens(cfg, a + b, 60 + r) for r, (a, b) in enumerate(zip(first, then))]
    cache = eng.new_cache(len(seqs), 640)
    slots = [cache.alloc() for _ in seqs]
    a = eng.forward(cache, slots, [t for s, n in zip(seqs, first) for t in s[:n]], first, want=range(sum(first))).clone()
    b = eng.forward(cache, slots, [t for s, n in zip(seqs, first) for t in s[n:]], then, want=range(sum(then))).clone()
    for r, s in enumerate(seqs):
        i, j = sum(first[:r]), sum(then[:r])
        close(torch.cat([a[i:i + first[r]], b[j:j + then[r]]]), O.run(cfg, W, s), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_gru_in_runs_as_walked(dtype):
    """4,100 rows of few channels go in runs; in portions of 410 they are walked."""
    cfg = C.model([C.gru(64)], width=64, streams=1, groups=1)
    eng, _ = build(cfg, dtype)
    toks = tokens(cfg, 4100, 9)
    cache = eng.new_cache(2, 4112)
    whole = eng.forward(cache, [cache.alloc()], toks, [len(toks)], want=range(len(toks))).clone()
    close(feed(eng, cache, cache.alloc(), toks, [410]), whole.double().cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,kv", [(8, 8), (12, 4), (6, 1)])
@pytest.mark.parametrize("lens", [[700, 33, 900, 129, 500], [64, 1, 65]])
def test_attention_of_several_prompts(lens, heads, kv, dtype):
    """More pieces than CUs and fewer, in the order of their keys, as each sequence's alone."""
    cfg = C.model([C.attn(heads, kv, 16, 16, 300)], width=64, streams=1, groups=1)
    eng, _ = build(cfg, dtype)
    seqs = [tokens(cfg, n, 70 + r) for r, n in enumerate(lens)]
    cache = eng.new_cache(len(lens) + 1, 1024)
    got = eng.forward(cache, [cache.alloc() for _ in lens], [t for s in seqs for t in s], lens, want=range(sum(lens))).clone()
    for r, s in enumerate(seqs):
        alone = cache.alloc()
        one = eng.forward(cache, [alone], s, [len(s)], want=range(len(s)))
        cache.free(alone)
        close(got[sum(lens[:r]):sum(lens[:r + 1])], one.double().cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(ALL))
def test_token_by_token(name, dtype):
    cfg = ALL[name]
    eng, W = build(cfg, dtype)
    toks = tokens(cfg, 100, 1)
    cache = eng.new_cache(2, 128)
    got = feed(eng, cache, cache.alloc(), toks, [1], graph=True)
    close(got, O.run(cfg, W, toks), dtype)


@pytest.mark.parametrize("heads,kv,dim,vdim,window", [(8, 2, 64, 64, 900), (6, 3, 24, 36, 150), (4, 1, 128, 128, 192),
                                                      (2, 1, 256, 256, 700), (4, 2, 96, 128, 129), (3, 3, 40, 200, 300)])
@pytest.mark.parametrize("lens", [[129], [192, 1], [257, 64, 130], [321]])
def test_attention_of_two_teams(heads, kv, dim, vdim, window, lens):
    """Tiles of an odd and an even number of key tiles, a team without one, windows that leave keys behind, padded and whole heads;
    then portions over the keys that are there."""
    cfg = C.model([C.attn(heads, kv, dim, vdim, window)], width=72, streams=1, groups=1)
    eng, W = build(cfg, "bfloat16")
    seqs = [tokens(cfg, n + 200, 60 + r) for r, n in enumerate(lens)]
    cache = eng.new_cache(len(lens), 640)
    slots = [cache.alloc() for _ in lens]
    a = eng.forward(cache, slots, [t for s, n in zip(seqs, lens) for t in s[:n]], lens, want=range(sum(lens))).clone()
    b = eng.forward(cache, slots, [t for s, n in zip(seqs, lens) for t in s[n:]], [200] * len(lens), want=range(200 * len(lens))).clone()
    for r, (s, n) in enumerate(zip(seqs, lens)):
        i = sum(lens[:r])
        close(torch.cat([a[i:i + n], b[200 * r:200 * (r + 1)]]), O.run(cfg, W, s), "bfloat16")


@pytest.mark.parametrize("heads,kv,dim,vdim,window", [(8, 2, 64, 64, 900), (6, 2, 40, 256, 1500), (16, 4, 32, 128, 1990),
                                                      (128, 1, 16, 8, 300), (4, 4, 24, 128, 2500)])
def test_one_row_merges_its_attention(heads, kv, dim, vdim, window):
    """One sequence's steps whose output projection merges the attention's 1 to 16 partials itself (K of 512 to 2048; with 20
    they keep their launch): empty partials, and windows that leave the first keys behind."""
    cfg = C.model([C.attn(heads, kv, dim, vdim, window, ff=72), C.attn(heads, kv, dim, vdim, 40)], width=96, streams=2, groups=2)
    eng, W = build(cfg, "bfloat16")
    toks = tokens(cfg, 420, 6)
    cache = eng.new_cache(2, 2600)
    got = feed(eng, cache, cache.alloc(), toks, [1, 1, 1, 140, 1, 1, 270, 1], graph=True)
    close(got, O.run(cfg, W, toks), "bfloat16")


@pytest.mark.parametrize("window,at", [(900, 10), (900, 415), (1990, 300), (100, 400), (2500, 10)])
def test_one_row_over_a_key_that_is_not_a_number(window, at):
    """Scores that are not numbers take the heads that meet them out of a step, whichever of the attention's partials they are
    in (the others' average would look like an answer): 8 and 16 partials merged by the output projection, one, and 20 that
    keep their launch."""
    cfg = C.model([C.attn(8, 2, 64, 64, window)], width=96, streams=2, groups=2)
    W = O.random_weights(cfg, 3)
    bad = cfg["vocab"] - 1
    broken = {k: np.array(v) for k, v in W.items()}
    broken["embed"][bad] = np.nan
    eng, _ = build(cfg, "bfloat16", weights=broken)
    toks = [t if t != bad else 0 for t in tokens(cfg, 421, 9)]
    want = O.run(cfg, O.Weights(dict(W, **{"l0.mix.o": np.zeros_like(W["l0.mix.o"])})), toks)[-1:, :bad]
    toks[at] = bad
    cache = eng.new_cache(1, 2600)
    slot = cache.alloc()
    eng.step(cache, [slot], [toks[:-1]])
    close(eng.step(cache, [slot], [toks[-1:]])[:, :bad], want, "bfloat16")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("sizes", [[2], [3], [1, 2, 5, 4], [17, 1, 40], [63, 2], [64], [65, 64], [130, 3]])
@pytest.mark.parametrize("name", ["mixed_a", "mixed_b"])
def test_portions(name, sizes, dtype):
    cfg = ALL[name]
    eng, W = build(cfg, dtype)
    toks = tokens(cfg, 200, 2)
    cache = eng.new_cache(3, 256)
    cache.alloc()
    got = feed(eng, cache, cache.alloc(), toks, sizes)
    close(got, O.run(cfg, W, toks), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lens", [[1, 70], [5, 1, 130], [64, 65, 63, 2, 129], [2 + r for r in range(17)]])
def test_unequal_batch_then_decoding(lens, dtype):
    """Prompts of unequal lengths in one step, then single tokens together; sequences leave one by one, so every
    batch size down to one is decoded (every form of the decode projections: one row, up to 16, more)."""
    cfg = C.MIXED["a"]
    eng, W = build(cfg, dtype)
    extra = 12
    seqs = [tokens(cfg, n + extra, 10 + n) for n in lens]
    want = [O.run(cfg, W, s) for s in seqs]
    cache = eng.new_cache(17, 160)
    slots = [cache.alloc() for _ in lens]
    lg = eng.step(cache, slots, [s[:n] for s, n in zip(seqs, lens)], want=list(range(sum(lens))))
    close(lg, np.concatenate([w[:n] for w, n in zip(want, lens)]), dtype)
    live = list(range(len(lens)))
    for t in range(extra):
        if t and t % 3 == 0 and len(live) > 1:
            cache.free(slots[live.pop(0)])
        lg = eng.step(cache, [slots[r] for r in live], [[seqs[r][lens[r] + t]] for r in live])
        close(lg, np.stack([want[r][lens[r] + t] for r in live]), dtype)


def test_mixed_portions_and_single_tokens_in_one_step():
    cfg = C.MIXED["b"]
    eng, W = build(cfg, "float32")
    seqs = [tokens(cfg, 90, 20), tokens(cfg, 90, 21), tokens(cfg, 90, 22)]
    want = [O.run(cfg, W, s) for s in seqs]
    cache = eng.new_cache(3, 100)
    slots = [cache.alloc() for _ in seqs]
    at = [0, 0, 0]
    for ns in ([40, 2, 7], [1, 30, 2], [2, 1, 66], [47, 57, 15]):
        lg = eng.step(cache, slots, [s[a:a + n] for s, a, n in zip(seqs, at, ns)], want=list(range(sum(ns))))
        close(lg, np.concatenate([w[a:a + n] for w, a, n in zip(want, at, ns)]), "float32")
        at = [a + n for a, n in zip(at, ns)]


@pytest.mark.parametrize("dtype", DTYPES)
def test_batch_equals_alone(dtype):
    cfg = C.MIXED["b"]
    eng, _ = build(cfg, dtype)
    seqs = [tokens(cfg, n, 30 + n) for n in (3, 64, 90, 17)]
    cache = eng.new_cache(6, 128)
    slots = [cache.alloc() for _ in seqs]
    together = eng.step(cache, slots, seqs).clone()
    for s in slots:
        cache.free(s)
    for r, s in enumerate(seqs):
        slot = cache.alloc()
        alone = eng.step(cache, [slot], [s])
        close(together[r:r + 1], alone.double().cpu().numpy(), dtype, 0.5)
        cache.free(slot)


def test_freed_slots_start_clean():
    cfg = C.MIXED["a"]
    eng, W = build(cfg, "float32")
    cache = eng.new_cache(2, 120)
    cache.slab.fill_(0x7F)  # NaN-like patterns everywhere: nothing of an old state may be read
    for k in range(4):
        toks = tokens(cfg, 30 + 20 * k, 40 + k)
        slot = cache.alloc()
        sizes = [[len(toks)], [1], [2], [25, 1]][k]
        close(feed(eng, cache, slot, toks, sizes), O.run(cfg, W, toks), "float32")
        cache.free(slot)
    with pytest.raises(ValueError):
        cache.free(slot)
    with pytest.raises(ValueError):
        eng.step(cache, [slot], [[1]])


# ---------------------------------------------------------------- window edges, far keys
def standout(cfg, n_pairs, seed=6):
    """A single attention layer over three-part embeddings: the first part is a token's query code, the second its key
    code, the third feeds the values.  Tokens come in pairs (key vocab - 2k - 2, query vocab - 2k - 1) whose codes
    agree, so that one score stands out among all keys of the window."""
    W = O.random_weights(cfg, seed)
    P = cfg["width"] // 3
    for k in range(n_pairs):
        W["embed"][cfg["vocab"] - 2 * k - 1][:P] = W["embed"][cfg["vocab"] - 2 * k - 2][P:2 * P]
    m = cfg["layers"][0]["mixer"]
    code = O.random_weights({**cfg, "vocab": 4}, seed + 1)["l0.mix.k"][:, :P].reshape(m["kv_heads"], m["dim"], P)
    q, k = np.zeros_like(W["l0.mix.q"]), np.zeros_like(W["l0.mix.k"])
    q[:, :P] = np.repeat(code, m["heads"] // m["kv_heads"], 0).reshape(-1, P)
    k[:, P:2 * P] = code.reshape(-1, P)
    W["l0.mix.q"], W["l0.mix.k"] = q, k
    W["l0.mix.v"][:, :2 * P] = 0
    for n in ("l0.mix.q.b", "l0.mix.k.b"):
        W[n] = W[n] * 0
    W["l0.mix.r1"] = W["l0.mix.r1"] * 0 + 0.25
    W["l0.mix.v"], W["l0.mix.o"] = W["l0.mix.v"] * 2, W["l0.mix.o"] * 2
    return W


def plain_tokens(cfg, n, n_pairs, seed):
    return [int(t) for t in np.random.default_rng(seed).integers(0, cfg["vocab"] - 2 * n_pairs, n)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("size,heads,kv,dim,vdim", [(2, 4, 2, 32, 24), (63, 3, 1, 64, 64), (64, 4, 4, 40, 72),
                                                    (65, 8, 2, 96, 96), (200, 6, 3, 48, 128)])
def test_window_edges(size, heads, kv, dim, vdim, dtype, monkeypatch):
    """A matching key exactly at the window's last place, one place outside, and near them: in a prompt and decoded.
    The oracle with its window one wider or narrower must be far away at those positions."""
    cfg = C.model([C.attn(heads, kv, dim, vdim, size, scale=13.0 / dim)], width=96, streams=2, groups=3, vocab=400,
                  escale=1.5)
    Wr = standout(cfg, 6)
    eng, W = build(cfg, dtype, weights=Wr)
    n = 3 * size + 80
    toks = plain_tokens(cfg, n, 6, 7)
    pairs = []
    for k, dist in enumerate((size - 1, size, size - 1, size, max(1, size - 2), size + 1)):
        i = n - 1 - 6 * k
        toks[i - dist], toks[i] = cfg["vocab"] - 2 * k - 2, cfg["vocab"] - 2 * k - 1
        pairs.append(i)
    want = O.run(cfg, W, toks)
    keys = O.window_keys
    for wrong in (-1, 1):
        monkeypatch.setattr(O, "window_keys", lambda i, s, w=wrong: keys(i, max(1, s + w)))
        off = rel(O.run(cfg, W, toks), want)[pairs].max()
        monkeypatch.setattr(O, "window_keys", keys)
        assert off > 3 * TOL[dtype], off
    cache = eng.new_cache(4, n)
    slot = cache.alloc()
    close(eng.step(cache, [slot], [toks], want=list(range(n))), want, dtype)
    cache.free(slot)
    slot, cut = cache.alloc(), n - 40
    got = feed(eng, cache, slot, toks, [cut, 1], graph=True)
    close(got, want, dtype)
    cache.free(slot)
    slots = [cache.alloc() for _ in range(3)]  # the batched decode form
    eng.step(cache, slots, [toks[:cut]] * 3)
    for t in range(cut, n):
        lg = eng.step(cache, slots, [[toks[t]]] * 3)
        close(lg, np.stack([want[t]] * 3), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_far_key_among_hundreds(dtype):
    """One matching key hundreds of tokens back, at a tile border or not, inside a window of many tiles."""
    cfg = C.model([C.attn(4, 2, 64, 64, 700, scale=14.0 / 64)], width=96, streams=2, groups=3, vocab=900, escale=1.5)
    Wr = standout(cfg, 5)
    eng, W = build(cfg, dtype, weights=Wr)
    toks = plain_tokens(cfg, 760, 5, 9)
    places = ((759, 64), (750, 63), (741, 128), (701, 2), (699, 0))
    for k, (i, j) in enumerate(places):
        toks[j], toks[i] = cfg["vocab"] - 2 * k - 2, cfg["vocab"] - 2 * k - 1
    want = O.run(cfg, W, toks)
    lost = list(toks)
    for _, j in places:
        lost[j] = 5
    off = rel(O.run(cfg, W, lost), want)[[i for i, _ in places]].min()
    assert off > 3 * TOL[dtype], off
    cache = eng.new_cache(2, 800)
    close(eng.step(cache, [cache.alloc()], [toks], want=list(range(760))), want, dtype)
    got = feed(eng, cache, cache.alloc(), toks, [690, 1], graph=True)
    close(got[690:], want[690:], dtype)


# ---------------------------------------------------------------- long decoding, graphs, generation
@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(dtype):
    cfg = C.MIXED["a"]
    eng, W = build(cfg, dtype)
    toks = tokens(cfg, 420, 50)
    cache = eng.new_cache(2, 420)
    got = feed(eng, cache, cache.alloc(), toks, [5, 1], graph=True)
    close(got, O.run(cfg, W, toks), dtype)


@pytest.mark.parametrize("B", [1, 2, 3, 6])
def test_replayed_steps_equal_eager_steps(B):
    """Every replay against the eager step: same kernels, same bits; slots change between replays."""
    cfg = C.MIXED["b"]
    eng, _ = build(cfg, "bfloat16")
    prompts = [tokens(cfg, 5 + 9 * r, 60 + r) for r in range(B)]
    ca, cb = eng.new_cache(B + 2, 128), eng.new_cache(B + 2, 128)
    sa, sb = [ca.alloc() for _ in range(B)], [cb.alloc() for _ in range(B)][::-1]
    eng.step(ca, sa, prompts)
    eng.step(cb, sb, prompts)
    ia = torch.arange(B, device="cuda") * 3 + 1
    ib = ia.clone()
    la = torch.empty((B, cfg["vocab"]), device="cuda")
    lb = torch.empty((B, cfg["vocab"]), device="cuda")
    for t in range(9):
        eng.decode(ca, sa, ia, logits=la, next_ids=ia, graph=True)
        x = (la * 2).sum()  # the program's own work between replays
        eng.decode(cb, sb, ib, logits=lb, next_ids=ib, graph=False)
        assert torch.equal(la, lb) and torch.equal(ia, ib), t
        assert torch.isfinite(x)
    # several steps per launch
    rec = torch.empty((4, B), dtype=torch.int64, device="cuda")
    for t in range(3):
        eng.decode(ca, sa, ia, n_steps=4, logits=la, next_ids=ia, tokens=rec, graph=True)
        for k in range(4):
            eng.decode(cb, sb, ib, logits=lb, next_ids=ib, graph=False)
            assert torch.equal(rec[k], ib), (t, k)
        assert torch.equal(la, lb)


@pytest.mark.parametrize("B", [1, 2, 4])
def test_greedy_generation(B):
    """generate() through the registry's engine: the oracle's own greedy tokens (fp32; a token may differ only where
    the oracle's two best logits are within the tolerance)."""
    cfg = C.MIXED["a"]
    eng, W = build(cfg, "float32")
    prompts = [tokens(cfg, n, 70 + n) for n in (4, 37, 12, 81)[:B]]
    n = 21
    out = eng.generate(prompts, n, prefill_tokens=50).cpu().numpy()
    for r in range(B):
        toks, lg = O.greedy(cfg, W, prompts[r], n)
        for t in range(n):
            if out[r, t] != toks[t]:
                top = np.sort(lg[t])
                assert top[-1] - top[-2] < 1e-3 * np.abs(lg[t]).max(), (r, t)
                break


def test_generation_stop_tokens_and_sampling():
    cfg = C.MIXED["a"]
    eng, _ = build(cfg, "bfloat16")
    prompts = [tokens(cfg, 9, 80), tokens(cfg, 30, 81), tokens(cfg, 3, 82)]
    free = eng.generate(prompts, 16).cpu()
    eos = int(free[1, 5])
    out, lens = eng.generate(prompts, 16, eos_token_id=eos, pad_token_id=0, sync_every=4, return_lengths=True)
    for r in range(3):
        hit = (free[r] == eos).nonzero()
        n = int(hit[0]) + 1 if len(hit) else 16
        assert int(lens[r]) == n and torch.equal(out[r, :n].cpu(), free[r, :n])
        assert (out[r, n:] == 0).all()
    g = torch.Generator(device="cuda").manual_seed(5)
    a = eng.generate(prompts, 8, do_sample=True, temperature=0.9, top_p=0.8, generator=g).cpu()
    b = eng.generate(prompts, 8, do_sample=True, temperature=0.9, top_p=0.8,
                     generator=torch.Generator(device="cuda").manual_seed(5)).cpu()
    assert torch.equal(a, b) and int(a.min()) >= 0 and int(a.max()) < cfg["vocab"]
    tiny = eng.generate(prompts, 8, do_sample=True, temperature=0.9, top_p=1e-9).cpu()
    assert torch.equal(tiny, free[:, :8])  # a nucleus of one token is the argmax


# ---------------------------------------------------------------- loading, refusals, the runner
def test_load_model_and_trace_runner(tmp_path):
    import utils
    cfg = C.MIXED["b"]
    Wr = O.random_weights(cfg, 8)
    save(cfg, Wr, tmp_path)
    W = O.Weights(Wr)
    eng = utils.load_model(str(tmp_path), device="cuda:0")
    toks = {"x": tokens(cfg, 40, 90), "y": tokens(cfg, 25, 91), "z": tokens(cfg, 1, 92)}
    want = {k: O.run(cfg, W, v) for k, v in toks.items()}
    cache = eng.new_cache(1, 64)
    close(eng.step(cache, [cache.alloc()], [toks["x"]], want=range(40)), want["x"], "bfloat16")
    del eng
    steps = [({"x": 30, "y": 20, "z": 1}, ["z"])] + [({"x": 1, "y": 1}, [])] * 4 + [({"x": 1, "y": 1}, ["y"])] + \
            [({"x": 1}, [])] * 4 + [({"x": 1}, ["x"])]
    steps.append(({"z": 1}, ["z"]))
    for dtype in DTYPES:
        out = tmp_path / dtype
        out.mkdir()
        at, lines, rows = {}, [], []
        for n, (bring, end) in enumerate(steps):
            if n == len(steps) - 1:
                at["z"] = 0
            entries, w = [], []
            for k, c in bring.items():
                lo = at.get(k, 0)
                places = [] if n == 2 else sorted({0, c - 1})
                entries.append({"id": k + ("2" if n == len(steps) - 1 else ""), "tokens": toks[k][lo:lo + c], "want": places})
                w += [want[k][lo + p] for p in places]
                at[k] = lo + c
            ends = [e + "2" for e in end] if n == len(steps) - 1 else end
            lines.append(json.dumps({"step": n, "entries": entries, "end": ends}))
            rows.append(w)
        p = subprocess.run([sys.executable, os.path.join(REPO, "bin", "trace_run"), "--model", str(tmp_path), "--dtype", dtype,
                            "--out", str(out), "--max-tokens", "64"], input="\n".join(lines) + "\n", capture_output=True,
                           text=True, timeout=100)
        assert p.returncode == 0, p.stderr[-2000:]
        assert [x for x in p.stdout.splitlines() if x.startswith("done")] == [f"done {n}" for n in range(len(steps))]
        for n, w in enumerate(rows):
            f = out / f"{n}.f32"
            assert f.exists() == bool(w)
            if w:
                close(np.fromfile(f, "<f4").reshape(len(w), -1).astype(np.float64), np.stack(w), dtype)


def test_command_line(tmp_path):
    from pgmi import registry
    cfg = C.MIXED["a"]
    save(cfg, O.random_weights(cfg, 11), tmp_path)
    prompts = [tokens(cfg, 6, 95), tokens(cfg, 14, 96)]
    want = registry.load_decoder(str(tmp_path)).generate(prompts, 7).cpu().tolist()
    cmd = [sys.executable, "-m", "pgmi", "--model", str(tmp_path), "--max-new-tokens", "7"]
    for p in prompts:
        cmd += ["--prompt", ",".join(map(str, p))]
    out = subprocess.run(cmd, capture_output=True, text=True, timeout=100,
                         cwd=os.path.join(REPO, "multimodal-financial-analysis-tool-using-paligemma_amd"))
    assert out.returncode == 0, out.stderr[-2000:]
    assert [[int(t) for t in x.split(",")] for x in out.stdout.split()] == want


def test_refusals():
    cfg = C.MECHANISMS["gru"]
    eng, _ = build(cfg, "bfloat16", max_batch=2)
    cache = eng.new_cache(3, 16)
    a, b, c = (cache.alloc() for _ in range(3))
    with pytest.raises(MemoryError):
        cache.alloc()
    with pytest.raises(ValueError):
        eng.step(cache, [a], [[cfg["vocab"]]])
    with pytest.raises(ValueError):
        eng.step(cache, [a], [[1] * 17])
    with pytest.raises(ValueError):
        eng.step(cache, [a, a], [[1], [2, 3]])
    with pytest.raises(ValueError):
        eng.step(cache, [a, b, c], [[1], [2], [3, 4]])
    with pytest.raises(ValueError):
        eng.step(cache, [a], [[]])
    eng.step(cache, [a], [[1] * 16])
    with pytest.raises(ValueError):
        eng.step(cache, [a], [[1]])
    assert cache.length[a] == 16
