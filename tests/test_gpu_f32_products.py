"""fp32 products on the bf16 matrix units (csrc/tile_f32.h): every form of them against float64 at the edges of its tiles,
K slices and rows, and values that the exact split does not carry."""
import ctypes

import numpy as np
import pytest
import torch

import decoder_cases as C
import raritar_cases as R
from decoder_helpers import build, close, tokens
from oracle import decoder_np, raritar_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    return build(R.MECHANISMS["taps_1"], "float32")[0]


def product(eng, A, W, N, mode, out, split=True):
    from pgmi import _native as N_
    M, K = A.shape
    sp, scratch = ctypes.c_int(), torch.empty((M, 2 * N), device="cuda")
    N_.check(eng.lib.pgmi_op_matmul(eng.ctx, A.data_ptr(), A.stride(0), W.data_ptr(), W.stride(0), M, N, K,
                                    2 if A.dtype is torch.float32 else 0, mode, None, out.data_ptr(), out.shape[-1],
                                    out.numel() * 4, scratch.data_ptr(), ctypes.byref(sp) if split else None,
                                    N_.stream_handle(eng.device)))
    return sp.value


# 32 x 64 and 64 x 128 tiles, odd numbers of 64-deep steps, K past where the sums move (1024), one slice and eight
@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (17, 64, 64), (32, 65, 72), (33, 63, 200), (64, 130, 1032), (65, 4099, 136),
                                   (513, 4096, 128), (500, 1024, 4160), (200, 8200, 1096)])
def test_every_mode_against_float64(eng, M, N, K):
    g = torch.Generator("cuda").manual_seed(M + N + K)
    A = torch.randn((M, K + 8), device="cuda", generator=g)[:, :K]
    W = torch.randn((2 * N, K), device="cuda", generator=g).bfloat16()
    ref = A.double() @ W.double().t()
    # a K-term fp32 sum: (K / 32 accumulations of 3 pieces + 8 slices) roundings of partial sums of at most sum |a w|
    bound = (A.double().abs() @ W.double().abs().t()) * 2.0 ** -24 * (3 * min(K, 1024) / 32 + K / 1024 + 10)
    out = torch.full((M, N), float("nan"), device="cuda")
    product(eng, A, W, N, 1, out)
    assert ((out.double() - ref[:, :N]).abs() <= bound[:, :N]).all()
    slabs = torch.full((8, M, N), float("nan"), device="cuda")
    sp = product(eng, A, W, N, 2, slabs)
    assert 1 <= sp <= 8 and ((slabs[:sp].double().sum(0) - ref[:, :N]).abs() <= bound[:, :N]).all()
    ldo = (N + 7) // 8 * 8
    out = torch.full((M, ldo), float("nan"), device="cuda")
    product(eng, A, W, N, 3, out)
    want = torch.nn.functional.silu(ref[:, :N]) * ref[:, N:]
    # |d silu| <= 1.1 |d gate|; silu itself to a few ulp
    tol = 1.1 * bound[:, :N] * (ref[:, N:].abs() + bound[:, N:]) + ref[:, :N].abs() * bound[:, N:] + 1e-6 * want.abs() + 1e-30
    assert ((out[:, :N].double() - want).abs() <= tol).all() and (out[:, N:] == 0).all()


@pytest.mark.parametrize("M,N,K", [(33, 65, 200), (300, 4096, 136)])
def test_operands_aligned_as_single_values(eng, M, N, K):
    """Rows that begin 4 bytes, weights that begin 2 bytes past a 16-byte boundary."""
    g = torch.Generator("cuda").manual_seed(M)
    A = torch.randn(M * (K + 8) + 1, device="cuda", generator=g)[1:].view(M, K + 8)[:, :K]
    W = torch.randn(N * K + 1, device="cuda", generator=g).bfloat16()[1:].view(N, K)
    assert A.data_ptr() % 16 == 4 and W.data_ptr() % 16 == 2
    out, same = torch.empty((M, N), device="cuda"), torch.empty((M, N), device="cuda")
    product(eng, A, W, N, 1, out)
    product(eng, A.clone(memory_format=torch.contiguous_format), W.clone(), N, 1, same)
    assert torch.equal(out, same)


def test_gate_and_up_without_scratch(eng):
    """Refused for fp32 rows, as include/pgmi.h has it."""
    from pgmi import _native as N_
    A, W, out = torch.ones((4, 8), device="cuda"), torch.ones((16, 8), device="cuda").bfloat16(), torch.zeros((4, 8), device="cuda")
    status = eng.lib.pgmi_op_matmul(eng.ctx, A.data_ptr(), 8, W.data_ptr(), 8, 4, 8, 8, 2, 3, None, out.data_ptr(), 8, 128, None, None,
                                    N_.stream_handle(eng.device))
    assert status != 0 and not out.any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_slabs_for_a_caller_that_asks_for_no_split(eng, dtype):
    """One slab, the whole product, though the output has room for more."""
    g = torch.Generator("cuda").manual_seed(5)
    A = torch.randn((40, 4096), device="cuda", generator=g).to(dtype)
    W = torch.randn((64, 4096), device="cuda", generator=g).bfloat16()
    out = torch.zeros((8, 40, 64), device="cuda")
    assert product(eng, A, W, 64, 2, out) > 1
    out.zero_()
    product(eng, A, W, 64, 2, out, split=False)
    ref = A.double() @ W.double().t()
    assert (out[0].double() - ref).norm() <= 1e-5 * ref.norm() and not out[1:].any()


@pytest.mark.parametrize("M,N", [(20, 70), (300, 4096)])
def test_values_that_are_not_finite_and_the_largest(eng, M, N):
    """Infinities, not-a-numbers (payload in the low bits only, too) and the largest finite values, in rows and weights, give
    what the FMA chain gives, and leave the other outputs alone."""
    K = 200
    g = torch.Generator("cuda").manual_seed(M)
    A = torch.randn((M, K), device="cuda", generator=g)
    W = torch.randn((N, K), device="cuda", generator=g).bfloat16()
    W[:, 7] = W[:, 7].abs() + 0.5
    W[:, :2] = torch.tensor([0.0, 1.0], device="cuda").bfloat16()
    clean = A.double() @ W.double().t()
    A[1, 7], A[2, 7], A[4, 100] = float("inf"), float("-inf"), float("nan")
    A[5].view(torch.int32)[9] = 0x7F800001
    A[6, 7] = 3.4028234663852886e38  # times 0.5 or more: finite or inf, by the weight
    A[7, 0] = float("inf")  # meets a weight of zero
    A[8] = 0.0
    A[9] = 1.0000001
    W[3, 11] = float("inf")
    out = torch.empty((M, N), device="cuda")
    product(eng, A, W, N, 1, out)
    a, w = A.cpu(), W.float().cpu()
    chain = torch.zeros((M, N))
    for k in range(K):
        chain = chain + a[:, k, None] * w[None, :, k]
    got = out.cpu()
    there = torch.ones(M, dtype=torch.bool)
    there[6] = False  # at the edge of overflow a fused step and this one may part
    assert torch.equal(torch.isnan(got), torch.isnan(chain))
    assert torch.equal(got[there][chain[there].isinf()], chain[there][chain[there].isinf()])
    fin = torch.isfinite(chain)
    assert ((got - chain).abs()[fin] <= 1e-5 * chain.abs()[fin] + 1e-3).all()
    ordinary = torch.ones((M, N), dtype=torch.bool)
    ordinary[1:10], ordinary[:, 3] = False, False
    assert ((got - clean.cpu()).abs()[ordinary] < 1e-4).all()


def milliseconds(fn, n=4):
    """The fastest of n calls."""
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(n + 1)]
    fn()
    for e in ev[:-1]:
        e.record()
        fn()
    ev[-1].record()
    torch.cuda.synchronize()
    return min(a.elapsed_time(b) for a, b in zip(ev, ev[1:]))


@pytest.mark.parametrize("M,N,K", [(500, 1024, 4096), (500, 4096, 1024), (17, 64, 4096)])
def test_time_where_nothing_is_finite(eng, M, N, K):
    """Chains formed by whole workgroups: 5 to 8 times the finite product's time measured; a lane per chain took 110 to 170 times."""
    A, W, out = torch.randn((M, K), device="cuda"), torch.randn((N, K), device="cuda").bfloat16(), torch.empty((M, N), device="cuda")
    finite = milliseconds(lambda: product(eng, A, W, N, 1, out))
    A.fill_(float("nan"))
    assert milliseconds(lambda: product(eng, A, W, N, 1, out)) <= 25 * finite
    assert out.isnan().all()


# fp32: the output matrix of a step of four rows; bf16: its form that walks several groups of outputs, one input short of whole
@pytest.mark.parametrize("dtype,width,vocab", [("float32", 8192, 512), ("bfloat16", 2040, 9001)])
def test_time_and_values_of_a_step_where_a_weight_is_not_finite(dtype, width, vocab):
    """Only its own output is lost, and the step is not held up by it (0.33 ms for 0.074, and 0.046 for 0.046; a lane per output
    0.59 and 0.18)."""
    cfg = C.model([C.gru(512)], width=width, vocab=vocab, streams=1, groups=1)
    times, logits = [], []
    for bad in (False, True):
        W = decoder_np.random_weights(cfg, 3)
        if bad:
            W["embed"][5, 0], W["embed"][5, 3], W["embed"][6, width - 1], W["embed"][7, 0] = np.inf, -np.inf, np.nan, np.inf
        eng, _ = build(cfg, dtype, weights=W, max_batch=4)
        cache = eng.new_cache(4, 64)
        slots, ids = [cache.alloc() for _ in range(4)], torch.arange(10, 14, device="cuda")
        logits.append(eng.decode(cache, slots, ids).clone())
        times.append(milliseconds(lambda: eng.decode(cache, slots, ids), 12))
    fine, broken = logits
    keep = torch.ones(vocab, dtype=torch.bool)
    keep[5:8] = False
    assert torch.equal(fine[:, keep], broken[:, keep])
    assert not broken[:, 5].isfinite().any() and broken[:, 6].isnan().all() and broken[:, 7].isinf().all()
    assert times[1] <= (6 if dtype == "float32" else 2) * times[0], times


@pytest.mark.parametrize("B", [3, 16])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_row_that_is_not_finite(dtype, B):
    """One sequence's activations, through products whose K is cut over workgroups too: the others are the same to the bit."""
    cfg = C.model([C.gru(512, ff=8192), C.mamba(1032, 16, 8, 4)], width=264, vocab=300, streams=2, groups=1)
    W = decoder_np.random_weights(cfg, 3)
    W["embed"][5], W["embed"][6] = np.inf, np.nan
    eng, _ = build(cfg, dtype, weights=W, max_batch=16)
    logits = []
    for bad in (None, 5, 6):
        cache, ids = eng.new_cache(B, 4), torch.arange(10, 10 + B, device="cuda")
        if bad is not None:
            ids[1] = bad
        logits.append(eng.decode(cache, [cache.alloc() for _ in range(B)], ids).clone())
    others = torch.arange(B, device="cuda") != 1
    columns = torch.ones(300, dtype=torch.bool, device="cuda")
    columns[5:7] = False  # (the table is the output matrix too)
    fine = logits[0][others][:, columns]
    assert fine.isfinite().all()
    for broken in logits[1:]:
        assert torch.equal(broken[others][:, columns], fine) and not broken[1].isfinite().any()


@pytest.mark.parametrize("part", ["gate", "up", "down"])
@pytest.mark.parametrize("rows", [40, 300])  # both sizes of tile
def test_an_expert_whose_weight_is_not_finite(rows, part):
    """Lost are the rows that chose it (those that another value of the weight changes); the others are the same to the bit."""
    cfg = R.MECHANISMS["experts_few"]
    name, toks, logits = f"l0.mlp.e1.{part}", tokens(cfg, rows, 8), []
    for value in (None, 50.0, np.inf):
        W = raritar_np.random_weights(cfg, 3)
        if value is not None:
            W[name][3, 2] = value
        eng, _ = build(cfg, "float32", weights=W)
        cache = eng.new_cache(1, rows)
        logits.append(eng.step(cache, [cache.alloc()], [toks], want=list(range(rows))).clone())
    fine, other, broken = logits
    chose = (fine != other).any(1)
    assert 0 < int(chose.sum()) < rows
    assert torch.equal(~broken.isfinite().all(1), chose) and torch.equal(broken[~chose], fine[~chose])


@pytest.mark.parametrize("rows", [3, 16, 17, 40])
def test_decode_rows(rows):
    """One token each: the skinny form (to 16 rows) and the tiles, mixtures of experts included."""
    cfg = R.MIXED["b"]
    eng, W = build(cfg, "float32", max_batch=64)
    seqs = [tokens(cfg, 4, 60 + r) for r in range(rows)]
    want = [raritar_np.run(cfg, W, s) for s in seqs[:6]]
    cache = eng.new_cache(rows, 16)
    slots = [cache.alloc() for _ in seqs]
    for t in range(4):
        lg = eng.step(cache, slots, [[s[t]] for s in seqs])
        close(lg[:6], np.stack([w[t] for w in want]), "float32")


@pytest.mark.parametrize("B", [3, 16])
@pytest.mark.parametrize("K", [2048, 8192, 16384])
def test_long_sums_of_few_rows(K, B):
    """The output matrix over K positive terms, where sums drift the most: no further from float64 than a chain of fused
    multiply-adds, which rounds K times."""
    cfg = C.model([C.gru(8)], width=K, vocab=64, streams=1, groups=1, escale=1.0)
    W = decoder_np.random_weights(cfg, 3)
    E = np.random.default_rng(K).random((64, K), dtype=np.float32) * np.float32(0.9) + np.float32(0.1)
    W["embed"] = (E.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    for n in W:
        if n.startswith("l0.hc") or "norm" in n:
            W[n] = np.ones_like(W[n])
    W["l0.mix.o"] = np.zeros_like(W["l0.mix.o"])  # the residual stays the token's embedding
    eng, _ = build(cfg, "float32", weights=W, max_batch=16)
    cache = eng.new_cache(B, 4)
    got = eng.decode(cache, [cache.alloc() for _ in range(B)], torch.arange(B, device="cuda")).double().cpu().numpy()
    E = W["embed"].astype(np.float64)
    h = E[:B] / np.sqrt((E[:B] ** 2).mean(-1, keepdims=True) + cfg["norm"]["eps"])
    want, chain = h @ E.T, np.zeros((B, 64), np.float32)
    h = h.astype(np.float32).astype(np.float64)
    for k in range(K):
        chain = (chain + h[:, k, None] * E[None, :, k]).astype(np.float32)
    err = lambda x: np.sqrt(((x - want) ** 2).mean())
    assert err(got) <= err(chain.astype(np.float64)), (err(got) / want.mean(), err(chain) / want.mean())
