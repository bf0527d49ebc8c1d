// tile_f32.h -- output tiles of A [rows][K] fp32 . W [N][K]^T bf16 on the bf16 matrix units, at fp32 precision.
//
// A value a is cut, not rounded, into three bf16 pieces: its top 8 significant bits, the next 8, the last 8.  Each piece
// and each difference is exact, the pieces' products with a bf16 weight are exact in the matrix unit, and only their fp32
// sums round: K / 32 accumulations of each piece where an FMA chain has K roundings.  (Pieces below 2^-133, of values
// below 2^-117, are lost.)  A value or weight that is infinite or not a number makes inf - inf or 0 inf of the pieces, and
// so a result that is not finite: the workgroup forms a tile with such outputs again as FMA chains, and there their answer stands
// (500 rows of NaN, 1024 x 4096 and 4096 x 1024: 0.17 ms each; a lane per chain 3.8, FMA tiles 0.44 and 0.105).
//
// What bounds it: a tile is a chain of K / 64 steps (read, cut, write to LDS, multiply); a step's LDS traffic and its cuts
// (5.5 vector operations a value) each take about as long as its products, so two steps of global loads are kept in flight
// in registers while a third is multiplied, and the compiler runs the cuts between the products.  500 rows, 1024 x 4096 and
// 4096 x 1024: 21 us each (200 TFLOP/s of 833: three products a value on 2.5 PFLOP/s), FMA tiles of 64 x 64 436 and 111 us;
// error against 64 bits 2.4e-7 and 3.4e-7, FMA chains 1.2e-6 and 5.7e-7.  Weights straight from memory into registers
// (an LDS pass less) were no faster.
#pragma once
#include "common.h"

namespace pgmi {

// 16 bytes of an operand that may be aligned as single values only (a caller's own view): one load all the same
template <typename V>
__device__ __forceinline__ V any16(const void* p) {
    V v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// the three pieces of 8 values, as fragments' 16 bytes
struct F32Pieces { uint4 p[3]; };
__device__ __forceinline__ uint32_t top_halves(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }
__device__ __forceinline__ F32Pieces cut8(const float4 a, const float4 b) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t q[3][8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        q[0][i] = __float_as_uint(v[i]);
        const float r = v[i] - __uint_as_float(q[0][i] & 0xFFFF0000u);
        q[1][i] = __float_as_uint(r);
        q[2][i] = __float_as_uint(r - __uint_as_float(q[1][i] & 0xFFFF0000u));
    }
    F32Pieces o;
#pragma unroll
    for (int s = 0; s < 3; ++s)
        o.p[s] = make_uint4(top_halves(q[s][0], q[s][1]), top_halves(q[s][2], q[s][3]), top_halves(q[s][4], q[s][5]),
                            top_halves(q[s][6], q[s][7]));
    return o;
}
__device__ __forceinline__ bool not_finite(float v) { return (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u; }

constexpr size_t tile_f32_lds(int BM, int BN, int NB) { return (size_t)2 * (3 * BM + NB * BN) * 128; }

// One tile: rows [0, BM) of the caller's (source(m): the A row of tile row m, always a readable one), columns n0 .. n0 + BN
// of W and, with NB = 2, the same columns `up` elements further on; k in [k0, k1), both multiples of 8.  WM x WN waves of
// TM x TN 16 x 16 blocks.  put(m, n, v, v_up, bias(n)) gets every element of the tile with n < ncol; columns past N hold the last
// column's values.  A row past the caller's own is dropped by put.
template <int WM, int WN, int TM, int TN, int NB, typename Source, typename Bias, typename Put>
__device__ __forceinline__ void tile_f32(const float* __restrict__ A, int lda, const uint16_t* __restrict__ W, int ldw, long up,
                                         int N, int ncol, int n0, int k0, int k1, const Source& source, const Bias& bias, const Put& put) {
    constexpr int NT = 64 * WM * WN, BM = 16 * WM * TM, BN = 16 * WN * TN;
    constexpr int CA = BM * 8 / NT, CW = NB * BN * 8 / NT;  // 8-element chunks that a thread moves per step
    static_assert(CA * NT == BM * 8 && CW * NT == NB * BN * 8, "whole chunks");
    constexpr int PL = BM * 128, WAT = 3 * PL, BUF = WAT + NB * BN * 128;  // bytes: a piece's plane, the weights, a buffer
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_f32[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, c8 = tid & 7;
    const float* ap[CA];
    const uint16_t* wp[CW];
#pragma unroll
    for (int i = 0; i < CA; ++i) ap[i] = A + (long)source((tid + NT * i) >> 3) * lda;
#pragma unroll
    for (int i = 0; i < CW; ++i) {
        const int r = (tid + NT * i) >> 3;
        wp[i] = W + (NB == 2 ? (r / BN) * up : 0L) + (long)min(n0 + r % BN, N - 1) * ldw;
    }
    // ahead of the steps: asked for where it is added, each output waits for its own load, and for the store of the one before
    // (500 rows, 3,072 and 1,536 outputs of K = 1,024: 21.9 and 16.0 us, so 20.7 and 15.1)
    float bv[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bv[j] = bias(n0 + (wn * TN + j) * 16 + (lane & 15));
    struct Step { float4 a[CA][2]; uint4 w[CW]; };
    auto load = [&](int t, Step& s) {  // a chunk at or past k1 is read at k0 instead, and its weights are zero
        const int k = k0 + t * 64 + c8 * 8, kk = k < k1 ? k : k0;
#pragma unroll
        for (int i = 0; i < CA; ++i) {
            s.a[i][0] = any16<float4>(ap[i] + kk);
            s.a[i][1] = any16<float4>(ap[i] + kk + 4);
        }
#pragma unroll
        for (int i = 0; i < CW; ++i) s.w[i] = any16<uint4>(wp[i] + kk);
    };
    // 128-byte rows of 8 chunks, chunk c of row r at place c ^ (r & 7): the fragment reads of 16 rows spread over all banks
    auto write = [&](int t, const Step& s) {
        uint8_t* buf = smem_f32 + (t & 1) * BUF;
        const bool ok = k0 + t * 64 + c8 * 8 < k1;
#pragma unroll
        for (int i = 0; i < CA; ++i) {
            const int r = (tid + NT * i) >> 3, at = r * 128 + ((c8 ^ (r & 7)) << 4);
            const F32Pieces q = cut8(s.a[i][0], s.a[i][1]);
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<uint4*>(buf + p * PL + at) = q.p[p];
        }
#pragma unroll
        for (int i = 0; i < CW; ++i) {
            const int r = (tid + NT * i) >> 3;
            *reinterpret_cast<uint4*>(buf + WAT + r * 128 + ((c8 ^ (r & 7)) << 4)) = ok ? s.w[i] : make_uint4(0, 0, 0, 0);
        }
    };
    f32x4 acc[NB][TM][TN];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int li = lane & 15, lg = lane >> 4;
    auto multiply = [&](int t) {
        const uint8_t* buf = smem_f32 + (t & 1) * BUF;
        short8 a[2][3][TM], b[2][NB][TN];
        auto read = [&](int kk) {
            const int ch = ((kk * 4 + lg) ^ (li & 7)) << 4;
#pragma unroll
            for (int d = 0; d < NB; ++d)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    b[kk][d][j] = *reinterpret_cast<const short8*>(buf + WAT + (d * BN + (wn * TN + j) * 16 + li) * 128 + ch);
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    a[kk][p][i] = *reinterpret_cast<const short8*>(buf + p * PL + ((wm * TM + i) * 16 + li) * 128 + ch);
        };
        read(0);
        read(1);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int d = 0; d < NB; ++d)
#pragma unroll
                        for (int j = 0; j < TN; ++j) acc[d][i][j] = mfma16(a[kk][p][i], b[kk][d][j], acc[d][i][j]);
    };
    const int nt = (k1 - k0 + 63) / 64;
    Step s0, s1;
    load(0, s0);
    load(1, s1);
    write(0, s0);
    __syncthreads();
    // step t: its buffer is complete; step t + 1 is in registers or on its way, step t + 2 is asked for.  Steps go in pairs
    // (an odd last one has a partner of zero weights: a loop without exits in its middle keeps the loads in their registers).
    // The matrix unit's accumulation cuts where it should round: every 1024 of k the sums move to sums of their own, which
    // keeps the drift of a long sum of equal signs below an FMA chain's error (measured, K = 16384: 6.5e-6 without)
    f32x4 sum[NB][TM][TN];
    auto gather = [&](bool first) {
#pragma unroll
        for (int d = 0; d < NB; ++d)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    sum[d][i][j] = first ? acc[d][i][j] : sum[d][i][j] + acc[d][i][j];
                    acc[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
    };
    gather(true);
    for (int t = 0; t < nt; t += 2) {
        load(t + 2, s0);
        __builtin_amdgcn_sched_barrier(0);  // asked for here, not where the registers are next written
        multiply(t);
        write(t + 1, s1);
        __syncthreads();
        load(t + 3, s1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(t + 1);
        write(t + 2, s0);
        __syncthreads();
        if ((t & 14) == 14) gather(false);
    }
    gather(false);
    // outputs that are not finite: the tile's FMA chains over [k0, k1), kFmaK of k at a time through LDS
    bool bad = false;
#pragma unroll
    for (int d = 0; d < NB; ++d)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) bad |= not_finite(sum[d][i][j][r]);
    int* flag = reinterpret_cast<int*>(smem_f32);  // (the steps' last barrier has passed)
    const bool wave_bad = __any(bad);
    if (lane == 0) flag[wave] = wave_bad;
    __syncthreads();
    int again = 0;
#pragma unroll
    for (int q = 0; q < WM * WN; ++q) again |= flag[q];
    if (again) {
        constexpr int kFmaK = 16, SA = BM + 4, SW = NB * BN + 4;
        static_assert((size_t)kFmaK * (SA + SW) * 4 <= tile_f32_lds(BM, BN, NB), "the chains' operands fit");
        float* fa = reinterpret_cast<float*>(smem_f32);  // [kFmaK][SA]
        float* fw = fa + kFmaK * SA;                     // [kFmaK][SW]
        f32x4 c[NB][TM][TN];
#pragma unroll
        for (int d = 0; d < NB; ++d)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) c[d][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
        for (int k = k0; k < k1; k += kFmaK) {
            const int nk = min(kFmaK, k1 - k);
            __syncthreads();
#pragma clang loop unroll(disable)
            for (int x = tid; x < (BM + NB * BN) * kFmaK; x += NT) {
                const int r = x / kFmaK, q = x % kFmaK, kk = k + min(q, nk - 1);
                if (r < BM) fa[q * SA + r] = A[(long)source(r) * lda + kk];
                else fw[q * SW + r - BM] = bf2f(W[(NB == 2 ? ((r - BM) / BN) * up : 0L) + (long)min(n0 + (r - BM) % BN, N - 1) * ldw + kk]);
            }
            __syncthreads();
#pragma unroll 4
            for (int q = 0; q < nk; ++q)
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const f32x4 av = *reinterpret_cast<const f32x4*>(fa + q * SA + (wm * TM + i) * 16 + lg * 4);
#pragma unroll
                    for (int d = 0; d < NB; ++d)
#pragma unroll
                        for (int j = 0; j < TN; ++j) {
                            const float wv = fw[q * SW + d * BN + (wn * TN + j) * 16 + li];
#pragma unroll
                            for (int r = 0; r < 4; ++r) c[d][i][j][r] = fmaf(av[r], wv, c[d][i][j][r]);
                        }
                }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (not_finite(sum[0][i][j][r]) || not_finite(sum[NB - 1][i][j][r]))
#pragma unroll
                        for (int d = 0; d < NB; ++d) sum[d][i][j][r] = c[d][i][j][r];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (wn * TN + j) * 16 + li;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n < ncol) put((wm * TM + i) * 16 + lg * 4 + r, n, sum[0][i][j][r], sum[NB - 1][i][j][r], bv[j]);
        }
}

}  // namespace pgmi
