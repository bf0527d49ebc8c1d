// kernels_scan.hip -- the recurrent mechanisms of the layered decoders, over packed rows of unequal sequences:
// the causal convolution and selective scan of Mamba, and the minimal gated recurrence (minGRU).
//
// A sequence's rows are cut into chunks.  With one chunk a workgroup walks it from the sequence's state.  With
// several, three launches run them in parallel: (A) every chunk but the last from a zero state (its end
// state and its total decay), (B) one short walk over the chunks that turns these into the chunks' entry states,
// (C) every chunk again from its entry state, writing the outputs; the last chunk leaves the sequence's state.
// The decay of a chunk is exp(A sum(dt)), so (A) keeps sums of steps and no products.
// A scan of 9 to 16 states walks its sequences whole instead, a lane per state, where that is predicted to be faster (scan_walks).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "act.h"
#include "decoder.h"
#include "runs.h"

namespace pgmi {

namespace {

// ---------------------------------------------------------------- causal convolution + silu
// the input at the sequence's relative row p < 0: the taps kept from earlier steps (zero at the start)
template <typename T>
__device__ __forceinline__ float tap_at(const SeqInfo& q, const float* taps, int K, int C, int p, int c) {
    const int j = K - 1 + p;
    return (q.start > 0 && j >= 0) ? taps[((long)q.slot * (K - 1) + j) * C + c] : 0.0f;
}

// V == 8: eight channels per lane, KT taps held in registers, each wave a run of consecutive rows.
// KT == 0: any number of taps, one channel per lane.
// keep: the wave that ends a sequence leaves its window as the sequence's taps (every sequence from its start: no wave reads
// earlier ones).  A launch of its own for them is 4.2 to 4.8 us of a layer: 500 rows of 2,048 fp32 channels 5.4 + 4.2 -> 5.4,
// 1,540 rows of 4,096 bf16 8.9 + 4.7 -> 9.1.
template <typename T, int KT>
__global__ void __launch_bounds__(256) k_conv_silu(const T* __restrict__ xz, int ldxz, int C, int K,
                                                   const uint16_t* __restrict__ w, const uint16_t* __restrict__ b,
                                                   const SeqInfo* __restrict__ seqs, const ChunkInfo* __restrict__ chunks,
                                                   const float* __restrict__ taps, float* __restrict__ keep,
                                                   T* __restrict__ out, int ldo) {
    const ChunkInfo ck = chunks[blockIdx.y];
    const SeqInfo q = seqs[ck.seq];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int run = (ck.len + 3) / 4, r0 = wave * run, r1 = min(ck.len, r0 + run);
    if constexpr (KT > 0) {
        const int c = (blockIdx.x * 64 + lane) * 8;
        if (c >= C || r0 >= r1) return;
        float wk[KT][8], bias[8], win[KT][8];
        {
            float f[KT * 8];
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                float g[8];
                ld8(w + (long)c * KT + 8 * t, g);
#pragma unroll
                for (int v = 0; v < 8; ++v) f[8 * t + v] = g[v];
            }
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int v = 0; v < 8; ++v) wk[t][v] = f[v * KT + t];
        }
        ld8(b + c, bias);
#pragma unroll
        for (int t = 0; t < KT - 1; ++t) {  // the KT - 1 inputs before the run
            const int p = ck.rel + r0 - (KT - 1) + t;
            if (p >= 0) {
                ld8(xz + (long)(q.off + p) * ldxz + c, win[t]);
            } else {
#pragma unroll
                for (int v = 0; v < 8; ++v) win[t][v] = tap_at<T>(q, taps, KT, C, p, c + v);
            }
        }
#pragma unroll 4
        for (int r = r0; r < r1; ++r) {
            ld8(xz + (long)(ck.row + r) * ldxz + c, win[KT - 1]);
            float y[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                y[v] = bias[v];
#pragma unroll
                for (int t = 0; t < KT; ++t) y[v] = fmaf(wk[t][v], win[t][v], y[v]);
                y[v] = siluf_(y[v]);
#pragma unroll
                for (int t = 0; t + 1 < KT; ++t) win[t][v] = win[t + 1][v];
            }
            st8(out + (long)(ck.row + r) * ldo + c, y);
        }
        if (keep && ck.rel + r1 == q.len) {
#pragma unroll
            for (int t = 0; t < KT - 1; ++t)
#pragma unroll
                for (int v = 0; v < 8; ++v) keep[((long)q.slot * (KT - 1) + t) * C + c + v] = win[t][v];
        }
    } else {
        const int c = blockIdx.x * 64 + lane;
        if (c >= ldo) return;
        for (int r = r0; r < r1; ++r) {
            float y = 0.0f;
            if (c < C) {
                y = bf2f(b[c]);
                for (int k = 0; k < K; ++k) {
                    const int p = ck.rel + r - (K - 1) + k;
                    const float x = p >= 0 ? ldf(xz + (long)(q.off + p) * ldxz + c) : tap_at<T>(q, taps, K, C, p, c);
                    y = fmaf(bf2f(w[(long)c * K + k]), x, y);
                }
                y = siluf_(y);
            }
            stf(out + (long)(ck.row + r) * ldo + c, y);
        }
    }
}

// the last K - 1 inputs of each sequence become its taps (one thread per channel, ascending j: new tap j is
// an older tap at j + len, not yet overwritten, or a row of this step)
template <typename T>
__global__ void __launch_bounds__(256) k_conv_taps(const T* __restrict__ xz, int ldxz, int C, int K,
                                                   const SeqInfo* __restrict__ seqs, float* __restrict__ taps) {
    const SeqInfo q = seqs[blockIdx.y];
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    for (int j = 0; j < K - 1; ++j) {
        const int p = q.len - (K - 1) + j;
        const float v = p >= 0 ? ldf(xz + (long)(q.off + p) * ldxz + c) : tap_at<T>(q, taps, K, C, p, c);
        taps[((long)q.slot * (K - 1) + j) * C + c] = v;
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_scan_inputs(const float* __restrict__ slabs, int split, int rows, int R, int N,
                                                     T* __restrict__ dtl, int ldd, float* __restrict__ bc) {
    const int M = R + 2 * N;
    const int row = blockIdx.x;
    for (int i = threadIdx.x; i < M; i += 256) {
        float v = 0.0f;
        for (int z = 0; z < split; ++z) v += slabs[((long)z * rows + row) * M + i];
        if (i < R) stf(dtl + (long)row * ldd + i, v);
        else bc[(long)row * 2 * N + i - R] = v;
    }
    for (int i = R + threadIdx.x; i < ldd; i += 256) stf(dtl + (long)row * ldd + i, 0.0f);
}

// ---------------------------------------------------------------- selective scan
constexpr int kSub = 32;  // rows whose B | C are staged in LDS at a time
constexpr int kPre = 8;   // rows whose step, input and gate are in flight ahead of the recurrence

// LPC lanes per channel, NPL states per lane (N <= LPC * NPL; states past N are inert: B = C = 0).
// PHASE 0: (A) zero entry state, no output; 1: (C) / single-chunk walk.
template <typename T, int NPL, int LPC, int PHASE>
__global__ void __launch_bounds__(256, LPC == 1 ? 2 : LPC == 4 || LPC == 8 ? 3 : 1) k_scan(ScanArgs a) {
    constexpr int CPB = 256 / LPC;  // channels per workgroup
    constexpr int NP = NPL * LPC;
    constexpr bool AHEAD = LPC == 1;  // the next row's B | C read under this one's sums (they cost lanes that share a channel a wave)
    __shared__ __attribute__((aligned(16))) float sB[kSub][NP], sC[PHASE ? kSub : 1][PHASE ? NP : 4];
    const ChunkInfo ck = a.chunks[blockIdx.y];
    const bool last = ck.idx + 1 == ck.nch;
    if (PHASE == 0 && last) return;  // only earlier chunks feed others
    const SeqInfo q = a.seqs[ck.seq];
    const int tid = threadIdx.x, sub = tid % LPC;
    const int c = blockIdx.x * CPB + tid / LPC;
    const bool ok = c < a.C;
    const int cc = ok ? c : a.C - 1;
    const int n0 = sub * NPL;
    const int N = a.N;
    float A[NPL], S[NPL];
    const long sbase = ((long)q.slot * a.C + cc) * N, cbase = ((long)blockIdx.y * a.C + cc) * N;
    // every load of the start before the first wait, wide where the states fill the lanes: one after the other, each behind its
    // own bounds check, they were 6 us of every workgroup ((A) of 500 rows of 2,048 channels 18.3 us, now 12.4; (A) and (C) of
    // 1,540 rows of 4,096 channels 85 / 70)
    const float* from = ck.nch > 1 ? a.cstate + cbase : a.state + sbase;
    const bool entry = PHASE == 1 && (ck.nch > 1 || q.start > 0);
    const bool whole = N == NP && ((reinterpret_cast<uintptr_t>(a.A_log) | reinterpret_cast<uintptr_t>(a.cstate) |
                                    reinterpret_cast<uintptr_t>(a.state)) & 15) == 0;
    uint16_t al[NPL];
    if (whole) {
#pragma unroll
        for (int i = 0; i < NPL; i += 8) {
            const short8 v = __builtin_bit_cast(short8, *reinterpret_cast<const uint4*>(a.A_log + (long)cc * N + n0 + i));
#pragma unroll
            for (int e = 0; e < 8; ++e) al[i + e] = (uint16_t)v[e];
        }
        if constexpr (PHASE == 1)
#pragma unroll
            for (int i = 0; i < NPL; i += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(from + n0 + i);
#pragma unroll
                for (int e = 0; e < 4; ++e) S[i + e] = v[e];
            }
    } else {
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            const int n = min(n0 + i, N - 1);
            al[i] = a.A_log[(long)cc * N + n];
            if constexpr (PHASE == 1) S[i] = from[n];
        }
    }
    const float bias = bf2f(a.dtb[cc]), Dc = bf2f(a.Dw[cc]);
    const float* __restrict__ dp = a.dt + (long)ck.row * a.C + cc;
    const T* __restrict__ xp = reinterpret_cast<const T*>(a.x) + (long)ck.row * a.ldx + cc;
    const T* __restrict__ zp = reinterpret_cast<const T*>(a.z) + (long)ck.row * a.ldz + cc;
    T* __restrict__ yp = reinterpret_cast<T*>(a.y) + (long)ck.row * a.ldy + c;
    float dsum = 0.0f;
    float pd[kPre];
    T px[kPre], pz[kPre];
    // B | C of the next kSub rows, where a thread holds few of them
    constexpr int IT = kSub * NP / 256;
    constexpr bool HELD = IT <= 4;
    float hb[HELD ? IT : 1], hc[HELD ? IT : 1];
    auto hold = [&](int t0) {
        if constexpr (HELD)
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                const int i = tid + 256 * k, n = min(i % NP, N - 1);
                const float* r = a.bc + (long)(ck.row + min(t0 + i / NP, ck.len - 1)) * 2 * N;
                hb[k] = r[n];
                if constexpr (PHASE == 1) hc[k] = r[N + n];
            }
    };
    auto fetch = [&](int t0) {  // rows past the chunk repeat its last one (never used)
#pragma unroll
        for (int t = 0; t < kPre; ++t) {
            const long r = min(t0 + t, ck.len - 1);
            pd[t] = dp[r * a.C];
            px[t] = xp[r * a.ldx];
            if constexpr (PHASE == 1) pz[t] = zp[r * a.ldz];
        }
    };
    hold(0);
    fetch(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        const int n = n0 + i;
        // dt A in powers of two: exp(dt A) = exp2(dt A log2 e)
        A[i] = n < N ? -expf(bf2f(al[i])) * 1.4426950408889634f : 0.0f;
        if (!entry || n >= N) S[i] = 0.0f;
    }
    // this lane's staged states, as whole vectors: indexed by single states the compiler read them in halves where lanes share a
    // channel ((C) of 1,540 rows of 2,048 channels of 256 states 709 us, so 410)
    const f32x4* lB = reinterpret_cast<const f32x4*>(&sB[0][0]) + sub * (NPL / 4);
    const f32x4* lC = reinterpret_cast<const f32x4*>(&sC[0][0]) + sub * (NPL / 4);
    for (int t0 = 0; t0 < ck.len; t0 += kSub) {
        const int nt = min(kSub, ck.len - t0);
        __syncthreads();
        if constexpr (HELD) {
#pragma unroll
            for (int k = 0; k < IT; ++k) {
                const int i = tid + 256 * k, t = i / NP, n = i % NP;
                sB[t][n] = n < N ? hb[k] : 0.0f;
                if constexpr (PHASE == 1) sC[t][n] = n < N ? hc[k] : 0.0f;
            }
        } else {
            for (int i = tid; i < nt * NP; i += 256) {
                const int t = i / NP, n = i % NP;
                const float* r = a.bc + (long)(ck.row + t0 + t) * 2 * N;
                sB[t][n] = n < N ? r[n] : 0.0f;
                if constexpr (PHASE == 1) sC[t][n] = n < N ? r[N + n] : 0.0f;
            }
        }
        __syncthreads();
        if (t0 + kSub < ck.len) hold(t0 + kSub);
        // kPre rows; all of them there: no branch between them, so that the next row's B | C are read under this one's sums.
        // (A) / (C), us, a branch and reads of its own before each row -> now: 1,540 rows of 4,096 channels of 16 states
        // 31.0 / 39.4 -> 28.6 / 35.9, 500 rows 15.3 / 19.6 -> 13.2 / 16.2, 2,048 channels of 64 states 54.5 / 76.5 -> 50.7 /
        // 68.4, of 256 203 / 439 -> 187 / 395.  The step's softplus in its product's epilogue instead: (A) 24, the product
        // 10.4 -> 18.3, which nothing there covers.
        auto walk = [&](auto full, int tb) {
            float dt[kPre], x[kPre], g[kPre];
#pragma unroll
            for (int t = 0; t < kPre; ++t) {
                dt[t] = softplus_of<T>(pd[t] + bias);
                x[t] = ldf(&px[t]);
                g[t] = 0.0f;
                if constexpr (PHASE == 1) g[t] = siluf_(ldf(&pz[t]));
            }
            if (t0 + tb + kPre < ck.len) fetch(t0 + tb + kPre);
            f32x4 B[1 + AHEAD][NPL / 4], Cv[1 + AHEAD][PHASE ? NPL / 4 : 1];
            auto read = [&](int t, int to) {
#pragma unroll
                for (int i = 0; i < NPL / 4; ++i) {
                    B[to][i] = lB[(tb + t) * (NP / 4) + i];
                    if constexpr (PHASE == 1) Cv[to][i] = lC[(tb + t) * (NP / 4) + i];
                }
            };
            if constexpr (AHEAD) read(0, 0);
#pragma unroll
            for (int t = 0; t < kPre; ++t) {
                if (!full && tb + t >= nt) break;
                const int at = AHEAD ? t & 1 : 0;
                if constexpr (AHEAD) {
                    if (t + 1 < kPre) read(t + 1, (t + 1) & 1);  // (of a broken block, rows of LDS that are not used)
                    __builtin_amdgcn_sched_barrier(0);
                } else {
                    read(t, 0);
                }
                const float dx = dt[t] * x[t];
                dsum += dt[t];
                float y0 = 0.0f, y1 = 0.0f;
#pragma unroll
                for (int i = 0; i < NPL; ++i)
                    S[i] = fmaf(__builtin_amdgcn_exp2f(dt[t] * A[i]), S[i], dx * B[at][i / 4][i % 4]);
                if constexpr (PHASE == 1) {
#pragma unroll
                    for (int i = 0; i < NPL; i += 2) {
                        y0 = fmaf(S[i], Cv[at][i / 4][i % 4], y0);
                        y1 = fmaf(S[i + 1], Cv[at][i / 4][i % 4 + 1], y1);
                    }
                    float y = y0 + y1;
                    y = lanes_join<LPC>(y, SumOp{});
                    g[t] *= fmaf(Dc, x[t], y);
                    asm volatile("" : "+v"(g[t]));  // (else the sum moves into the stores' branch, with every row's states)
                }
                if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (PHASE == 1) {
                if (sub == 0 && c < a.ldy) {  // columns C .. ldy - 1 are zero
#pragma unroll
                    for (int t = 0; t < kPre; ++t) {
                        if (!full && tb + t >= nt) break;
                        stf(yp + (long)(t0 + tb + t) * a.ldy, ok ? g[t] : 0.0f);
                    }
                }
            }
        };
        int tb = 0;
        for (; tb + kPre <= nt; tb += kPre) walk(std::true_type{}, tb);
        if (tb < nt) walk(std::false_type{}, tb);
    }
    if (!ok) return;
    if (PHASE == 0 && sub == 0) a.csum[(long)blockIdx.y * a.C + c] = dsum;
    if (PHASE == 1 && !last) return;
    float* to = (PHASE == 0 ? a.cstate + cbase : a.state + sbase) + n0;
    if (whole) {
#pragma unroll
        for (int i = 0; i < NPL; i += 4) *reinterpret_cast<f32x4*>(to + i) = f32x4{S[i], S[i + 1], S[i + 2], S[i + 3]};
    } else {
#pragma unroll
        for (int i = 0; i < NPL; ++i)
            if (n0 + i < N) to[i] = S[i];
    }
}

// (B) the chunks' entry states, in place of their end states
__global__ void __launch_bounds__(256) k_scan_carry(ScanArgs a) {
    const ChunkInfo ck = a.chunks[blockIdx.y];
    if (ck.idx != 0 || ck.nch < 2) return;  // one walk per sequence, from its first chunk
    const SeqInfo q = a.seqs[ck.seq];
    const long i = (long)blockIdx.x * 256 + threadIdx.x, CN = (long)a.C * a.N;
    if (i >= CN) return;
    const int c = (int)(i / a.N);
    const float A = -expf(bf2f(a.A_log[i])) * 1.4426950408889634f;
    float S = q.start > 0 ? a.state[(long)q.slot * CN + i] : 0.0f;
    float* e = a.cstate + (long)blockIdx.y * CN + i;
    const float* ds = a.csum + (long)blockIdx.y * a.C + c;
    const int n = ck.nch - 1;  // the last chunk left no end state
    for (int k0 = 0; k0 <= n; k0 += kPre) {
        float end[kPre], f[kPre];
#pragma unroll
        for (int k = 0; k < kPre; ++k) {
            const long r = min(k0 + k, n - 1);
            end[k] = e[r * CN];
            f[k] = ds[r * a.C];
        }
#pragma unroll
        for (int k = 0; k < kPre; ++k)
            if (k0 + k <= n) {
                e[(long)(k0 + k) * CN] = S;
                S = fmaf(__builtin_amdgcn_exp2f(A * f[k]), S, end[k]);
            }
    }
}

// ---- sequences walked whole, a lane per state
// Bound by the vector units: an instruction of 64 lanes takes a SIMD of 16 four clocks (measured 4.5 to 5.5, an exponential 8.4), so that
// walking waves which share a SIMD gain nothing: a step takes a CU's share of all rows, or its longest sequence's where that is
// longer.  It is one exponential, two products with a value of the channel (broadcast within the instruction, DPP), an FMA (fp32:
// two), a product with C and two additions of the sum over the states: 24 ns a row (fp32 35), 18 of them those instructions'.  So
// everything else is another four waves' work.  One wave for both: 36 ns; with its loads and stores straight from memory, 16 rows
// of 4 channels an instruction, 43.  us a layer: see scan_walks.
constexpr int kWalk = 16;  // channels of a workgroup, lanes of a channel, and rows of a block

// step t's value of a channel's 16 lanes
template <int t>
__device__ __forceinline__ float of_step(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + t, 0xF, 0xF, true));
}
template <typename F, int... t>
__device__ __forceinline__ void each_step(const F& f, std::integer_sequence<int, t...>) {
    (f(std::integral_constant<int, t>{}), ...);
}
// lane j of each 16 gets the sum of p[j] over the 16: halves and quarters exchanged by lanes that write only their own part (two
// additions where a choice and an addition would be three), then the four lanes of a quarter
__device__ __forceinline__ float sum_of_step(const float (&p)[kWalk], int lane) {
    float a[8], b[4];
#define HALF_(k, lo, hi) "v_add_f32_dpp %" #k ", %" #lo ", %" #lo " row_ror:8 row_mask:0xf bank_mask:0x3\n" \
                         "v_add_f32_dpp %" #k ", %" #hi ", %" #hi " row_ror:8 row_mask:0xf bank_mask:0xc\n"
#define QUARTER_(k, lo, hi) "v_add_f32_dpp %" #k ", %" #lo ", %" #lo " row_half_mirror row_mask:0xf bank_mask:0x5\n" \
                            "v_add_f32_dpp %" #k ", %" #hi ", %" #hi " row_half_mirror row_mask:0xf bank_mask:0xa\n"
    asm("s_nop 1\n" HALF_(0, 8, 16) HALF_(1, 9, 17) HALF_(2, 10, 18) HALF_(3, 11, 19) HALF_(4, 12, 20) HALF_(5, 13, 21)
        HALF_(6, 14, 22) HALF_(7, 15, 23)
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(a[4]), "=&v"(a[5]), "=&v"(a[6]), "=&v"(a[7])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]), "v"(p[8]), "v"(p[9]),
          "v"(p[10]), "v"(p[11]), "v"(p[12]), "v"(p[13]), "v"(p[14]), "v"(p[15]));
    asm("s_nop 1\n" QUARTER_(0, 4, 8) QUARTER_(1, 5, 9) QUARTER_(2, 6, 10) QUARTER_(3, 7, 11) "s_nop 1\n"
        : "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]));
#undef HALF_
#undef QUARTER_
    auto other = [](float v, auto ctrl) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    const bool o1 = lane & 1, o2 = lane & 2;
    using X1 = std::integral_constant<int, 0xB1>;  // quad_perm 1 0 3 2
    using X2 = std::integral_constant<int, 0x4E>;  // quad_perm 2 3 0 1
    const float c0 = (o1 ? b[1] : b[0]) + other(o1 ? b[0] : b[1], X1{}), c1 = (o1 ? b[3] : b[2]) + other(o1 ? b[2] : b[3], X1{});
    return (o2 ? c1 : c0) + other(o2 ? c0 : c1, X2{});
}

__device__ __forceinline__ float sum_of_lanes(float v) {  // of a channel's 16
    auto turned = [](float x, auto by) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + decltype(by)::value, 0xF, 0xF, true));
    };
    v += turned(v, std::integral_constant<int, 8>{});
    v += turned(v, std::integral_constant<int, 4>{});
    v += turned(v, std::integral_constant<int, 2>{});
    return v + turned(v, std::integral_constant<int, 1>{});
}

// Four waves walk 16 channels, four others have the rest: they fetch the rows (asked for 64 rows ahead of their use), form the
// steps and inputs of the next 64 rows while these are walked, and gate and store the 64 rows before.  V4: such a thread has four
// channels of one row, else one channel of four rows.  WHOLE: 16 states.
template <typename T, bool V4, bool WHOLE>
__global__ void __launch_bounds__(512) k_scan_walk(ScanArgs a) {
    constexpr int ROWS = 64, LD = ROWS + 4, NB = ROWS / kWalk, CD = kWalk + 4;  // strides of B | C's columns, of a row's channels
    // fp32: the state goes from block to block by one decay over the sum of the block's steps, as it does from run to run.  Error against
    // 64 bits, 500 rows of 2,048 channels, outputs / state: runs 1.10e-7 / 1.02e-7, step by step 1.20e-7 / 1.25e-7, so 1.10e-7 /
    // 0.98e-7 (a 500-token prompt 0.6 % longer).  bf16 rows round 10,000 times as much: 40 prompts' and steps' error 1.001 +- 0.006 of
    // that of runs.
    constexpr bool LEAP = sizeof(T) == 4;
    __shared__ __attribute__((aligned(16))) float sbc[2][2 * kWalk][LD], sdt[2][ROWS][CD], sdx[2][ROWS][CD], sy[2][ROWS][CD];
    const SeqInfo q = a.seqs[blockIdx.y];
    // an XCD's workgroups have neighbouring channels, which share the lines of every row
    const int per = gridDim.x / 8, c0 = ((blockIdx.x % 8) * per + blockIdx.x / 8) * kWalk;
    const int tid = threadIdx.x & 255, N = a.N, len = q.len, ngr = (len + ROWS - 1) / ROWS;
    if (c0 >= max(a.C, a.ldy)) return;
    if (threadIdx.x < 256) {
        const int lane = tid & 63, j = tid & 15, ch = tid >> 4, c = c0 + ch;
        const bool mine = c < a.C && j < N;
        const int cc = min(c, a.C - 1), n = min(j, N - 1);
        const long at = ((long)q.slot * a.C + cc) * N + n;
        const float al = bf2f(a.A_log[(long)cc * N + n]), s0 = a.state[at];
        // dt A in powers of two: exp(dt A) = exp2(dt A log2 e)
        const float A = j < N ? -expf(al) * 1.4426950408889634f : 0.0f;
        float S = q.start > 0 && j < N ? s0 : 0.0f;
        __syncthreads();
        for (int i = 0; i < ngr; ++i) {
            const int k = i & 1, rows = min(ROWS, len - i * ROWS);
            struct Block { f32x4 B[4], C[4]; float dt, dx; };
            auto read = [&](int b, Block& o) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    o.B[v] = *reinterpret_cast<const f32x4*>(&sbc[k][j][b * kWalk + 4 * v]);
                    o.C[v] = *reinterpret_cast<const f32x4*>(&sbc[k][kWalk + j][b * kWalk + 4 * v]);
                }
                o.dt = sdt[k][b * kWalk + j][ch];  // lane j has row j of the block
                o.dx = sdx[k][b * kWalk + j][ch];
            };
            // n: rows of the block; those past the sequence's end leave the state (their step of 0 does not where A is -inf, nor does
            // their input of 0 where the last row's B, which they repeat, is not finite)
            auto walk = [&](auto full, int b, int n, const Block& o) {
                float e[kWalk], w[kWalk], p[kWalk];
                each_step([&](auto ti) {  // decays and inputs: none waits for another
                    constexpr int t = decltype(ti)::value;
                    e[t] = __builtin_amdgcn_exp2f(of_step<t>(o.dt) * A);
                    w[t] = of_step<t>(o.dx) * o.B[t / 4][t % 4];
                }, std::make_integer_sequence<int, kWalk>{});
                __builtin_amdgcn_sched_barrier(0);
                const float entry = S;
                float own = 0.0f;  // the block's state from its own inputs
#pragma unroll
                for (int t = 0; t < kWalk; ++t) {
                    const bool there = full || t < n;
                    S = there ? fmaf(e[t], S, w[t]) : S;
                    if constexpr (LEAP) own = there ? fmaf(e[t], own, w[t]) : own;
                    p[t] = S * o.C[t / 4][t % 4];
                }
                sy[k][b * kWalk + j][ch] = sum_of_step(p, lane);
                if constexpr (LEAP) S = fmaf(__builtin_amdgcn_exp2f(sum_of_lanes(o.dt) * A), entry, own);
            };
            Block o[2];
            read(0, o[0]);
            if (rows > ROWS - kWalk) {
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    if (b + 1 < NB) read(b + 1, o[(b + 1) & 1]);
                    if (b + 1 < NB || rows == ROWS) walk(std::true_type{}, b, kWalk, o[b & 1]);
                    else walk(std::false_type{}, b, rows - b * kWalk, o[b & 1]);
                }
            } else {
#pragma clang loop unroll(disable)
                for (int b = 0; b * kWalk < rows; ++b) {
                    if (b) read(b, o[0]);
                    walk(std::false_type{}, b, rows - b * kWalk, o[0]);
                }
            }
            __syncthreads();
        }
        if (mine) a.state[at] = S;
        return;
    }
    typedef T T4 __attribute__((ext_vector_type(4)));
    const float* __restrict__ dp = a.dt + (long)q.off * a.C;
    const T* __restrict__ xp = reinterpret_cast<const T*>(a.x) + (long)q.off * a.ldx;
    const T* __restrict__ zp = reinterpret_cast<const T*>(a.z) + (long)q.off * a.ldz;
    T* __restrict__ yp = reinterpret_cast<T*>(a.y) + (long)q.off * a.ldy;
    const float* __restrict__ bc = a.bc + (long)q.off * 2 * N;
    // element e of a thread: V4: row r0, channel c0 + h0 + e; else row r0 + 16 e, channel c0 + h0
    const int r0 = V4 ? tid >> 2 : tid >> 4, h0 = V4 ? (tid & 3) * 4 : tid & 15, hc = V4 ? c0 + h0 : min(c0 + h0, a.C - 1);
    auto row_of = [&](int e) { return V4 ? r0 : r0 + 16 * e; };
    f32x4 bias, Dc;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        bias[e] = bf2f(a.dtb[V4 ? hc + e : hc]);
        Dc[e] = bf2f(a.Dw[V4 ? hc + e : hc]);
    }
    // B | C: WHOLE: columns 4 (tid % 8) .. of rows tid / 8 and tid / 8 + 32; else column tid % 32 of rows tid / 32 + 8 i
    const int col = WHOLE ? (tid & 7) * 4 : tid & 31, rb = WHOLE ? tid >> 3 : tid >> 5, cn = col & 15;
    f32x4 hbc[2], hd;
    T4 hx, hz;
    auto hold = [&](int t0) {  // rows past the end repeat the last one (never used)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if constexpr (WHOLE) {
                hbc[i] = *reinterpret_cast<const f32x4*>(bc + (long)min(t0 + rb + 32 * i, len - 1) * 32 + col);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    hbc[i][e] = cn < N ? bc[(long)min(t0 + rb + 8 * (4 * i + e), len - 1) * 2 * N + (col < 16 ? cn : N + cn)] : 0.0f;
            }
        if constexpr (V4) {
            const long r = min(t0 + r0, len - 1);
            hd = *reinterpret_cast<const f32x4*>(dp + r * a.C + hc);
            hx = *reinterpret_cast<const T4*>(xp + r * a.ldx + hc);
            hz = *reinterpret_cast<const T4*>(zp + r * a.ldz + hc);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const long r = min(t0 + row_of(e), len - 1);
                hd[e] = dp[r * a.C + hc];
                hx[e] = xp[r * a.ldx + hc];
                hz[e] = zp[r * a.ldz + hc];
            }
        }
    };
    struct Gate { f32x4 g, dx; };  // of a row that is being walked: the gate, and what the input adds by itself
    auto stage = [&](int to, int t0, Gate& gate) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if constexpr (WHOLE) sbc[to][col + e][rb + 32 * i] = hbc[i][e];
                else sbc[to][col][rb + 8 * (4 * i + e)] = hbc[i][e];
        f32x4 dt, dx;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const T xe = hx[e], ze = hz[e];
            const bool row = t0 + row_of(e) < len;  // no step past the end
            const float x = ldf(&xe);
            gate.g[e] = siluf_(ldf(&ze));
            gate.dx[e] = x;
            dt[e] = row ? softplus_of<T>(hd[e] + bias[e]) : 0.0f;
            dx[e] = row ? dt[e] * x : 0.0f;
        }
        if constexpr (V4) {
            *reinterpret_cast<f32x4*>(&sdt[to][r0][h0]) = dt;
            *reinterpret_cast<f32x4*>(&sdx[to][r0][h0]) = dx;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sdt[to][row_of(e)][h0] = dt[e];
                sdx[to][row_of(e)][h0] = dx[e];
            }
        }
    };
    auto leave = [&](int from, int t0, const Gate& gate) {
        T4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = gate.g[e] * fmaf(Dc[e], gate.dx[e], sy[from][row_of(e)][V4 ? h0 + e : h0]);
            T r;
            stf(&r, c0 + h0 < a.C ? v : 0.0f);  // columns C .. ldy - 1 are zero
            o[e] = r;
        }
        if constexpr (V4) {
            if (t0 + r0 < len) *reinterpret_cast<T4*>(yp + (long)(t0 + r0) * a.ldy + hc) = o;
        } else if (c0 + h0 < a.ldy) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (t0 + row_of(e) < len) yp[(long)(t0 + row_of(e)) * a.ldy + c0 + h0] = o[e];
        }
    };
    Gate before, now, next;
    hold(0);
    stage(0, 0, now);
    if (1 < ngr) hold(ROWS);
    __syncthreads();
    for (int i = 0; i < ngr; ++i) {
        if (i > 0) leave(~i & 1, (i - 1) * ROWS, before);
        if (i + 1 < ngr) {
            stage(~i & 1, (i + 1) * ROWS, next);
            if (i + 2 < ngr) hold((i + 2) * ROWS);
        }
        before = now;
        now = next;
        __syncthreads();
    }
    leave(~ngr & 1, (ngr - 1) * ROWS, before);
}

template <typename T, int NPL, int LPC>
void launch_scan(hipStream_t s, const ScanArgs& a) {
    const int CPB = 256 / LPC;
    const dim3 grid((std::max(a.C, a.ldy) + CPB - 1) / CPB, a.nchunk);
    if (a.multi) {
        hipLaunchKernelGGL((k_scan<T, NPL, LPC, 0>), grid, dim3(256), 0, s, a);
        const long CN = (long)a.C * a.N;
        hipLaunchKernelGGL(k_scan_carry, dim3((unsigned)((CN + 255) / 256), a.nchunk), dim3(256), 0, s, a);
    }
    hipLaunchKernelGGL((k_scan<T, NPL, LPC, 1>), grid, dim3(256), 0, s, a);
}

template <typename T>
void launch_walk(hipStream_t s, const ScanArgs& a) {
    const dim3 grid(((std::max(a.C, a.ldy) + kWalk - 1) / kWalk + 7) / 8 * 8, a.nseq), blk(512);
    const uintptr_t at = reinterpret_cast<uintptr_t>(a.dt) | reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.z) |
                         reinterpret_cast<uintptr_t>(a.y);
    const bool v4 = a.C % kWalk == 0 && a.ldy == a.C && a.ldx % 4 == 0 && a.ldz % 4 == 0 && at % 16 == 0;
    const bool whole = a.N == 16 && reinterpret_cast<uintptr_t>(a.bc) % 16 == 0;
    if (v4 && whole) hipLaunchKernelGGL((k_scan_walk<T, true, true>), grid, blk, 0, s, a);
    else if (v4) hipLaunchKernelGGL((k_scan_walk<T, true, false>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((k_scan_walk<T, false, false>), grid, blk, 0, s, a);
}

template <typename T>
void scan_t(hipStream_t s, const ScanArgs& a) {
    if (a.walk) return launch_walk<T>(s, a);
    switch (scan_lanes(a.N)) {
        case 1:
            if (a.N <= 8) launch_scan<T, 8, 1>(s, a);
            else launch_scan<T, 16, 1>(s, a);
            break;
        case 2: launch_scan<T, 16, 2>(s, a); break;
        case 4: launch_scan<T, 16, 4>(s, a); break;
        case 8: launch_scan<T, 16, 8>(s, a); break;
        default: launch_scan<T, 16, 16>(s, a); break;
    }
}

// ---------------------------------------------------------------- minGRU
// V channels per lane (2 where rows allow it, else 1)
template <typename T, int PHASE, int V>
__global__ void __launch_bounds__(64) k_gru(GruArgs a) {
    const ChunkInfo ck = a.chunks[blockIdx.y];
    const bool last = ck.idx + 1 == ck.nch;
    if (PHASE == 0 && last) return;
    const SeqInfo q = a.seqs[ck.seq];
    const int c = (blockIdx.x * 64 + threadIdx.x) * V;
    const T* __restrict__ zp = reinterpret_cast<const T*>(a.zug) + (long)ck.row * a.ld + c;
    T* __restrict__ yp = reinterpret_cast<T*>(a.y) + (long)ck.row * a.ldy + c;
    if (c >= a.C) {  // columns C .. ldy - 1 are zero (V == 1 only)
        if (PHASE == 1 && c < a.ldy)
            for (int t = 0; t < ck.len; ++t) stf(yp + (long)t * a.ldy, 0.0f);
        return;
    }
    float S[V], keep[V];
    float* cs = a.cstate + ((long)blockIdx.y * 2) * a.C + c;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        S[v] = 0.0f;
        keep[v] = 1.0f;
        if constexpr (PHASE == 1) {
            if (ck.nch > 1) S[v] = cs[v];
            else if (q.start > 0) S[v] = a.state[(long)q.slot * a.C + c + v];
        }
    }
    struct alignas(sizeof(T) * V) Raw { T v[V]; };
    Raw rz[kPre], ru[kPre], rg[PHASE ? kPre : 1];
    auto fetch = [&](int t0) {  // rows past the chunk repeat its last one (never used)
#pragma unroll
        for (int t = 0; t < kPre; ++t) {
            const T* r = zp + (long)min(t0 + t, ck.len - 1) * a.ld;
            rz[t] = *reinterpret_cast<const Raw*>(r);
            ru[t] = *reinterpret_cast<const Raw*>(r + a.C);
            if constexpr (PHASE == 1) rg[t] = *reinterpret_cast<const Raw*>(r + 2 * a.C);
        }
    };
    fetch(0);
    for (int t0 = 0; t0 < ck.len; t0 += kPre) {
        float z[kPre][V], u[kPre][V], g[kPre][V];
#pragma unroll
        for (int t = 0; t < kPre; ++t)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                z[t][v] = ldf(&rz[t].v[v]);
                u[t][v] = ldf(&ru[t].v[v]);
                if constexpr (PHASE == 1) g[t][v] = ldf(&rg[t].v[v]);
            }
        if (t0 + kPre < ck.len) fetch(t0 + kPre);
#pragma unroll
        for (int t = 0; t < kPre; ++t) {
            if (t0 + t >= ck.len) break;
            float y[V];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const float zz = sigmoidf_(z[t][v]);
                S[v] = fmaf(1.0f - zz, S[v], zz * gru_candidate(u[t][v]));
                if constexpr (PHASE == 0) keep[v] *= 1.0f - zz;
                else y[v] = S[v] * siluf_(g[t][v]);
            }
            if constexpr (PHASE == 1) {
                Raw o;
#pragma unroll
                for (int v = 0; v < V; ++v) stf(&o.v[v], y[v]);
                *reinterpret_cast<Raw*>(yp + (long)(t0 + t) * a.ldy) = o;
            }
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        if constexpr (PHASE == 0) {
            cs[v] = S[v];
            cs[a.C + v] = keep[v];
        } else if (last) {
            a.state[(long)q.slot * a.C + c + v] = S[v];
        }
    }
}

__global__ void __launch_bounds__(64) k_gru_carry(GruArgs a) {
    const ChunkInfo ck = a.chunks[blockIdx.y];
    if (ck.idx != 0 || ck.nch < 2) return;
    const SeqInfo q = a.seqs[ck.seq];
    const int c = blockIdx.x * 64 + threadIdx.x;
    if (c >= a.C) return;
    float S = q.start > 0 ? a.state[(long)q.slot * a.C + c] : 0.0f;
    float* e = a.cstate + ((long)blockIdx.y * 2) * a.C + c;
    const int n = ck.nch - 1;
    for (int k0 = 0; k0 <= n; k0 += kPre) {
        float end[kPre], keep[kPre];
#pragma unroll
        for (int k = 0; k < kPre; ++k) {
            const long r = min(k0 + k, n - 1);
            end[k] = e[r * 2 * a.C];
            keep[k] = e[r * 2 * a.C + a.C];
        }
#pragma unroll
        for (int k = 0; k < kPre; ++k)
            if (k0 + k <= n) {
                e[(long)(k0 + k) * 2 * a.C] = S;
                S = fmaf(keep[k], S, end[k]);
            }
    }
}

// ---- sequences walked whole: one wave has 16 channels' states, eight others the rest
// The gates, candidates and outputs of 128 rows are formed around the walk, ahead of it and after it, as in k_scan_walk.  V4: a thread of
// the eight waves has four channels of one row, else one channel of four rows.
// The walking wave takes 32 rows at a time, as runs of 8 side by side: what each leaves by itself and keeps, the state before each from
// these, then its rows.  Row after row instead, the roundings of a whole sequence add up: error against 64 bits, 500 fp32 rows, gates of
// sigmoid(-4), outputs / state, of that of three launches over runs 1.08 / 1.13, as it is now 0.99 / 1.00.
// Bound by the other waves' three sigmoids a value, two waves a SIMD: 8 ns a row of the longest sequence (four waves and 64 rows 18, rows held
// one group ahead or two alike).  us a layer, three launches of runs / this: 1,024 + 387 + 129 rows of 2,048 channels 21.7 / 12.6, 500
// rows of 1,024 fp32 channels 14.7 / 6.8; the line between them: gru_walks.

// v of lanes 0 .. 15, 16 .. 31, 32 .. 47 and 48 .. 63, in all four
__device__ __forceinline__ void of_parts(float v, float (&o)[4]) {
    const unsigned u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);  // of the even parts, of the odd ones
    const auto b = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false), c = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
    o[0] = __uint_as_float(b[0]), o[1] = __uint_as_float(c[0]), o[2] = __uint_as_float(b[1]), o[3] = __uint_as_float(c[1]);
}

template <typename T, bool V4>
__global__ void __launch_bounds__(576) k_gru_walk(GruArgs a) {
    constexpr int ROWS = 128, LD = ROWS + 4;
    __shared__ __attribute__((aligned(16))) float sa[2][kWalk][LD], sb[2][kWalk][LD], ss[2][kWalk][LD];  // keep, add, states
    const SeqInfo q = a.seqs[blockIdx.y];
    // an XCD's workgroups have neighbouring channels, which share the lines of every row
    const int per = gridDim.x / 8, c0 = ((blockIdx.x % 8) * per + blockIdx.x / 8) * kWalk;
    const int len = q.len, ngr = (len + ROWS - 1) / ROWS;
    if (c0 >= max(a.C, a.ldy)) return;
    if (threadIdx.x >= 512) {
        // 8 of 32 rows each: lanes 0 .. 15 the first, 16 .. 31 the next, ..
        const int ch = threadIdx.x & 15, part = (threadIdx.x & 63) >> 4, c = c0 + ch;
        const bool mine = c < a.C;
        float* st = a.state + (long)q.slot * a.C + min(c, a.C - 1);
        float S = q.start > 0 ? *st : 0.0f;
        __syncthreads();
        for (int i = 0; i < ngr; ++i) {
            const int k = i & 1, rows = len - i * ROWS;
            struct Piece { f32x4 a[2], b[2]; float own, kept; };  // what 8 rows leave of no state, and keep of one
            auto read = [&](int h, Piece& w) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    w.a[r] = *reinterpret_cast<const f32x4*>(&sa[k][ch][h + 8 * part + 4 * r]);
                    w.b[r] = *reinterpret_cast<const f32x4*>(&sb[k][ch][h + 8 * part + 4 * r]);
                }
            };
            auto sum = [&](Piece& w) {
                w.own = 0.0f, w.kept = 1.0f;
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    w.own = fmaf(w.a[r / 4][r % 4], w.own, w.b[r / 4][r % 4]);
                    w.kept *= w.a[r / 4][r % 4];
                }
            };
            auto walk = [&](int h, Piece& w) {
                float o[4], f[4], e = S;
                of_parts(w.own, o);
                of_parts(w.kept, f);
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    if (part == n) e = S;
                    S = fmaf(f[n], S, o[n]);
                }
                const int at = h + 8 * part;
#pragma unroll
                for (int r = 0; r < 2; ++r) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) w.b[r][v] = e = fmaf(w.a[r][v], e, w.b[r][v]);
                    *reinterpret_cast<f32x4*>(&ss[k][ch][at + 4 * r]) = w.b[r];
                }
                if (mine && at < rows && at + 8 >= rows) *st = e;  // the sequence's last row
            };
            Piece w[ROWS / 32];
            if (rows > ROWS - 32) {
#pragma unroll
                for (int n = 0; n < ROWS / 32; ++n) read(32 * n, w[n]);
#pragma unroll
                for (int n = 0; n < ROWS / 32; ++n) sum(w[n]);
#pragma unroll
                for (int n = 0; n < ROWS / 32; ++n) walk(32 * n, w[n]);
            } else {
#pragma clang loop unroll(disable)
                for (int h = 0; h < rows; h += 32) {  // rows past the end keep the state
                    read(h, w[0]);
                    sum(w[0]);
                    walk(h, w[0]);
                }
            }
            __syncthreads();
        }
        return;
    }
    typedef T T4 __attribute__((ext_vector_type(4)));
    const int tid = threadIdx.x;
    const T* __restrict__ zp = reinterpret_cast<const T*>(a.zug) + (long)q.off * a.ld;
    T* __restrict__ yp = reinterpret_cast<T*>(a.y) + (long)q.off * a.ldy;
    // element e of a thread: V4: row r0, channel c0 + h0 + e; else row r0 + e, channel c0 + h0; 16 rows a wave
    const int r0 = V4 ? tid >> 2 : (tid >> 4) * 4, w0 = (tid >> 6) * 16, h0 = V4 ? (tid & 3) * 4 : tid & 15, hc = V4 ? c0 + h0 : min(c0 + h0, a.C - 1);
    auto row_of = [&](int e) { return V4 ? r0 : r0 + e; };
    struct Held { T4 z, u, g; };
    auto hold = [&](int t0, Held& h) {  // rows past the end repeat the last one (never used)
        if constexpr (V4) {
            const T* r = zp + (long)min(t0 + r0, len - 1) * a.ld + hc;
            h.z = *reinterpret_cast<const T4*>(r);
            h.u = *reinterpret_cast<const T4*>(r + a.C);
            h.g = *reinterpret_cast<const T4*>(r + 2 * a.C);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const T* r = zp + (long)min(t0 + row_of(e), len - 1) * a.ld + hc;
                h.z[e] = r[0];
                h.u[e] = r[a.C];
                h.g[e] = r[2 * a.C];
            }
        }
    };
    auto stage = [&](int to, int t0, const Held& h, f32x4& gate) {
        if (w0 >= (len - t0 + 31 & ~31)) return;  // the walker stops there
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const T ze = h.z[e], ue = h.u[e], ge = h.g[e];
            const bool row = t0 + row_of(e) < len;
            const float zz = sigmoidf_(ldf(&ze));
            const int ch = V4 ? h0 + e : h0;
            sa[to][ch][row_of(e)] = row ? 1.0f - zz : 1.0f;
            sb[to][ch][row_of(e)] = row ? zz * gru_candidate(ldf(&ue)) : 0.0f;
            gate[e] = siluf_(ldf(&ge));
        }
    };
    auto leave = [&](int from, int t0, const f32x4& gate) {
        T4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            T r;
            stf(&r, c0 + h0 < a.C ? ss[from][V4 ? h0 + e : h0][row_of(e)] * gate[e] : 0.0f);  // columns C .. ldy - 1 are zero
            o[e] = r;
        }
        if constexpr (V4) {
            if (t0 + r0 < len) *reinterpret_cast<T4*>(yp + (long)(t0 + r0) * a.ldy + hc) = o;
        } else if (c0 + h0 < a.ldy) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (t0 + row_of(e) < len) yp[(long)(t0 + row_of(e)) * a.ldy + c0 + h0] = o[e];
        }
    };
    f32x4 before{}, now{}, next{};
    Held even, odd;  // two groups of rows on their way
    auto turn = [&](int i, Held& h) {  // h: group i + 1
        if (i > 0) leave(~i & 1, (i - 1) * ROWS, before);
        if (i + 1 < ngr) {
            stage(~i & 1, (i + 1) * ROWS, h, next);
            if (i + 3 < ngr) hold((i + 3) * ROWS, h);
        }
        before = now;
        now = next;
        __syncthreads();
    };
    hold(0, even);
    if (1 < ngr) hold(ROWS, odd);
    stage(0, 0, even, now);
    if (2 < ngr) hold(2 * ROWS, even);
    __syncthreads();
    for (int i = 0; i < ngr; i += 2) {
        turn(i, odd);
        if (i + 1 < ngr) turn(i + 1, even);
    }
    leave(~ngr & 1, (ngr - 1) * ROWS, before);
}

template <typename T>
void launch_gru_walk(hipStream_t s, const GruArgs& a) {
    const dim3 grid(((std::max(a.C, a.ldy) + kWalk - 1) / kWalk + 7) / 8 * 8, a.nseq), blk(576);
    const uintptr_t at = reinterpret_cast<uintptr_t>(a.zug) | reinterpret_cast<uintptr_t>(a.y);
    if (a.C % kWalk == 0 && a.ldy == a.C && a.ld % 4 == 0 && at % 16 == 0) hipLaunchKernelGGL((k_gru_walk<T, true>), grid, blk, 0, s, a);
    else hipLaunchKernelGGL((k_gru_walk<T, false>), grid, blk, 0, s, a);
}

template <typename T, int V>
void gru_v(hipStream_t s, const GruArgs& a) {
    const int cols = std::max(a.C, V == 1 ? a.ldy : a.C);
    const dim3 grid((cols + 64 * V - 1) / (64 * V), a.nchunk);
    if (a.multi) {
        hipLaunchKernelGGL((k_gru<T, 0, V>), grid, dim3(64), 0, s, a);
        hipLaunchKernelGGL(k_gru_carry, dim3((a.C + 63) / 64, a.nchunk), dim3(64), 0, s, a);
    }
    hipLaunchKernelGGL((k_gru<T, 1, V>), grid, dim3(64), 0, s, a);
}

template <typename T>
void gru_t(hipStream_t s, const GruArgs& a) {
    if (a.walk) return launch_gru_walk<T>(s, a);
    if (a.C % 8 == 0 && a.ld % 8 == 0) gru_v<T, 2>(s, a);
    else gru_v<T, 1>(s, a);
}

template <typename T>
void conv_t(hipStream_t s, const T* xz, int ldxz, int C, int K, const uint16_t* w, const uint16_t* b,
            const SeqInfo* seqs, int nseq, const ChunkInfo* chunks, int nchunk, bool fresh, float* taps, T* out, int ldo) {
    const dim3 gv((C / 8 + 63) / 64, nchunk), g1((ldo + 63) / 64, nchunk), blk(256);
#define CONV_(kt, grid) hipLaunchKernelGGL((k_conv_silu<T, kt>), grid, blk, 0, s, xz, ldxz, C, K, w, b, seqs, chunks, taps, keep, out, ldo)
    const bool vec = C % 8 == 0 && ldxz % 8 == 0;
    float* keep = vec && fresh && K >= 2 && K <= 5 ? taps : nullptr;
    if (vec && K == 2) CONV_(2, gv);
    else if (vec && K == 3) CONV_(3, gv);
    else if (vec && K == 4) CONV_(4, gv);
    else if (vec && K == 5) CONV_(5, gv);
    else CONV_(0, g1);
#undef CONV_
    if (K > 1 && !keep)
        hipLaunchKernelGGL((k_conv_taps<T>), dim3((C + 255) / 256, nseq), dim3(256), 0, s, xz, ldxz, C, K, seqs, taps);
}

}  // namespace

int scan_max_state() { return 256; }

void conv_silu(hipStream_t s, Act act, const void* xz, int ldxz, int C, int K, const uint16_t* w, const uint16_t* b,
               const SeqInfo* seqs, int nseq, const ChunkInfo* chunks, int nchunk, bool fresh, float* taps, void* out, int ldo) {
    if (act == ACT_F32)
        conv_t(s, reinterpret_cast<const float*>(xz), ldxz, C, K, w, b, seqs, nseq, chunks, nchunk, fresh, taps,
               reinterpret_cast<float*>(out), ldo);
    else
        conv_t(s, reinterpret_cast<const uint16_t*>(xz), ldxz, C, K, w, b, seqs, nseq, chunks, nchunk, fresh, taps,
               reinterpret_cast<uint16_t*>(out), ldo);
}

void scan_inputs(hipStream_t s, Act act, const float* slabs, int split, int rows, int R, int N, void* dtl, int ldd,
                 float* bc) {
    if (act == ACT_F32)
        hipLaunchKernelGGL((k_scan_inputs<float>), dim3(rows), dim3(256), 0, s, slabs, split, rows, R, N,
                           reinterpret_cast<float*>(dtl), ldd, bc);
    else
        hipLaunchKernelGGL((k_scan_inputs<uint16_t>), dim3(rows), dim3(256), 0, s, slabs, split, rows, R, N,
                           reinterpret_cast<uint16_t*>(dtl), ldd, bc);
}

void selective_scan(hipStream_t s, Act act, const ScanArgs& a) {
    if (act == ACT_F32) scan_t<float>(s, a);
    else scan_t<uint16_t>(s, a);
}

void mingru_scan(hipStream_t s, Act act, const GruArgs& a) {
    if (act == ACT_F32) gru_t<float>(s, a);
    else gru_t<uint16_t>(s, a);
}

}  // namespace pgmi
