// kernels_step.hip -- one token per sequence: projections as weight-streaming GEMVs or skinny MFMA products
// (up to 16 rows) of any size with the surrounding steps fused (streams' read + grouped norm in front; convolution step, minGRU step, gated
// activation, streams' update or argmax behind), and the selective-scan step.
#include <algorithm>
#include <cassert>
#include <type_traits>

#include "act.h"
#include "decoder.h"
#include "tile_f32.h"

namespace pgmi {

namespace {

constexpr int UN = 4;  // K steps (512 elements each) whose weight loads are in flight together

// eight activations as loaded
struct X8b { uint4 q; };
struct X8f { float4 a, b; };
template <typename T> struct X8 { typedef X8b type; };
template <> struct X8<float> { typedef X8f type; };
__device__ __forceinline__ void ldx(const uint16_t* p, X8b& x) { x.q = *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ void ldx(const float* p, X8f& x) {
    x.a = *reinterpret_cast<const float4*>(p);
    x.b = *reinterpret_cast<const float4*>(p + 4);
}
__device__ __forceinline__ float dotx(const uint4 w, const X8b& x, float acc) { return dot8(w, x.q, acc); }
__device__ __forceinline__ float dotx(const uint4 w, const X8f& x, float acc) {
    const uint32_t q[4] = {w.x, w.y, w.z, w.w};
    const float v[8] = {x.a.x, x.a.y, x.a.z, x.a.w, x.b.x, x.b.y, x.b.z, x.b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        acc = fmaf(__uint_as_float(q[i] << 16), v[2 * i], acc);
        acc = fmaf(__uint_as_float(q[i] & 0xFFFF0000u), v[2 * i + 1], acc);
    }
    return acc;
}

constexpr int unit_rows(int mode) { return mode == GR_GRU ? 3 : 2; }
// outputs a unit covers (plain modes: two rows; GRU, SwiGLU: one channel)
constexpr int unit_outs(int mode) { return mode == GR_GRU || mode == GR_SWIGLU ? 1 : 2; }

// The step that follows a projection.  Its operands are asked for ahead of the sums: read where they are used, in turn and each behind
// its own wait, they were most of a small projection's time (a step of the 1,024-wide
// streams model, these and the scan's and attention's below: 280 -> 249 us).
struct StepIn {  // of output n of row b
    int slot, pos;
    float v[8];     // the state, or the streams
    uint16_t w[5];  // bias, or taps
};
// the streams' coefficients (up to 8 streams), a lane each: in[s], out[t] and mix[s S + t]
struct StepMix {
    int in, out, mix;
};
template <int MODE, bool IN>
__device__ __forceinline__ StepMix step_mix(const GemvRtArgs& a) {
    StepMix m{};
    const int lane = threadIdx.x & 63;
    if constexpr (IN) m.in = (a.in ? a.in : a.nw)[min(lane, a.S - 1)];
    if constexpr (MODE == GR_STREAMS) {
        m.out = (a.mix ? a.wout : a.W)[a.mix ? min(lane, a.S - 1) : 0];
        m.mix = (a.mix ? a.mix : a.W)[a.mix ? min(lane, a.S * a.S - 1) : 0];
    }
    return m;
}

// (the slot and position by lanes, also where all have the same: a scalar load would be waited for with the arguments, before
// anything else is asked for)
template <int MODE>
__device__ __forceinline__ void step_slot(const GemvRtArgs& a, int b, StepIn& e) {
    if constexpr (MODE == GR_CONV || MODE == GR_GRU) {
        e.slot = a.slot[b];
        e.pos = a.pos[b];
    }
}
// n and b past the last ones: the last ones'.  MS: streams at most
template <int MODE, int MS>
__device__ __forceinline__ void step_load(const GemvRtArgs& a, int n, int b, StepIn& e) {
    n = min(n, a.N - 1);
    if constexpr (MODE == GR_ACT) {
        e.w[0] = (a.bias ? a.bias : a.W)[n];
    } else if constexpr (MODE == GR_CONV) {
        const int c = min(n, a.C - 1), KT = a.taps_k;
#pragma unroll
        for (int j = 0; j < 4; ++j) e.w[j] = a.cw[(long)c * KT + min(j, KT - 1)];
        e.w[4] = a.cb[c];
    } else if constexpr (MODE == GR_GRU) {
        e.w[0] = a.bias[n];
        e.w[1] = a.bias[a.N + n];
    } else if constexpr (MODE == GR_STREAMS) {
        const float* p = a.X + (long)min(b, a.B - 1) * a.S * a.D + n;
#pragma unroll
        for (int s = 0; s < 2; ++s) e.v[s] = p[(long)min(s, a.S - 1) * a.D];
        if (a.S > 2)
#pragma unroll
            for (int s = 2; s < MS; ++s) e.v[s] = p[(long)min(s, a.S - 1) * a.D];
    }
}
// what is found by the slot
template <int MODE>
__device__ __forceinline__ void step_state(const GemvRtArgs& a, int n, StepIn& e) {
    if constexpr (MODE == GR_CONV) {
        const int KT = a.taps_k;
        const float* tp = a.state + (long)e.slot * (KT - 1) * a.C + min(n, a.C - 1);
#pragma unroll
        for (int j = 0; j < 3; ++j) e.v[j] = (KT > 1 ? tp : a.state)[(long)max(0, min(j, KT - 2)) * a.C];
    } else if constexpr (MODE == GR_GRU) {
        e.v[0] = a.state[(long)e.slot * a.N + min(n, a.N - 1)];
    }
}
// output n of row b (v: its sum over K; GR_GRU: v = z, v1 = u, v2 = g; GR_SWIGLU: v = gate, v1 = up), `mine` where both are there and
// this thread's: every (n, b) is handled by one thread.  Called by whole waves: the streams' coefficients are read from the lanes that
// hold them, which a branch around the call would have switched off.
template <typename T, int MODE, int MS>
__device__ __forceinline__ void step_store(const GemvRtArgs& a, bool mine, int n, int b, float v, float v1, float v2, const StepIn& e,
                                           const StepMix& m) {
    if constexpr (MODE == GR_STREAMS) {  // the whole column of streams at once
        float* Xr = a.X + (long)b * a.S * a.D + n;
        if (!a.mix) {
            if (mine) *Xr = fmaf(a.mult, v, e.v[0]);
            return;
        }
        for (int t = 0; t < a.S; ++t) {
            float y = of_lane(m.out, t) * v;
#pragma unroll
            for (int s = 0; s < MS; ++s)
                if (s < a.S) y = fmaf(of_lane(m.mix, s * a.S + t), e.v[s], y);
            if (mine) Xr[(long)t * a.D] = y;
        }
        return;
    }
    if (!mine) return;
    T* out = reinterpret_cast<T*>(a.out) + (long)b * a.ldo + n;
    if constexpr (MODE == GR_ACT) {
        stf(out, a.bias ? v + bf2f(e.w[0]) : v);
    } else if constexpr (MODE == GR_LOGITS || MODE == GR_F32) {
        reinterpret_cast<float*>(a.out)[(long)b * a.ldo + n] = v;
    } else if constexpr (MODE == GR_CONV) {
        if (n >= a.C) {
            stf(reinterpret_cast<T*>(a.out2) + (long)b * a.ldo2 + n - a.C, v);
            return;
        }
        const int KT = a.taps_k;
        const uint16_t* cw = a.cw + (long)n * KT;
        float* tp = a.state + (long)e.slot * (KT - 1) * a.C + n;
        const uint16_t w0 = e.w[0], w1 = e.w[1], w2 = e.w[2], w3 = e.w[3];  // (a choice among an array's places keeps it in memory)
        const uint16_t last = KT == 4 ? w3 : KT == 3 ? w2 : KT == 2 ? w1 : w0;
        float y = fmaf(bf2f(KT > 4 ? cw[KT - 1] : last), v, bf2f(e.w[4]));
        auto tap = [&](int j, uint16_t w, float was) {
            const float o = e.pos == 0 ? 0.0f : was;
            y = fmaf(bf2f(w), o, y);
            if (j > 0) tp[(long)(j - 1) * a.C] = o;
        };
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < KT - 1) tap(j, e.w[j], e.v[j]);
        for (int j = 3; j < KT - 1; ++j) tap(j, cw[j], tp[(long)j * a.C]);
        if (KT > 1) tp[(long)(KT - 2) * a.C] = v;
        stf(out, siluf_(y));
    } else if constexpr (MODE == GR_GRU) {
        const float z = sigmoidf_(v + bf2f(e.w[0]));
        const float S = fmaf(1.0f - z, e.pos > 0 ? e.v[0] : 0.0f, z * gru_candidate(v1 + bf2f(e.w[1])));
        a.state[(long)e.slot * a.N + n] = S;
        stf(out, S * siluf_(v2));
    } else if constexpr (MODE == GR_SWIGLU) {
        stf(out, siluf_(v) * v1);
    }
}

// the columns that pad an activation row to a multiple of 8 are zero
template <typename T, int MODE>
__device__ __forceinline__ void step_pads(const GemvRtArgs& a) {
    if constexpr (MODE == GR_GRU || MODE == GR_SWIGLU || MODE == GR_CONV) {
        const int n = MODE == GR_CONV ? a.C : a.N;
        if (blockIdx.x == 0 && (int)threadIdx.x < a.B)
            for (int k = n; k < a.ldo; ++k) stf(reinterpret_cast<T*>(a.out) + (long)threadIdx.x * a.ldo + k, 0.0f);
    }
}

// WK: waves of the workgroup that share a unit, each a K slice.  XG: the input is rows of activations, loaded with the
// weights; else the streams' read and norm, staged in LDS by the prologue.
template <typename T, int NB, int MODE, int WK, bool XG>
__global__ void __launch_bounds__(256) k_gemv_rt(GemvRtArgs a) {
    constexpr int RW = unit_rows(MODE), UO = unit_outs(MODE), UPB = 4 / WK;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    T* xs = reinterpret_cast<T*>(smem);  // [NB][K]
    __shared__ float red[64];
    __shared__ float part[WK > 1 ? 4 : 1][RW * NB];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nunit = (a.N + UO - 1) / UO, K = a.K;
    const int ustep = gridDim.x * UPB, kw = wave % WK;
    int unit = blockIdx.x * UPB + wave / WK;
    uint4 w[2][RW][UN];
    typename X8<T>::type xr[2][XG ? NB : 1][XG ? UN : 1];
    auto xload = [&](int buf, int k0) {
        if constexpr (XG) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const T* p = reinterpret_cast<const T*>(a.x) + (long)(b < a.B ? b : 0) * a.ldx;
#pragma unroll
                for (int i = 0; i < UN; ++i) {
                    const int k = k0 + (i * WK + kw) * 512 + lane * 8;
                    ldx(p + (k < K ? k : 0), xr[buf][b][i]);
                }
            }
        }
    };
    auto wload = [&](uint4 (&q)[RW][UN], int u, int k0) {
        const int uu = u < nunit ? u : nunit - 1;
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            int n;
            if constexpr (UO == 1) n = r * a.N + uu;
            else { n = uu * 2 + r; n = n < a.N ? n : a.N - 1; }
            const uint16_t* p = a.W + (long)n * a.ldw;
#pragma unroll
            for (int i = 0; i < UN; ++i) {
                const int k = k0 + (i * WK + kw) * 512 + lane * 8;
                q[r][i] = ldg16_sel(p + k, k < K, p);
            }
        }
    };
    wload(w[0], unit, 0);  // in flight during the prologue
    // lane (r, b) of the unit's first wave finishes output r of row b
    const int lr = lane / NB, lb = lane % NB;
    StepIn e;
    step_slot<MODE>(a, min(lb, a.B - 1), e);
    const StepMix mix = step_mix<MODE, false>(a);
    if constexpr (XG) {
        xload(0, 0);
    } else {
        // the streams' read and grouped norm of each row, as streams_norm
        float* u_ = reinterpret_cast<float*>(smem + (size_t)NB * K * sizeof(T));  // [D], then [groups]
        float* inv = u_ + a.D;
        const int P = a.D / a.groups, D = a.D;
        for (int b = 0; b < NB && b < a.B; ++b) {
            const float* Xr = a.X + (long)b * a.S * D;
            if (P % 256 == 0 && D <= 8192) {
                // a wave's 64 x 4 elements lie in one group: one partial per (piece, wave)
                constexpr int PC = 8;
                const int np = (D + 1023) / 1024;
                float4 u[PC];
                ushort4 nw[PC];
#pragma unroll
                for (int i = 0; i < PC; ++i) {
                    u[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    nw[i] = make_ushort4(0, 0, 0, 0);
                    const int d = i * 1024 + tid * 4;
                    if (i < np && d < D) {
                        nw[i] = *reinterpret_cast<const ushort4*>(a.nw + d);
                        for (int s = 0; s < a.S; ++s) {
                            const float c = a.in ? bf2f(a.in[s]) : 1.0f;
                            const float4 q = *reinterpret_cast<const float4*>(Xr + (long)s * D + d);
                            u[i].x = fmaf(c, q.x, u[i].x); u[i].y = fmaf(c, q.y, u[i].y);
                            u[i].z = fmaf(c, q.z, u[i].z); u[i].w = fmaf(c, q.w, u[i].w);
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < PC; ++i)
                    if (i < np) {
                        const float q = wave_sum(u[i].x * u[i].x + u[i].y * u[i].y + u[i].z * u[i].z + u[i].w * u[i].w);
                        if (lane == 0) red[i * 4 + wave] = q;
                    }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < PC; ++i) {
                    const int d = i * 1024 + tid * 4;
                    if (i < np && d < D) {
                        const int p0 = d / P * (P / 256);
                        float q = 0.0f;
                        for (int t = 0; t < P / 256; ++t) q += red[p0 + t];
                        const float f = 1.0f / sqrtf(q / (float)P + a.eps);
                        T* o = xs + b * K + d;
                        stf(o, u[i].x * f * bf2f(nw[i].x));
                        stf(o + 1, u[i].y * f * bf2f(nw[i].y));
                        stf(o + 2, u[i].z * f * bf2f(nw[i].z));
                        stf(o + 3, u[i].w * f * bf2f(nw[i].w));
                    }
                }
                __syncthreads();
                continue;
            }
            for (int d = tid; d < D; d += 256) {
                float u = 0.0f;
                for (int s = 0; s < a.S; ++s) u = fmaf(a.in ? bf2f(a.in[s]) : 1.0f, Xr[(long)s * D + d], u);
                u_[d] = u;
            }
            __syncthreads();
            for (int g = wave; g < a.groups; g += 4) {
                float q = 0.0f;
                for (int i = lane; i < P; i += 64) q = fmaf(u_[g * P + i], u_[g * P + i], q);
                q = wave_sum(q);
                if (lane == 0) inv[g] = 1.0f / sqrtf(q / (float)P + a.eps);
            }
            __syncthreads();
            for (int d = tid; d < K; d += 256) stf(xs + b * K + d, d < D ? u_[d] * inv[d / P] * bf2f(a.nw[d]) : 0.0f);
            __syncthreads();
        }
    }
    float best[NB];
    int bi[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) { best[b] = -INFINITY; bi[b] = 0x7fffffff; }
    float acc[RW][NB];
    auto mac = [&](int buf, int k0) {
#pragma unroll
        for (int i = 0; i < UN; ++i) {
            const int k = k0 + (i * WK + kw) * 512 + lane * 8;
            if (k < K) {
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    typename X8<T>::type x;
                    if constexpr (XG) x = xr[buf][b][i];
                    else ldx(xs + b * K + k, x);
#pragma unroll
                    for (int r = 0; r < RW; ++r) acc[r][b] = dotx(w[buf][r][i], x, acc[r][b]);
                }
            }
        }
    };
    constexpr int KB = UN * WK * 512;  // K elements per block
    // every wave of a workgroup runs the same number of rounds (WK > 1 meets at a barrier)
    for (int u0 = blockIdx.x * UPB; u0 < nunit; u0 += ustep, unit += ustep) {
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[r][b] = 0.0f;
        for (int k0 = 0; k0 < K; k0 += 2 * KB) {
            if (k0 + KB < K) {
                wload(w[1], unit, k0 + KB);
                xload(1, k0 + KB);
            }
            mac(0, k0);
            if (k0 + KB < K) {
                if (k0 + 2 * KB < K) {
                    wload(w[0], unit, k0 + 2 * KB);
                    xload(0, k0 + 2 * KB);
                }
                mac(1, k0 + KB);
            }
        }
        const int n = unit * UO + min(lr, UO - 1);
        step_load<MODE, 8>(a, n, lb, e);
        step_state<MODE>(a, n, e);
        asm volatile("" ::: "memory");
        if (u0 + ustep < nunit) {
            wload(w[0], unit + ustep, 0);
            xload(0, 0);
        }
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[r][b] = wave_sum(acc[r][b]);
        if constexpr (WK > 1) {
            __syncthreads();
            if (lane == 0)
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int b = 0; b < NB; ++b) part[wave][r * NB + b] = acc[r][b];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    float t = 0.0f;
#pragma unroll
                    for (int q = 0; q < WK; ++q) t += part[(wave / WK) * WK + q][r * NB + b];
                    acc[r][b] = t;
                }
        }
        if (unit >= nunit) continue;
        if constexpr (MODE == GR_LOGITS) {
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const int o = unit * 2 + r;
                    if (o < a.N && acc[r][b] > best[b]) { best[b] = acc[r][b]; bi[b] = o; }
                }
        }
        float v = 0.0f, v1 = 0.0f, v2 = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (UO == 1) {
                if (lb == b) { v = acc[0][b]; v1 = acc[1][b]; v2 = acc[RW - 1][b]; }
            } else {
#pragma unroll
                for (int r = 0; r < RW; ++r)
                    if (lr == r && lb == b) v = acc[r][b];
            }
        }
        if (kw == 0) step_store<T, MODE, 8>(a, lr < UO && lb < a.B && n < a.N, n, lb, v, v1, v2, e, mix);
    }
    if constexpr (MODE == GR_LOGITS) {
        __shared__ float sv[4][NB];
        __shared__ int si[4][NB];
        if (lane == 0)
#pragma unroll
            for (int b = 0; b < NB; ++b) { sv[wave][b] = best[b]; si[wave][b] = bi[b]; }
        __syncthreads();
        if (tid < NB && tid < a.B) {
            float v = sv[0][tid];
            int ix = si[0][tid];
            for (int q = 1; q < 4; ++q)
                if (sv[q][tid] > v || (sv[q][tid] == v && si[q][tid] < ix)) { v = sv[q][tid]; ix = si[q][tid]; }
            a.pmax[(long)tid * gridDim.x + blockIdx.x] = v;
            a.pidx[(long)tid * gridDim.x + blockIdx.x] = ix;
        }
    }
    step_pads<T, MODE>(a);
}

// ---------------------------------------------------------------- one row of bf16, K a multiple of 512 up to 2048
// A wave owns a unit's rows whole, the row x of activations in registers.  What bounds it is latency (a unit is one trip to
// memory) and, in the long products, the stream, so
//   - x, or the streams it is made of, is asked for before the first weights: the norm runs while they arrive, a quarter of it
//     in each wave (every wave for itself: 2 streams of 2,048 read four times, 13.2 us where the other form took 12.8);
//   - a unit's epilogue operands are asked for before the next unit's weights, which would otherwise have to land first
//     (loads return in order), the first unit's behind its weights, and the last unit is peeled off so that no branch hides what
//     is in flight;
//   - the streams' few coefficients come before everything else, a lane each (behind the weights, they held up the norm until those
//     were there).
// us, the LDS form / this one, 2 streams of 2,048 values: gate|up 27.3 / 21.7, mamba in + convolution 12.8 / 9.3, minGRU
// 11.2 / 7.9, q|k|v 9.1 / 6.0, output matrix 187 / 158, mamba out 8.4 / 5.8, down 16.6 / 14.4; a step 0.83 / 0.67 ms.
constexpr int one_rows(int mode) { return mode == GR_LOGITS ? 4 : unit_rows(mode); }
constexpr int one_outs(int mode) { return mode == GR_LOGITS ? 4 : unit_outs(mode); }

// CH: K / 512.  NS: 0: x is a row of activations; NS > 0: up to NS streams, read and normed here; NS < 0: up to -NS partials of
// every head of an attention, merged here as k_wattn_dc does (a launch of 5.1 us;
// here 1,024 values of 8 partials take 1.1: 3.3 -> 4.4 us)
template <int MODE, int CH, int NS>
__global__ void __launch_bounds__(256) k_gemv_one(GemvRtArgs a) {
    constexpr int RW = one_rows(MODE), UO = one_outs(MODE);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nunit = (a.N + UO - 1) / UO, ustep = gridDim.x * 4, K = a.K;
    int unit = blockIdx.x * 4 + wave;
    uint4 w[RW][CH], x[CH], nw;
    float4 X[NS > 0 ? NS : 1][2];
    constexpr int MS = NS < 0 ? -NS : 1;
    float2 pv[MS][4], ml[MS];
    // the streams' read and norm are shared out: a wave takes one piece of 512 (of fewer pieces the last one twice)
    const int piece = min(wave, CH - 1), px = piece * 512 + lane * 8;
    static_assert(CH <= 4, "a piece per wave");
    StepIn e;
    step_slot<MODE>(a, min(lane, a.B - 1), e);
    const StepMix mix = step_mix<MODE, (NS > 0)>(a);
    if constexpr (NS == 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c) x[c] = ldg16(reinterpret_cast<const uint16_t*>(a.x) + c * 512 + lane * 8);
    } else if constexpr (NS < 0) {
        const float* p = a.part + (long)(px / a.pe) * a.nsplit * a.prs;
#pragma unroll
        for (int s = 0; s < MS; ++s) {
            const float* q = p + (long)min(s, a.nsplit - 1) * a.prs;
            ml[s] = *reinterpret_cast<const float2*>(q + a.prs - 2);
#pragma unroll
            for (int i = 0; i < 4; ++i) pv[s][i] = *reinterpret_cast<const float2*>(q + px % a.pe + 2 * i);
        }
    } else {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const float* p = a.X + (long)min(s, a.S - 1) * K + px;
            X[s][0] = *reinterpret_cast<const float4*>(p);
            X[s][1] = *reinterpret_cast<const float4*>(p + 4);
        }
        nw = ldg16(a.nw + px);
    }
    auto wload = [&](int u) {
        u = min(u, nunit - 1);  // a wave without a unit repeats the last one's loads, and stores nothing
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            const uint16_t* p = a.W + (UO == 1 ? (long)r * a.N + u : (long)min(u * UO + r, a.N - 1)) * a.ldw + lane * 8;
#pragma unroll
            for (int c = 0; c < CH; ++c) w[r][c] = ldg_nt(p + c * 512);
        }
    };
    auto output = [&](int u) { return u * UO + (UO > 1 ? min(lane, UO - 1) : 0); };
    auto operands = [&](int u) {
        step_load<MODE, 4>(a, output(u), 0, e);
        step_state<MODE>(a, output(u), e);
    };
    wload(unit);
    operands(unit);
    asm volatile("" ::: "memory");  // the stream, and what its epilogue reads, stay ahead of the norm
    if constexpr (NS < 0) {
        __shared__ __attribute__((aligned(16))) uint16_t xs[CH * 512];
        float m = -1e30f, L = 0.0f, t[8] = {};  // an empty split's values were never written: weight 0, not taken
#pragma unroll
        for (int s = 0; s < MS; ++s)
            if (s < a.nsplit && ml[s].y > 0.0f) m = fmaxf(m, ml[s].x);
#pragma unroll
        for (int s = 0; s < MS; ++s) {
            const bool there = s < a.nsplit;
            ml[s].x = there && ml[s].y > 0.0f ? exp2f(ml[s].x - m) : 0.0f;
            L += there ? ml[s].y * ml[s].x : 0.0f;  // a sum that is not a number takes the whole head with it (NaN * 0), as there
        }
#pragma unroll
        for (int s = 0; s < MS; ++s) {
            const float w = ml[s].x / L;
#pragma unroll
            for (int i = 0; i < 8; ++i) t[i] = w > 0.0f ? fmaf(i & 1 ? pv[s][i / 2].y : pv[s][i / 2].x, w, t[i]) : t[i];
        }
        if (wave == piece)
            *reinterpret_cast<uint4*>(xs + px) =
                make_uint4(f2bf(t[0]) | (uint32_t)f2bf(t[1]) << 16, f2bf(t[2]) | (uint32_t)f2bf(t[3]) << 16,
                           f2bf(t[4]) | (uint32_t)f2bf(t[5]) << 16, f2bf(t[6]) | (uint32_t)f2bf(t[7]) << 16);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CH; ++c) x[c] = *reinterpret_cast<const uint4*>(xs + c * 512 + lane * 8);
    }
    if constexpr (NS > 0) {
        __shared__ __attribute__((aligned(16))) uint16_t xs[CH * 512];
        __shared__ float red[4];
        float u[8] = {}, q = 0.0f;
        const int P = K / a.groups;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const float f = a.in ? of_lane(mix.in, min(s, a.S - 1)) : 1.0f;
            const float t[8] = {X[s][0].x, X[s][0].y, X[s][0].z, X[s][0].w, X[s][1].x, X[s][1].y, X[s][1].z, X[s][1].w};
#pragma unroll
            for (int i = 0; i < 8; ++i) u[i] = s < a.S ? fmaf(f, t[i], u[i]) : u[i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) q = fmaf(u[i], u[i], q);
        // a group is whole pieces of 512, or a power of two of lanes
        q = lanes_join_n(q, P / 8, SumOp{});
        if (P > 512) {
            if (lane == 0 && wave == piece) red[piece] = q;
            __syncthreads();
            q = 0.0f;
            for (int c = piece * 512 / P * (P / 512), e = c + P / 512; c < e; ++c) q += red[c];
        }
        const float f = 1.0f / sqrtf(q / (float)P + a.eps);
        const uint32_t g[4] = {nw.x, nw.y, nw.z, nw.w};
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[i] = (uint32_t)f2bf(u[2 * i] * f * __uint_as_float(g[i] << 16)) |
                   ((uint32_t)f2bf(u[2 * i + 1] * f * __uint_as_float(g[i] & 0xFFFF0000u)) << 16);
        if (wave == piece) *reinterpret_cast<uint4*>(xs + px) = make_uint4(o[0], o[1], o[2], o[3]);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CH; ++c) x[c] = *reinterpret_cast<const uint4*>(xs + c * 512 + lane * 8);
    }
    float best = -INFINITY;
    int bi = 0x7fffffff;
    auto step = [&](auto more) {
        const int n = output(unit);
        const StepIn now = e;
        float acc[RW];
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            acc[r] = 0.0f;
#pragma unroll
            for (int c = 0; c < CH; ++c) acc[r] = dot8(w[r][c], x[c], acc[r]);
        }
        if constexpr (decltype(more)::value) {
            operands(unit + ustep);
            wload(unit + ustep);
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int r = 0; r < RW; ++r) acc[r] = wave_sum(acc[r]);
        float v = acc[0];
        if constexpr (UO > 1) {
#pragma unroll
            for (int r = 1; r < RW; ++r) v = lane == r ? acc[r] : v;
        }
        if constexpr (MODE == GR_LOGITS) {
#pragma unroll
            for (int r = 0; r < RW; ++r)
                if (unit * UO + r < a.N && acc[r] > best) { best = acc[r]; bi = unit * UO + r; }
        }
        step_store<uint16_t, MODE, 4>(a, lane < UO && n < a.N, n, 0, v, acc[RW > 1 ? 1 : 0], acc[RW - 1], now, mix);
        unit += ustep;
    };
    while (unit + ustep < nunit) step(std::true_type{});
    if (unit < nunit) step(std::false_type{});
    if constexpr (MODE == GR_LOGITS) {
        __shared__ float sv[4];
        __shared__ int si[4];
        if (lane == 0) { sv[wave] = best; si[wave] = bi; }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int q = 1; q < 4; ++q)
                if (sv[q] > best || (sv[q] == best && si[q] < bi)) { best = sv[q]; bi = si[q]; }
            a.pmax[blockIdx.x] = best;
            a.pidx[blockIdx.x] = bi;
        }
    }
    step_pads<uint16_t, MODE>(a);
}

// The same for the long rows of the output projections (GR_STREAMS) and small products (GR_F32): the four waves of a workgroup
// share a row of 2048 CH, one output per turn.
template <int MODE, int CH>
__global__ void __launch_bounds__(256) k_gemv_long(GemvRtArgs a) {
    __shared__ float part[2][4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k0 = wave * CH * 512 + lane * 8, N = a.N;
    int n = blockIdx.x, turn = 0;
    uint4 w[CH], x[CH];
    const StepMix mix = step_mix<MODE, false>(a);
#pragma unroll
    for (int c = 0; c < CH; ++c) x[c] = ldg16(reinterpret_cast<const uint16_t*>(a.x) + k0 + c * 512);
    auto wload = [&]() {
        const uint16_t* p = a.W + (long)n * a.ldw + k0;
#pragma unroll
        for (int c = 0; c < CH; ++c) w[c] = ldg_nt(p + c * 512);
    };
    wload();
    StepIn e;
    step_load<MODE, 4>(a, n, 0, e);
    asm volatile("" ::: "memory");
    auto step = [&](auto more) {
        const StepIn now = e;
        const int at = n;
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < CH; ++c) acc = dot8(w[c], x[c], acc);
        n += gridDim.x;
        if constexpr (decltype(more)::value) {
            step_load<MODE, 4>(a, n, 0, e);
            wload();
            asm volatile("" ::: "memory");
        }
        acc = wave_sum(acc);
        if (lane == 0) part[turn][wave] = acc;
        __syncthreads();  // (the sums of two turns back are read before the barrier in between)
        if (wave == 0)
            step_store<uint16_t, MODE, 4>(a, lane == 0, at, 0, part[turn][0] + part[turn][1] + part[turn][2] + part[turn][3], 0.0f, 0.0f, now, mix);
        turn ^= 1;
    };
    while (n + (int)gridDim.x < N) step(std::true_type{});
    step(std::false_type{});
}

bool gemv_long_fits(const GemvRtArgs& a, int mode) {
    return a.form == GF_STREAM && a.B == 1 && a.x && a.S <= 4 && (mode == GR_STREAMS || mode == GR_F32) &&
           (a.K == 4096 || a.K == 8192 || a.K == 16384);
}
template <int MODE>
void run_long(hipStream_t s, const GemvRtArgs& a) {
    const dim3 grid(std::min(a.N, a.K >= 16384 ? 512 : 1024)), block(256);
    if (a.K == 4096) hipLaunchKernelGGL((k_gemv_long<MODE, 2>), grid, block, 0, s, a);
    else if (a.K == 8192) hipLaunchKernelGGL((k_gemv_long<MODE, 4>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_gemv_long<MODE, 8>), grid, block, 0, s, a);
}

bool gemv_one_fits(const GemvRtArgs& a, int mode) {
    if (a.form != GF_STREAM || a.B != 1 || a.K % 512 != 0 || a.K > 2048 || a.S > 4) return false;
    if (mode == GR_CONV && a.taps_k > 4) return false;
    if (a.x) return true;
    const int P = a.K / std::max(1, a.groups);
    return (a.S <= 2 || a.K <= 1024) && a.D == a.K && a.groups >= 1 && a.K % a.groups == 0 && (P % 512 == 0 || (512 % P == 0 && P >= 8));
}

template <int MODE, int CH>
void run_one_ch(hipStream_t s, const GemvRtArgs& a, int blocks) {
    if constexpr (MODE == GR_STREAMS) {
        if (a.part) {
            if (a.nsplit <= 8) hipLaunchKernelGGL((k_gemv_one<MODE, CH, -8>), dim3(blocks), dim3(256), 0, s, a);
            else hipLaunchKernelGGL((k_gemv_one<MODE, CH, -16>), dim3(blocks), dim3(256), 0, s, a);
            return;
        }
    }
    if (MODE == GR_STREAMS || a.x) hipLaunchKernelGGL((k_gemv_one<MODE, CH, 0>), dim3(blocks), dim3(256), 0, s, a);
    else if constexpr (MODE != GR_STREAMS) {  // (the update's input is the sublayer's, never the streams)
        if (CH > 2 || a.S <= 2) hipLaunchKernelGGL((k_gemv_one<MODE, CH, 2>), dim3(blocks), dim3(256), 0, s, a);
        else if constexpr (CH <= 2) hipLaunchKernelGGL((k_gemv_one<MODE, CH, 4>), dim3(blocks), dim3(256), 0, s, a);
    }
}
template <int MODE>
void run_one(hipStream_t s, const GemvRtArgs& a) {
    const int blocks = gemv_rt_blocks(a, (GemvRtMode)MODE);
    switch (a.K / 512) {
        case 1: run_one_ch<MODE, 1>(s, a, blocks); break;
        case 2: run_one_ch<MODE, 2>(s, a, blocks); break;
        case 3: run_one_ch<MODE, 3>(s, a, blocks); break;
        default: run_one_ch<MODE, 4>(s, a, blocks); break;
    }
}

int k_split(const GemvRtArgs& a, int mode) { return mode != GR_LOGITS && a.K >= 4096 ? 4 : 1; }

template <typename T, int NB, int MODE, int WK>
void run_wk(hipStream_t s, const GemvRtArgs& a) {
    const dim3 grid(gemv_rt_blocks(a, (GemvRtMode)MODE));
    if (a.x) {
        hipLaunchKernelGGL((k_gemv_rt<T, NB, MODE, WK, true>), grid, dim3(256), 0, s, a);
        return;
    }
    const size_t lds = (size_t)NB * a.K * sizeof(T) + (size_t)(a.D + a.groups) * sizeof(float);
    if (lds > 60 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemv_rt<T, NB, MODE, WK, false>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((k_gemv_rt<T, NB, MODE, WK, false>), grid, dim3(256), lds, s, a);
}

template <typename T, int NB, int MODE>
void run(hipStream_t s, const GemvRtArgs& a) {
    if (MODE != GR_LOGITS && k_split(a, MODE) == 4) run_wk<T, NB, MODE, MODE == GR_LOGITS ? 1 : 4>(s, a);
    else run_wk<T, NB, MODE, 1>(s, a);
}

template <typename T, int NB>
void run_mode(hipStream_t s, GemvRtMode mode, const GemvRtArgs& a) {
    switch (mode) {
        case GR_ACT: run<T, NB, GR_ACT>(s, a); break;
        case GR_CONV: run<T, NB, GR_CONV>(s, a); break;
        case GR_GRU: run<T, NB, GR_GRU>(s, a); break;
        case GR_SWIGLU: run<T, NB, GR_SWIGLU>(s, a); break;
        case GR_STREAMS: run<T, NB, GR_STREAMS>(s, a); break;
        case GR_LOGITS: run<T, NB, GR_LOGITS>(s, a); break;
        case GR_F32: run<T, NB, GR_F32>(s, a); break;
    }
}

// ---------------------------------------------------------------- up to 16 rows: MFMA
// A workgroup owns 16 outputs (of each of the unit's matrices) and all rows; its 4 waves split K.  A lane reads 32
// contiguous bytes of its weight row per 64-deep step (4 lanes: one 128-byte line), so the two MFMAs of a step
// contract k = 16 lg .. 16 lg + 7 and 16 lg + 8 .. 16 lg + 15 of each lane group -- the activations (straight from
// L2, B fragments) use the same order.  After the waves' sums meet in LDS, thread (n, b) runs the step's epilogue.
// GR_F32 with gridDim.y > 1: K is cut over the y workgroups too, out holds their partial slabs [y][B][N].
// LU > 0: by whole lines (k_skinny_lines), up to 8 rows, a wave's steps of a slice being whole turns of LU.
template <typename T, int MODE, int LU = 0>
__global__ void __launch_bounds__(256, sizeof(T) == 4 && MODE != GR_GRU && MODE != GR_SWIGLU ? 4 : 1) k_skinny(GemvRtArgs a) {
    constexpr int NM = MODE == GR_GRU ? 3 : MODE == GR_SWIGLU ? 2 : 1;
    constexpr bool F32 = std::is_same<T, float>::value;
    constexpr int U = NM == 1 && !F32 ? 8 : 4;  // 64-deep steps in flight
    __shared__ float sums[4][NM][16][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4, n0 = blockIdx.x * 16, K = a.K;
    float v[3] = {0.f, 0.f, 0.f};
    const int b = tid & 15, n = n0 + (tid >> 4);
    const int nstep = (K + 63) / 64, per = (nstep + gridDim.y - 1) / gridDim.y, s_end = min(nstep, (int)(blockIdx.y + 1) * per);
    StepIn e;
    step_slot<MODE>(a, min(b, a.B - 1), e);
    if constexpr (!F32) step_load<MODE, 8>(a, n, b, e);  // (fp32: 128 registers are all in use)
    asm volatile("" ::: "memory");
    if constexpr (LU > 0) {
        const int k0 = wave * 64 + (li >> 3) * 32 + lg * 8;  // this lane's 8 of the wave's first step
        const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.x) + (long)min(li & 7, a.B - 1) * a.ldx + k0;
        const uint16_t* wp[NM][2];
        f32x4 acc[NM][2];
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                wp[m][h] = a.W + ((long)m * a.N + min(n0 + h * 8 + (li & 7), a.N - 1)) * a.ldw + k0;
                acc[m][h] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        for (int s0 = blockIdx.y * per; s0 < s_end; s0 += 4 * LU) {
            uint4 w[LU][NM][2], x[LU];
#pragma unroll
            for (int i = 0; i < LU; ++i) {
#pragma unroll
                for (int m = 0; m < NM; ++m)
#pragma unroll
                    for (int h = 0; h < 2; ++h) w[i][m][h] = ldg_nt(wp[m][h] + (s0 + 4 * i) * 64);
                x[i] = ldg16(xp + (s0 + 4 * i) * 64);
            }
            __builtin_amdgcn_sched_barrier(0);  // all in flight: left to itself the compiler keeps six
#pragma unroll
            for (int i = 0; i < LU; ++i)
#pragma unroll
                for (int m = 0; m < NM; ++m)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        acc[m][h] = mfma16(__builtin_bit_cast(short8, w[i][m][h]), __builtin_bit_cast(short8, x[i]), acc[m][h]);
        }
        step_state<MODE>(a, n, e);
        asm volatile("" ::: "memory");
        if ((lg >> 1) == (li >> 3))
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sums[wave][m][8 * h + 4 * (lg & 1) + r][li] = acc[m][h][r];
        __syncthreads();
        if (b < 8)
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int q = 0; q < 4; ++q) v[m] += sums[q][m][tid >> 4][b] + sums[q][m][tid >> 4][b + 8];
    } else {
        const uint16_t* wp[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int n = n0 + li < a.N ? n0 + li : a.N - 1;
            wp[m] = a.W + ((long)m * a.N + n) * a.ldw;
        }
        const T* xp = reinterpret_cast<const T*>(a.x) + (long)(li < a.B ? li : a.B - 1) * a.ldx;
        f32x4 acc[NM], sum[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) sum[m] = acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
        int turn = 0;
        for (int s0 = blockIdx.y * per + wave; s0 < s_end; s0 += 4 * U) {
            uint4 w[U][NM][2];
            typename X8<T>::type x[U][2];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const int k = (s0 + 4 * i) * 64 + lg * 16;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool ok = s0 + 4 * i < s_end && k + 8 * h < K;
#pragma unroll
                    for (int m = 0; m < NM; ++m) w[i][m][h] = ldg16_sel(wp[m] + k + 8 * h, ok, wp[m]);
                    if constexpr (F32) ldx(ok ? xp + k + 8 * h : xp, x[i][h]);  // past the end: the weights are zero
                    else x[i][h].q = ldg16_sel(xp + k + 8 * h, ok, xp);
                }
            }
#pragma unroll
            for (int i = 0; i < U; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if constexpr (F32) {  // tile_f32.h's pieces, the smallest first
                        const F32Pieces q = cut8(x[i][h].a, x[i][h].b);
#pragma unroll
                        for (int p = 2; p >= 0; --p)
#pragma unroll
                            for (int m = 0; m < NM; ++m)
                                acc[m] = mfma16(__builtin_bit_cast(short8, w[i][m][h]), __builtin_bit_cast(short8, q.p[p]), acc[m]);
                    } else {
#pragma unroll
                        for (int m = 0; m < NM; ++m)
                            acc[m] = mfma16(__builtin_bit_cast(short8, w[i][m][h]), __builtin_bit_cast(short8, x[i][h].q), acc[m]);
                    }
                }
            if (F32 && (++turn & 3) == 0) {  // 1024 of k, as tile_f32 (of K = 16384, positive: 3.6e-6 without, an FMA chain 2.0e-6)
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    sum[m] += acc[m];
                    acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
        }
        if constexpr (F32) step_load<MODE, 8>(a, n, b, e);
        step_state<MODE>(a, n, e);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) sums[wave][m][4 * lg + r][li] = F32 ? sum[m][r] + acc[m][r] : acc[m][r];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q) v[m] += sums[q][m][tid >> 4][b];
    }
    if constexpr (F32) {
        // what is not finite (of rows and outputs that there are): FMA chains over this workgroup's K slice, as tile_f32
        __shared__ int flag[4];
        bool bad = false;
#pragma unroll
        for (int m = 0; m < NM; ++m) bad |= b < a.B && n < a.N && not_finite(v[m]);
        const bool wave_bad = __any(bad);
        if (lane == 0) flag[wave] = wave_bad;
        __syncthreads();
        if (flag[0] | flag[1] | flag[2] | flag[3]) {
            constexpr int FK = 32, ST = FK + 1;
            static_assert((1 + NM) * 16 * ST <= 4 * NM * 16 * 17, "the chains' operands fit");
            float *xs = &sums[0][0][0][0], *ws = xs + 16 * ST;  // [row][k], [matrix and output][k]
            float c[NM] = {};
            const int k1 = min(K, s_end * 64);
#pragma clang loop unroll(disable)
            for (int k = blockIdx.y * per * 64; k < k1; k += FK) {
                const int nk = min(FK, k1 - k);
                __syncthreads();
#pragma clang loop unroll(disable)
                for (int i = tid; i < (1 + NM) * 16 * FK; i += 256) {
                    const int r = i / FK, q = i % FK, kk = k + min(q, nk - 1);
                    if (r < 16) xs[r * ST + q] = reinterpret_cast<const float*>(a.x)[(long)min(r, a.B - 1) * a.ldx + kk];
                    else ws[(r - 16) * ST + q] = bf2f(a.W[((long)(r / 16 - 1) * a.N + min(n0 + r % 16, a.N - 1)) * a.ldw + kk]);
                }
                __syncthreads();
#pragma clang loop unroll(disable)
                for (int q0 = 0; q0 < nk; q0 += 8)  // (K is a multiple of 8)
#pragma unroll
                    for (int q = q0; q < q0 + 8; ++q)
#pragma unroll
                        for (int m = 0; m < NM; ++m) c[m] = fmaf(xs[b * ST + q], ws[(m * 16 + (tid >> 4)) * ST + q], c[m]);
            }
#pragma unroll
            for (int m = 0; m < NM; ++m) v[m] = not_finite(v[m]) ? c[m] : v[m];
        }
    }
    if constexpr (MODE == GR_F32) {
        if (b < a.B && n < a.N)
            reinterpret_cast<float*>(a.out)[((long)blockIdx.y * a.B + b) * a.ldo + n] = v[0];
        return;
    }
    step_store<T, MODE, 8>(a, b < a.B && n < a.N, n, b, v[0], v[1], v[2], e, StepMix{});
    step_pads<T, MODE>(a);
}

// The same for bf16 and K up to 2048, the activations held in registers over several groups of 16 outputs per workgroup: what
// a group moves besides its weights is otherwise as many bytes of activations from L2 (8 rows: the output matrix of 257,216 x
// 2048 207 us, held 185; gate|up of 16,384 channels 32.0 / 25.7).  The next group's weights are asked for before this one's
// sums meet, the last group peeled off.  (fp32 rows, three pieces each, would take 200 registers.)
// ST: 64-deep steps of a wave, K / 256 rounded up.  PART: K is less than 256 ST; past it the last step loads the row's first weights,
// made zero where they are used (loads from zeros in memory: gate|up at 2048 26.9 us for 25.1).
template <int MODE, int ST, bool PART>
__global__ void __launch_bounds__(256) k_skinny_held(GemvRtArgs a) {
    constexpr int NM = MODE == GR_SWIGLU ? 2 : 1;
    __shared__ float sums[2][4][NM][16][17];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4, K = a.K, ngroup = (a.N + 15) / 16;
    const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.x) + (long)(li < a.B ? li : a.B - 1) * a.ldx;
    short8 x[ST][2];
#pragma unroll
    for (int i = 0; i < ST; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = (wave + 4 * i) * 64 + lg * 16 + 8 * h;
            x[i][h] = __builtin_bit_cast(short8, ldg16_sel(xp + k, !PART || i + 1 < ST || k < K, xp));
        }
    uint4 w[ST][NM][2];
    int grp = blockIdx.x, turn = 0;
    auto wload = [&]() {
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const uint16_t* p = a.W + ((long)m * a.N + min(grp * 16 + li, a.N - 1)) * a.ldw;
#pragma unroll
            for (int i = 0; i < ST; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int k = (wave + 4 * i) * 64 + lg * 16 + 8 * h;
                    w[i][m][h] = ldg16(p + (!PART || i + 1 < ST || k < K ? k : 0));
                }
        }
    };
    wload();
    auto step = [&](auto more) {
        const int n0 = grp * 16;
        f32x4 acc[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < ST; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    uint4 q = w[i][m][h];
                    if (PART && i + 1 == ST) {
                        const uint32_t keep = (wave + 4 * i) * 64 + lg * 16 + 8 * h < K ? ~0u : 0u;
                        q = make_uint4(q.x & keep, q.y & keep, q.z & keep, q.w & keep);
                    }
                    acc[m] = mfma16(__builtin_bit_cast(short8, q), x[i][h], acc[m]);
                }
        grp += gridDim.x;
        if constexpr (decltype(more)::value) wload();
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) sums[turn][wave][m][4 * lg + r][li] = acc[m][r];
        __syncthreads();  // (the sums of two turns back are read before the barrier in between)
        const int b = tid >> 4, n = n0 + (tid & 15);  // consecutive threads store consecutive outputs
        float v[2] = {0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q) v[m] += sums[turn][q][m][tid & 15][b];
        turn ^= 1;
        if (b >= a.B || n >= a.N) return;
        if constexpr (MODE == GR_F32) reinterpret_cast<float*>(a.out)[(long)b * a.ldo + n] = v[0];
        else step_store<uint16_t, MODE, 8>(a, true, n, b, v[0], v[1], 0.f, StepIn{}, StepMix{});
    };
    while (grp + (int)gridDim.x < ngroup) step(std::true_type{});
    step(std::false_type{});
    step_pads<uint16_t, MODE>(a);
}

// The same for up to 8 rows and K of 256 ST, by whole lines: 8 outputs and two halves of each 64-deep step are the 16 rows of one
// matrix operand, the 8 rows of activations and the same halves the 16 of the other, so a load instruction reads 8 rows by 128
// bytes, each line once and by one instruction (16 rows by half of a line, twice, need the cache between them, and are slower
// uncached).  Of the product's quarters the two of unlike halves are not used, the two others added.  8 rows, output matrix of 257,216 x
// 2,048 182 -> 172 us, 3 rows 187 -> 158; 256 to 1,280 workgroups measured equal.
template <int MODE, int ST>
__global__ void __launch_bounds__(256) k_skinny_lines(GemvRtArgs a) {
    constexpr int NM = MODE == GR_SWIGLU ? 2 : 1;
    __shared__ float sums[2][4][NM][16][17];  // [.][wave][matrix][output][half and row]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4, ngroup = (a.N + 15) / 16;
    const int k0 = wave * 64 + (li >> 3) * 32 + lg * 8;  // this lane's 8 of the wave's first step
    const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.x) + (long)min(li & 7, a.B - 1) * a.ldx + k0;
    short8 x[ST];
#pragma unroll
    for (int i = 0; i < ST; ++i) x[i] = __builtin_bit_cast(short8, ldg16(xp + i * 256));
    uint4 w[NM][2][ST];
    int grp = blockIdx.x, turn = 0;
    auto wload = [&]() {
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint16_t* p = a.W + ((long)m * a.N + min(grp * 16 + h * 8 + (li & 7), a.N - 1)) * a.ldw + k0;
#pragma unroll
                for (int i = 0; i < ST; ++i) w[m][h][i] = ldg_nt(p + i * 256);
            }
    };
    wload();
    auto step = [&](auto more) {
        const int n0 = grp * 16;
        f32x4 acc[NM][2];
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                acc[m][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < ST; ++i) acc[m][h] = mfma16(__builtin_bit_cast(short8, w[m][h][i]), x[i], acc[m][h]);
            }
        grp += gridDim.x;
        if constexpr (decltype(more)::value) wload();
        // lane: products of operand rows 4 lg .. (output % 8, half lg / 2) with column li (row % 8, half li / 8)
        if ((lg >> 1) == (li >> 3))
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sums[turn][wave][m][8 * h + 4 * (lg & 1) + r][li] = acc[m][h][r];
        __syncthreads();  // (the sums of two turns back are read before the barrier in between)
        const int b = tid >> 4, n = n0 + (tid & 15);  // consecutive threads store consecutive outputs
        float v[2] = {0.f, 0.f};
        if (b < 8)
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int q = 0; q < 4; ++q) v[m] += sums[turn][q][m][tid & 15][b] + sums[turn][q][m][tid & 15][b + 8];
        turn ^= 1;
        if (b >= a.B || n >= a.N) return;
        if constexpr (MODE == GR_F32) reinterpret_cast<float*>(a.out)[(long)b * a.ldo + n] = v[0];
        else step_store<uint16_t, MODE, 8>(a, true, n, b, v[0], v[1], 0.f, StepIn{}, StepMix{});
    };
    while (grp + (int)gridDim.x < ngroup) step(std::true_type{});
    step(std::false_type{});
    step_pads<uint16_t, MODE>(a);
}

template <int ST>
void run_lines(hipStream_t s, GemvRtMode mode, const GemvRtArgs& a, int blocks) {
    if (mode == GR_SWIGLU) hipLaunchKernelGGL((k_skinny_lines<GR_SWIGLU, ST>), dim3(blocks), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_skinny_lines<GR_F32, ST>), dim3(blocks), dim3(256), 0, s, a);
}

template <int ST, bool PART = true>
void run_held(hipStream_t s, GemvRtMode mode, const GemvRtArgs& a, int blocks) {
    if (PART && a.K % 256 == 0) return run_held<ST, false>(s, mode, a, blocks);
    if (mode == GR_SWIGLU) hipLaunchKernelGGL((k_skinny_held<GR_SWIGLU, ST, PART>), dim3(blocks), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_skinny_held<GR_F32, ST, PART>), dim3(blocks), dim3(256), 0, s, a);
}

template <typename T>
void run_skinny(hipStream_t s, GemvRtMode mode, const GemvRtArgs& a) {
    const dim3 grid((a.N + 15) / 16), block(256);
    constexpr int kHeldBlocks = 512;  // two per CU: 256, 512 and 768 measured equal, 1,024 and more slower
    // The held form pays from 512 inputs on.  us a step of four layers and the output matrix, plain / held: gate|up of 16,384 at width 320
    // 128 / 129 (2 rows), 135 / 136 (8), at 512 143 / 140 and 149 / 145, at 1,024 188 / 180 and 203 / 188, at 2,048 289 / 270 and 311 /
    // 285; 65,536 outputs at 512 122 / 117 and 130 / 122, at 1,000 137 / 137 and 143 / 142, at 2,048 181 / 178 and 195 / 186
    const bool pays = a.K >= 512 && (mode == GR_SWIGLU || mode == GR_F32 || mode == GR_LOGITS);
    if (std::is_same<T, uint16_t>::value && pays && a.K <= 2048 && a.split <= 1 && (int)grid.x > kHeldBlocks) {
        if (a.B <= 8 && a.K % 256 == 0) {
            switch (a.K / 256) {
                case 2: run_lines<2>(s, mode, a, kHeldBlocks); return;
                case 3: run_lines<3>(s, mode, a, kHeldBlocks); return;
                case 4: run_lines<4>(s, mode, a, kHeldBlocks); return;
                case 5: run_lines<5>(s, mode, a, kHeldBlocks); return;
                case 6: run_lines<6>(s, mode, a, kHeldBlocks); return;
                case 7: run_lines<7>(s, mode, a, kHeldBlocks); return;
                default: run_lines<8>(s, mode, a, kHeldBlocks); return;
            }
        }
        switch ((a.K + 255) / 256) {
            case 2: run_held<2>(s, mode, a, kHeldBlocks); break;
            case 3: run_held<3>(s, mode, a, kHeldBlocks); break;
            case 4: run_held<4>(s, mode, a, kHeldBlocks); break;
            case 5: run_held<5>(s, mode, a, kHeldBlocks); break;
            case 6: run_held<6>(s, mode, a, kHeldBlocks); break;
            case 7: run_held<7>(s, mode, a, kHeldBlocks); break;
            default: run_held<8>(s, mode, a, kHeldBlocks); break;
        }
        return;
    }
    // By whole lines: turns of 8 steps a wave (of several matrices 4), of short rows fewer.  us a step of the 2,048-wide streams model,
    // 2 and 8 rows: 801 -> 761, 867 -> 816.  Matrices under 4 MB, whose time is not their bytes', as before (1,536 outputs of
    // K = 1,024: a step of 8 layers 408 -> 411)
    int turn = 0;
    const int nm = mode == GR_GRU ? 3 : mode == GR_SWIGLU ? 2 : 1;
    if (std::is_same<T, uint16_t>::value && a.B <= 8 && a.K % (64 * std::max(1, a.split)) == 0 && (long)nm * a.N * a.K >= 2 << 20) {
        const int steps = a.K / 64 / std::max(1, a.split);  // of a slice, dealt to four waves
        for (int u = nm > 1 ? 4 : 8; u >= 2 && !turn; u /= 2)
            if (steps % (4 * u) == 0) turn = u;
    }
    auto go = [&](auto mode_c, dim3 g) {
        constexpr int MODE = decltype(mode_c)::value;
        if constexpr (std::is_same<T, uint16_t>::value) {
            if constexpr (MODE != GR_GRU && MODE != GR_SWIGLU)
                if (turn == 8) { hipLaunchKernelGGL((k_skinny<T, MODE, 8>), g, block, 0, s, a); return; }
            if (turn == 4) { hipLaunchKernelGGL((k_skinny<T, MODE, 4>), g, block, 0, s, a); return; }
            if (turn == 2) { hipLaunchKernelGGL((k_skinny<T, MODE, 2>), g, block, 0, s, a); return; }
        }
        hipLaunchKernelGGL((k_skinny<T, MODE>), g, block, 0, s, a);
    };
    assert(mode != GR_STREAMS);  // output projections in this form leave slabs (GR_F32), which the next streams pass joins
    switch (mode) {
        case GR_ACT: go(std::integral_constant<int, GR_ACT>{}, grid); break;
        case GR_CONV: go(std::integral_constant<int, GR_CONV>{}, grid); break;
        case GR_GRU: go(std::integral_constant<int, GR_GRU>{}, grid); break;
        case GR_SWIGLU: go(std::integral_constant<int, GR_SWIGLU>{}, grid); break;
        default: go(std::integral_constant<int, GR_F32>{}, dim3(grid.x, a.split < 1 ? 1 : a.split)); break;
    }
}

// ---------------------------------------------------------------- convolution step
template <typename T>
__global__ void __launch_bounds__(256) k_conv_step(const T* __restrict__ xz, int ldxz, int C, int K,
                                                   const uint16_t* __restrict__ w, const uint16_t* __restrict__ cb,
                                                   float* __restrict__ taps, const int* __restrict__ slot,
                                                   const int* __restrict__ pos, T* __restrict__ out, int ldo) {
    const int b = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    if (c >= ldo) return;
    float y = 0.0f;
    if (c < C) {
        float* tp = taps + (long)slot[b] * (K - 1) * C + c;
        const bool first = pos[b] == 0;
        const float v = ldf(xz + (long)b * ldxz + c);
        y = fmaf(bf2f(w[(long)c * K + K - 1]), v, bf2f(cb[c]));
        for (int j = 0; j < K - 1; ++j) {
            const float o = first ? 0.0f : tp[(long)j * C];
            y = fmaf(bf2f(w[(long)c * K + j]), o, y);
            if (j > 0) tp[(long)(j - 1) * C] = o;
        }
        if (K > 1) tp[(long)(K - 2) * C] = v;
        y = siluf_(y);
    }
    stf(out + (long)b * ldo + c, y);
}

// ---------------------------------------------------------------- selective-scan step
// LPC lanes per channel: they share the dt dot product over R and hold the channel's states.  What bounds it is latency: everything
// that does not hang on the projection's sums (the first AHEAD pieces of a channel's row of Wdt, the first AHEAD states of a lane
// and their A) is asked for together, ahead of them; read where it is used it was eight trips to memory, one behind the other (2,048
// channels of 16 states: 4.1 -> 3.2 us)
template <typename T, int LPC>
__global__ void __launch_bounds__(256) k_scan_step(ScanStepArgs a) {
    extern __shared__ __attribute__((aligned(16))) float sm[];  // [R + 2N] of this sequence, read to whole 8 of R
    constexpr int CPB = 256 / LPC, AHEAD = 2, SLABS = 4;
    const int b = blockIdx.y, tid = threadIdx.x, sub = tid % LPC;
    const int M = a.R + 2 * a.N;
    const int c = blockIdx.x * CPB + tid / LPC;
    const bool ok = c < a.C;
    const int cc = ok ? c : a.C - 1;
    int row = b;
    asm volatile("" : "+v"(row));  // (by vector loads: scalar ones would be waited for with the arguments)
    const int slot = a.slot[row], pos = a.pos[row];
    const uint16_t* wd = a.Wdt + (long)cc * a.ldwdt;  // rows of Wdt are 16-byte aligned, zero past R
    const uint16_t* Al = a.A_log + (long)cc * a.N;
    float part[SLABS];  // the sums' first slabs
    const float* slab = a.slabs + (long)b * M + min(tid, M - 1);
#pragma unroll
    for (int z = 0; z < SLABS; ++z) part[z] = slab[(long)min(z, a.split - 1) * a.B * M];
    uint4 wq[AHEAD];
    uint16_t aq[AHEAD];
    float sq[AHEAD];
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
        const int r = (q * LPC + sub) * 8;
        wq[q] = ldg16(wd + (r < a.R ? r : 0));
        aq[q] = Al[min(q * LPC + sub, a.N - 1)];
    }
    const uint16_t dtb = a.dtb[cc], Dw = a.Dw[cc];
    const float x = ldf(reinterpret_cast<const T*>(a.x) + (long)b * a.ldx + cc);
    const float gate = ldf(reinterpret_cast<const T*>(a.z) + (long)b * a.ldz + cc);
    float* st = a.state + ((long)slot * a.C + cc) * a.N;
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) sq[q] = st[min(q * LPC + sub, a.N - 1)];
    asm volatile("" ::: "memory");
    for (int i = tid; i < M; i += 256) {
        float v = 0.0f;
        if (i == tid) {
#pragma unroll
            for (int z = 0; z < SLABS; ++z) v += z < a.split ? part[z] : 0.0f;
        }
        for (int z = i == tid ? SLABS : 0; z < a.split; ++z) v += a.slabs[((long)z * a.B + b) * M + i];
        sm[i] = v;
    }
    __syncthreads();
    float dt = 0.0f;
    auto dot = [&](const uint4 w, int r) {
        const uint32_t h[4] = {w.x, w.y, w.z, w.w};
        const float* p = sm + (r < a.R ? r : 0);
        const f32x4 lo = *reinterpret_cast<const f32x4*>(p), hi = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const float f = fmaf(__uint_as_float(v & 1 ? h[v / 2] & 0xFFFF0000u : h[v / 2] << 16), v < 4 ? lo[v % 4] : hi[v % 4], dt);
            dt = r + v < a.R ? f : dt;
        }
    };
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) dot(wq[q], (q * LPC + sub) * 8);
    for (int r = (AHEAD * LPC + sub) * 8; r < a.R; r += LPC * 8) dot(ldg16(wd + r), r);
    dt = lanes_join<LPC>(dt, SumOp{});
    dt = softplusf_(dt + bf2f(dtb));
    const float dx = dt * x;
    const float* B = sm + a.R;
    const float* Cv = B + a.N;
    float y = 0.0f;
    auto state = [&](int n, uint16_t al, float old, float bn, float cn) {
        const float A = -expf(bf2f(al)) * 1.4426950408889634f;
        const float S = fmaf(__builtin_amdgcn_exp2f(dt * A), pos == 0 ? 0.0f : old, dx * bn);
        if (ok && n < a.N) st[n] = S;
        y = n < a.N ? fmaf(S, cn, y) : y;
    };
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) {
        const int n = q * LPC + sub, in = min(n, a.N - 1);
        state(n, aq[q], sq[q], B[in], Cv[in]);
    }
    for (int n = AHEAD * LPC + sub; n < a.N; n += LPC) state(n, Al[n], st[n], B[n], Cv[n]);
    y = lanes_join<LPC>(y, SumOp{});
    if (sub == 0 && c < a.ldy) {
        y = fmaf(bf2f(Dw), x, y);
        stf(reinterpret_cast<T*>(a.y) + (long)b * a.ldy + c, ok ? y * siluf_(gate) : 0.0f);
    }
}

template <typename T>
void scan_step_t(hipStream_t s, const ScanStepArgs& a) {
    const size_t lds = (size_t)((a.R + 7) / 8 * 8 + 2 * a.N) * sizeof(float);
    const int cols = std::max(a.C, a.ldy);
    if (a.N <= 16) hipLaunchKernelGGL((k_scan_step<T, 8>), dim3((cols + 31) / 32, a.B), dim3(256), lds, s, a);
    else hipLaunchKernelGGL((k_scan_step<T, 16>), dim3((cols + 15) / 16, a.B), dim3(256), lds, s, a);
}

// ---------------------------------------------------------------- minGRU step
template <typename T>
__global__ void __launch_bounds__(256) k_gru_step(const T* __restrict__ zug, int ld, int C, float* __restrict__ state,
                                                  const int* __restrict__ slot, const int* __restrict__ pos,
                                                  T* __restrict__ y, int ldy) {
    const int b = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
    if (c >= ldy) return;
    float v = 0.0f;
    if (c < C) {
        const T* r = zug + (long)b * ld + c;
        float* st = state + (long)slot[b] * C + c;
        const float z = sigmoidf_(ldf(r));
        const float S = fmaf(1.0f - z, pos[b] > 0 ? *st : 0.0f, z * gru_candidate(ldf(r + C)));
        *st = S;
        v = S * siluf_(ldf(r + 2 * C));
    }
    stf(y + (long)b * ldy + c, v);
}

// ---------------------------------------------------------------- end of a step
__global__ void __launch_bounds__(256) k_decode_finish(const float* __restrict__ pmax, const int* __restrict__ pidx,
                                                       int nparts, int64_t* __restrict__ next, int64_t* __restrict__ hist,
                                                       int* __restrict__ pos) {
    const int b = blockIdx.x, tid = threadIdx.x;
    __shared__ float sv[256];
    __shared__ int si[256];
    if (nparts > 0) {
        float best = -INFINITY;
        int bi = 0x7fffffff;
        for (int i = tid; i < nparts; i += 256) {
            const float v = pmax[(long)b * nparts + i];
            const int ix = pidx[(long)b * nparts + i];
            if (v > best || (v == best && ix < bi)) { best = v; bi = ix; }
        }
        sv[tid] = best;
        si[tid] = bi;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o && (sv[tid + o] > sv[tid] || (sv[tid + o] == sv[tid] && si[tid + o] < si[tid]))) {
                sv[tid] = sv[tid + o];
                si[tid] = si[tid + o];
            }
            __syncthreads();
        }
        // no finite logit: token 0 rather than an index out of the table
        if (tid == 0) next[b] = si[0] == 0x7fffffff ? 0 : si[0];
    }
    if (tid == 0) {
        if (hist) hist[b] = next[b];
        pos[b] += 1;
    }
}

}  // namespace

int gemv_rt_max_batch() { return 16; }
int gemv_rt_parts() { return 2 * 1024; }
GemvRtForm gemv_rt_form(int B, Act act, int streams, int width) {
    // fp32 activations: two rows.  bf16: one row, while every workgroup's own read of the streams stays small.  ms a step, this form /
    // the MFMA form: 2 streams of 1024 0.293 / 0.427, 4 of 1024 0.326 / 0.459, 2 of 2048 0.639 / 0.821, 2 of 4096 0.812 / 0.664.  Streams
    // times width is not all of it: 3 of 2048 (0.668 / 0.843) and 1 of 4096 (0.770 / 0.656) lie on the side that is slower for them
    if (act == ACT_F32 && B <= 2) return GF_STREAM;
    if (act == ACT_BF16 && B == 1 && streams * width <= 4096) return GF_STREAM;
    return B <= gemv_rt_max_batch() ? GF_SKINNY : GF_NONE;
}

bool gemv_rt_fits(GemvRtForm form, int K, Act act) {
    if (form == GF_STREAM) return (size_t)2 * K * (act == ACT_F32 ? 4 : 2) <= 96 * 1024;
    return form == GF_SKINNY;
}

bool gemv_rt_merges(const GemvRtArgs& a) {
    return a.act == ACT_BF16 && a.x && gemv_one_fits(a, GR_STREAMS) && a.nsplit <= 16 && a.pe % 8 == 0 && a.K % a.pe == 0 &&
           a.prs % 2 == 0;
}

int gemv_rt_split(GemvRtForm form, int N, int K) {
    if (form != GF_SKINNY) return 1;
    const int tiles = (N + 15) / 16, nstep = (K + 63) / 64;
    int split = 1;
    while (split < 8 && tiles * split < 512 && nstep / (split * 2) >= 4) split *= 2;
    const int per = (nstep + split - 1) / split;  // no empty slice
    return (nstep + per - 1) / per;
}

int gemv_rt_blocks(const GemvRtArgs& a, GemvRtMode mode) {
    if (a.act == ACT_BF16 && gemv_one_fits(a, mode)) {
        const int units = (a.N + one_outs(mode) - 1) / one_outs(mode);
        return std::max(1, std::min((units + 3) / 4, mode == GR_LOGITS ? 2048 : 1024));
    }
    const int units = (a.N + unit_outs(mode) - 1) / unit_outs(mode), upb = 4 / k_split(a, mode);
    return std::max(1, std::min((units + upb - 1) / upb, 1024));
}

void gemv_rt(hipStream_t s, Act act, GemvRtMode mode, const GemvRtArgs& a) {
    if (act == ACT_BF16 && gemv_one_fits(a, mode)) {
        switch (mode) {
            case GR_ACT: run_one<GR_ACT>(s, a); break;
            case GR_CONV: run_one<GR_CONV>(s, a); break;
            case GR_GRU: run_one<GR_GRU>(s, a); break;
            case GR_SWIGLU: run_one<GR_SWIGLU>(s, a); break;
            case GR_STREAMS: run_one<GR_STREAMS>(s, a); break;
            case GR_LOGITS: run_one<GR_LOGITS>(s, a); break;
            case GR_F32: run_one<GR_F32>(s, a); break;
        }
        return;
    }
    if (act == ACT_BF16 && gemv_long_fits(a, mode)) {
        if (mode == GR_STREAMS) run_long<GR_STREAMS>(s, a);
        else run_long<GR_F32>(s, a);
        return;
    }
    if (a.form == GF_SKINNY && act == ACT_BF16) run_skinny<uint16_t>(s, mode, a);
    else if (a.form == GF_SKINNY) run_skinny<float>(s, mode, a);
    else if (act == ACT_BF16) run_mode<uint16_t, 1>(s, mode, a);
    else if (a.B <= 1) run_mode<float, 1>(s, mode, a);
    else run_mode<float, 2>(s, mode, a);
}

void conv_step(hipStream_t s, Act act, const void* xz, int ldxz, int B, int C, int K, const uint16_t* w,
               const uint16_t* b, float* taps, const int* slot, const int* pos, void* out, int ldo) {
    const dim3 grid((ldo + 255) / 256, B);
    if (act == ACT_F32)
        hipLaunchKernelGGL((k_conv_step<float>), grid, dim3(256), 0, s, reinterpret_cast<const float*>(xz), ldxz, C, K, w,
                           b, taps, slot, pos, reinterpret_cast<float*>(out), ldo);
    else
        hipLaunchKernelGGL((k_conv_step<uint16_t>), grid, dim3(256), 0, s, reinterpret_cast<const uint16_t*>(xz), ldxz, C,
                           K, w, b, taps, slot, pos, reinterpret_cast<uint16_t*>(out), ldo);
}

void scan_step(hipStream_t s, Act act, const ScanStepArgs& a) {
    if (act == ACT_F32) scan_step_t<float>(s, a);
    else scan_step_t<uint16_t>(s, a);
}

void gru_step(hipStream_t s, Act act, const void* zug, int ld, int B, int C, float* state, const int* slot,
              const int* pos, void* y, int ldy) {
    const dim3 grid((ldy + 255) / 256, B);
    if (act == ACT_F32)
        hipLaunchKernelGGL((k_gru_step<float>), grid, dim3(256), 0, s, reinterpret_cast<const float*>(zug), ld, C, state,
                           slot, pos, reinterpret_cast<float*>(y), ldy);
    else
        hipLaunchKernelGGL((k_gru_step<uint16_t>), grid, dim3(256), 0, s, reinterpret_cast<const uint16_t*>(zug), ld, C,
                           state, slot, pos, reinterpret_cast<uint16_t*>(y), ldy);
}

void decode_finish(hipStream_t s, int B, const float* pmax, const int* pidx, int nparts, int64_t* next, int64_t* hist,
                   int* pos) {
    hipLaunchKernelGGL(k_decode_finish, dim3(B), dim3(256), 0, s, pmax, pidx, nparts, next, hist, pos);
}

}  // namespace pgmi
