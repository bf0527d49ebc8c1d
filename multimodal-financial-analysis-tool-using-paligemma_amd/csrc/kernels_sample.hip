// kernels_sample.hip -- temperature softmax + top-p (nucleus) sampling on the device
// (inference.py:15-24 _sample_top_p, with the softmax(logits / T) of :65).
//
// The reference sorts all 257,216 probabilities, takes the cumulative sum, zeroes every entry
// whose preceding mass already exceeds p, renormalises and draws with torch.multinomial.  The
// kept tokens are a prefix of the descending order, so both decisions are "the first sorted
// position whose inclusive cumulative mass exceeds a target": target p gives the nucleus
// cut-off k*, and target r = u * Z (Z = the kept mass, u ~ U[0,1) from the caller) gives the
// draw, which lands at or before k* because r < Z.  Each is a mass-weighted radix select over
// the fp32 bit patterns (probabilities are >= 0, so the bit order is the value order): the exponent
// field by the row's histogram, then three digits of the mantissa over the tokens of that exponent,
// walking bins from the top until the running mass crosses the target, then equal probabilities
// resolved in index order (our tie rule; torch.sort does not define one).  No sort and no materialised
// cumsum; masses in fp64.
//
// Four launches, each a short dependent chain; what bounds a draw is their length and number, not the
// vocabulary's megabyte.  257,216 logits of a peaked distribution: 42 us as five launches with four digits
// per select, maxima by LDS atomics (a turn per lane) and a select for the token after the cut-off at every draw, later 21.2, 19.6 since
// the masses of bins and the places of candidates are scanned by the vector unit's lane moves (common.h) and not through LDS, 18.7 with
// the slices' statistics and the candidates' tokens asked for ahead.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace pgmi {

constexpr int kSampleThreads = 1024;
// probability masses are summed as 2^-62 fixed point in u64: native integer LDS atomics (fp64
// atomics lower to CAS loops), order-independent and therefore deterministic sums; a row's total
// (<= 1 + rounding) stays below 2^63, and a single probability loses < 2^-62 to truncation
constexpr double kMassScale = 4611686018427387904.0;  // 2^62
constexpr double kMassUnit = 1.0 / kMassScale;
__device__ __forceinline__ unsigned long long mass_q(float v) { return (unsigned long long)((double)v * kMassScale); }

struct SelectOut {
    uint32_t key;  // bit pattern of the probability at the crossing position
    double mass;   // inclusive mass at the crossing
    int rank;      // it is the rank-th (index order, 0-based) token equal to key; ranked candidates: its place among them
    bool crossed;  // false: target >= the total mass (no crossing)
};

constexpr int kHeld = 2048;   // candidates that k_tp_select holds in LDS
constexpr int kRanked = 256;  // and those it orders by comparing each with all
constexpr int kDigit = 6;     // bits of the mantissa per level: a wave holds a level's bins
constexpr int kLevels = 4;
struct SampleSmem {
    float val[kHeld];
    unsigned hcnt[kLevels][64];
    unsigned long long hmq[kLevels][64];
    double row_suf[256 + 4];  // the row's suffix masses by exponent
    int top[2][4];            // per wave
    int scan[kSampleThreads / 64];
    int found;
    // the ranked candidates in descending order: value, inclusive mass, place
    float ord_val[kRanked];
    double ord_mass[kRanked];
    int ord_at[kRanked];
    int token[kRanked];  // of the first candidates
};

// suf[t] = mass of bins t .. 255 (mq in fixed point), t < 256: a wave scans its 64 bins from the highest down, then the higher
// waves' totals in a fixed order.  Every thread of the block must call it (suf: 260 doubles).
__device__ __forceinline__ void suffix_masses(const unsigned long long* mq, double* suf) {
    const int t = threadIdx.x, w = t >> 6, bin = t ^ 63;
    double v = 0.0;
    if (t < 256) {
        v = wave_scan((double)mq[bin] * kMassUnit);
        if ((t & 63) == 63) suf[256 + w] = v;  // the wave's total
    }
    __syncthreads();
    if (t < 256) {
        const double total[4] = {0.0, suf[257], suf[258], suf[259]};  // (read together)
#pragma unroll
        for (int q = 1; q < 4; ++q) v = q > w ? v + total[q] : v;
        suf[bin] = v;
    }
    __syncthreads();
}

// The largest t < 256 of the block's first four waves for which `is` holds, -1 if none: by ballots (a maximum by LDS atomics
// costs a turn for every lane that takes part).  Two barriers; every thread of the block calls it.
__device__ __forceinline__ int highest(bool is, int* top) {
    const unsigned long long m = __ballot(is);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if (w < 4 && (threadIdx.x & 63) == 0) top[w] = m ? 64 * w + 63 - __clzll((long long)m) : -1;
    __syncthreads();
    return max(max(top[0], top[1]), max(top[2], top[3]));
}

// The smallest such t, -1 if none; the block is its first four waves.  One barrier: calls in turn take turns with two tops.
__device__ __forceinline__ int lowest(bool is, int* top) {
    const unsigned long long m = __ballot(is);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) top[w] = m ? 64 * w + __ffsll((long long)m) - 1 : 256;
    __syncthreads();
    const int t = min(min(top[0], top[1]), min(top[2], top[3]));
    return t < 256 ? t : -1;
}

__device__ __forceinline__ void hist_add(unsigned* hcnt, unsigned long long* hmq, bool valid, int d, float v) {
    if (valid) {
        atomicAdd(&hcnt[d], 1u);
        atomicAdd(&hmq[d], mass_q(v));
    }
}

// The first position of the descending order whose inclusive cumulative mass exceeds target, found digit by digit of the
// mantissa among the candidates of its exponent.  value(i): candidate i of n; used: the row has tokens of exponent threadIdx.x.
template <typename Value>
__device__ __forceinline__ SelectOut radix_select(const Value& value, int n, int NT, double target, bool used, SampleSmem& sm) {
    const int t = threadIdx.x, lane = t & 63;
    __syncthreads();  // the previous select's readers are done
    for (int i = t; i < kLevels * 64; i += NT) {  // (behind highest()'s barriers for its users)
        (&sm.hcnt[0][0])[i] = 0u;
        (&sm.hmq[0][0])[i] = 0ull;
    }
    const int bin = highest(t < 256 && used && sm.row_suf[t & 255] > target, sm.top[0]);
    if (bin < 0) return SelectOut{0u, 0.0, 0, false};
    uint32_t prefix = (uint32_t)bin << 23, pmask = 0xFF800000u;
    double above = bin < 255 ? sm.row_suf[bin + 1] : 0.0;
#pragma unroll 1
    for (int level = 0; level < kLevels; ++level) {
        const int shift = max(0, 23 - kDigit * (level + 1)), bits = level + 1 < kLevels ? kDigit : 23 - kDigit * (kLevels - 1);
        const uint32_t digit = (1u << bits) - 1u;
#pragma unroll 1
        for (int i = t; i < n; i += NT) {
            const float v = value(i);
            const uint32_t k = __float_as_uint(v);
            hist_add(sm.hcnt[level], sm.hmq[level], (k & pmask) == prefix, (int)((k >> shift) & digit), v);
        }
        __syncthreads();
        // every wave, its lanes from the highest bin down: mass of the bin and those above, then the LARGEST bin whose mass
        // crosses (sums are monotone up to rounding; taking the largest keeps the answer unique)
        const unsigned long long own = sm.hmq[level][63 - lane], suf = wave_scan(own);
        const unsigned long long m = __ballot(sm.hcnt[level][63 - lane] != 0u && above + (double)suf * kMassUnit > target);
        if (!m) return SelectOut{0u, 0.0, 0, false};
        const int at = __ffsll((long long)m) - 1, d = 63 - at;
        above += (double)(unsigned long long)__shfl(suf - own, at, 64) * kMassUnit;
        prefix |= (uint32_t)d << shift;
        pmask |= digit << shift;
    }
    // tokens equal to the key: the crossing is at the smallest tie rank j with
    // above + (j + 1) * value > target
    const double val = (double)__uint_as_float(prefix);
    int rank = 0;
    if (val > 0.0) {
        double need = floor((target - above) / val);
        rank = need < 0.0 ? 0 : (need > 2e9 ? 2000000000 : (int)need);
        while (rank > 0 && above + (double)rank * val > target) --rank;
        while (!(above + (double)(rank + 1) * val > target)) ++rank;
    }
    return SelectOut{prefix, above + (double)(rank + 1) * val, rank, true};
}

// place of the rank-th candidate (index order) whose bit pattern equals key; -1 if fewer exist
template <typename Value>
__device__ __forceinline__ int nth_equal(const Value& value, int n, int NT, uint32_t key, int rank, SampleSmem& sm) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per = (n + NT - 1) / NT, i0 = min((int)threadIdx.x * per, n), i1 = min(i0 + per, n);  // contiguous slice per thread
    int c = 0;
#pragma unroll 1
    for (int i = i0; i < i1; ++i) c += (__float_as_uint(value(i)) == key);
    // exclusive prefix of the threads' counts: within the wave, then wave totals
    const int incl = wave_scan(c);
    __syncthreads();
    if (lane == 63) sm.scan[wave] = incl;
    if (threadIdx.x == 0) sm.found = -1;
    __syncthreads();
    int at = incl - c;
    for (int w = 0; w < wave; ++w) at += sm.scan[w];
    if (rank >= at && rank < at + c) {
#pragma unroll 1
        for (int i = i0; i < i1; ++i)
            if (__float_as_uint(value(i)) == key && at++ == rank) sm.found = i;
    }
    __syncthreads();
    return sm.found;
}

// ---------------------------------------------------------------- the multi-kernel pipeline
// Per row: (1) k_tp_stats, NB blocks: max and sum of exp of z = x / T per slice;
// (2) k_tp_hist, NB blocks: p = softmax, written once, per-block counts and the row's histogram of the fp32
// exponent field (256 bins of count and fixed-point mass);
// (3) k_tp_compact, NB blocks: from that histogram, each for itself, the cut-off bin c1 (where the running mass
// crosses p) and the highest bin c_hi the draw can reach (r = u Z >= u * mass above c1), so every position the
// two decisions can land on lies in bins [c1, c_hi]; then the tokens of these bins -> (value, index) in index
// order;
// (4) k_tp_select, one block: the two radix selects of the header over the candidates only.
constexpr int kTpThreads = 256;
constexpr int kShards = 8;  // copies of the row's histogram: blocks adding to one address wait for each other
constexpr int kTpHeld = 2048;  // tokens of a slice (tp_blocks) that a block holds in registers

struct TpLayout {
    size_t p, cv, ci, bm, bs, hc, hm, meta, stride;  // byte offsets within one row's scratch
};

inline size_t tp_align(size_t x) { return (x + 255) & ~(size_t)255; }

inline TpLayout tp_layout(int V, int NB) {
    TpLayout L;
    size_t o = 0;
    L.p = o; o = tp_align(o + (size_t)V * 4);
    L.cv = o; o = tp_align(o + (size_t)V * 4);
    L.ci = o; o = tp_align(o + (size_t)V * 4);
    L.bm = o; o = tp_align(o + (size_t)NB * 4);
    L.bs = o; o = tp_align(o + (size_t)NB * 8);
    L.hc = o; o = tp_align(o + (size_t)NB * 256 * 2);
    L.hm = o; o = tp_align(o + (size_t)kShards * 256 * 8);
    L.meta = o; o = tp_align(o + 16 * 8);
    // (no less than 1 KiB and 8 bytes per block: the workspace holds the same vocabularies whatever the histograms' layout)
    L.stride = std::max(o, L.hc + tp_align((size_t)NB * 1024) + 1024 + 2048 + tp_align((size_t)NB * 4) + 256);
    return L;
}

struct TpMeta {  // one row's plan (k_tp_compact -> k_tp_select)
    double a1;     // mass of the bins above c1
    double total;  // mass of the row
    int c1, c_hi;  // candidate bins [c1, c_hi]
    int n_cand;
    int crossed;   // the cut-off exists (p < total mass)
};

__device__ __forceinline__ int tp_bin(float v) { return (int)((__float_as_uint(v) >> 23) & 255u); }

__device__ __forceinline__ void tp_slice(int V, int NB, int b, int& i0, int& i1) {
    const int per = (V + NB - 1) / NB;
    i0 = b * per;
    i1 = min(V, i0 + per);
}

__global__ void __launch_bounds__(kTpThreads) k_tp_stats(const float* __restrict__ x, int V, float temperature,
                                                          int NB, uint8_t* __restrict__ scratch, TpLayout L) {
    __shared__ float red_f[kTpThreads / 64];
    __shared__ double red_d[kTpThreads / 64];
    const int b = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
    const float* xr = x + (long)row * V;
    uint8_t* base = scratch + (size_t)row * L.stride;
    int i0, i1;
    tp_slice(V, NB, b, i0, i1);
    // the slice's first kTpHeld tokens stay in registers between the two passes
    float z[kTpHeld / kTpThreads];
#pragma unroll
    for (int k = 0; k < kTpHeld / kTpThreads; ++k) {
        const int i = i0 + tid + k * kTpThreads;
        z[k] = xr[i < i1 ? i : i1 - 1] / temperature;
    }
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < kTpHeld / kTpThreads; ++k) m = fmaxf(m, z[k]);
    for (int i = i0 + tid + kTpHeld; i < i1; i += kTpThreads) m = fmaxf(m, xr[i] / temperature);
    m = wave_max(m);
    if ((tid & 63) == 0) red_f[tid >> 6] = m;
    __syncthreads();
    m = red_f[0];
    for (int w = 1; w < kTpThreads / 64; ++w) m = fmaxf(m, red_f[w]);
    double sum = 0.0;
    if (m != -INFINITY) {
#pragma unroll
        for (int k = 0; k < kTpHeld / kTpThreads; ++k)
            if (i0 + tid + k * kTpThreads < i1) sum += (double)expf(z[k] - m);
        for (int i = i0 + tid + kTpHeld; i < i1; i += kTpThreads) sum += (double)expf(xr[i] / temperature - m);
    }
    sum = wave_join(sum, SumOp{});
    if ((tid & 63) == 0) red_d[tid >> 6] = sum;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < kTpThreads / 64; ++w) t += red_d[w];
        reinterpret_cast<float*>(base + L.bm)[b] = m;
        reinterpret_cast<double*>(base + L.bs)[b] = t;
    }
    if (b == 0) {  // the row histogram k_tp_hist accumulates into
        for (int q = 0; q < kShards; ++q) reinterpret_cast<unsigned long long*>(base + L.hm)[q * 256 + tid] = 0ull;
    }
}

__global__ void __launch_bounds__(kTpThreads) k_tp_zero(uint8_t* __restrict__ scratch, TpLayout L) {
    uint8_t* base = scratch + (size_t)blockIdx.x * L.stride;
    for (int q = 0; q < kShards; ++q) reinterpret_cast<unsigned long long*>(base + L.hm)[q * 256 + threadIdx.x] = 0ull;
}

__global__ void __launch_bounds__(kTpThreads) k_tp_hist(const float* __restrict__ x, int V, float temperature, int NB,
                                                         uint8_t* __restrict__ scratch, TpLayout L) {
    __shared__ unsigned hcnt[256];
    __shared__ unsigned long long hmq[256];
    const int b = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
    const float* xr = x + (long)row * V;
    uint8_t* base = scratch + (size_t)row * L.stride;
    float* p = reinterpret_cast<float*>(base + L.p);
    hcnt[tid] = 0u;
    hmq[tid] = 0ull;
    __shared__ float red_f[kTpThreads / 64];
    __shared__ double red_d[kTpThreads / 64];
    int i0, i1;
    tp_slice(V, NB, b, i0, i1);
    float z[kTpHeld / kTpThreads];  // asked for before the slices' statistics are joined
#pragma unroll
    for (int k = 0; k < kTpHeld / kTpThreads; ++k) {
        const int i = i0 + tid + k * kTpThreads;
        z[k] = xr[i < i1 ? i : i1 - 1];
    }
    float m = 0.f, sumf = 1.f;
    if (temperature > 0.f) {  // softmax(x / T): global max, then the slices' sums of exp rescaled to it
        const float* bm = reinterpret_cast<const float*>(base + L.bm);
        const double* bs = reinterpret_cast<const double*>(base + L.bs);
        // (a thread's first slice asked for at once: the maximum, again behind the barrier, and the sum behind it were three trips)
        const float m0 = bm[min(tid, NB - 1)];
        const double s0 = bs[min(tid, NB - 1)];
        float mq = tid < NB ? m0 : -INFINITY;
        for (int q = tid + kTpThreads; q < NB; q += kTpThreads) mq = fmaxf(mq, bm[q]);
        mq = wave_max(mq);
        if ((tid & 63) == 0) red_f[tid >> 6] = mq;
        __syncthreads();
        m = red_f[0];
        for (int w = 1; w < kTpThreads / 64; ++w) m = fmaxf(m, red_f[w]);
        double S = tid < NB && m0 != -INFINITY ? s0 * exp((double)m0 - (double)m) : 0.0;
        for (int q = tid + kTpThreads; q < NB; q += kTpThreads)
            if (bm[q] != -INFINITY) S += bs[q] * exp((double)bm[q] - (double)m);
        S = wave_join(S, SumOp{});  // a fixed reduction tree: the same sum every run
        if ((tid & 63) == 0) red_d[tid >> 6] = S;
        __syncthreads();
        S = 0.0;
        for (int w = 0; w < kTpThreads / 64; ++w) S += red_d[w];
        sumf = (float)S;
    }
    __syncthreads();
    auto token = [&](int i, float x0) {
        float v = 0.f;
        if (i < i1) {
            v = temperature > 0.f ? expf(x0 / temperature - m) / sumf : x0;
            if (!(v > 0.f)) v = 0.f;  // negative / NaN probabilities carry no mass
            p[i] = v;
        }
        hist_add(hcnt, hmq, i < i1, tp_bin(v), v);
    };
    // (one body, its tokens through LDS: unrolled it is 6 KiB of code that every CU fetches)
    __shared__ float held[kTpHeld];
#pragma unroll
    for (int k = 0; k < kTpHeld / kTpThreads; ++k) held[tid + k * kTpThreads] = z[k];
#pragma unroll 1
    for (int i = i0 + tid; i < i1; i += kTpThreads) token(i, i - i0 < kTpHeld ? held[i - i0] : xr[i]);
    __syncthreads();
    {  // per-block counts of bins tid and higher (compaction offsets: two reads give any range of bins)
        __shared__ unsigned wsum[kTpThreads / 64];
        const int wave = tid >> 6, bin = tid ^ 63;  // (a wave's lanes from its highest bin down)
        unsigned n = wave_scan(hcnt[bin]);
        if ((tid & 63) == 63) wsum[wave] = n;
        __syncthreads();
        for (int w = wave + 1; w < kTpThreads / 64; ++w) n += wsum[w];
        reinterpret_cast<uint16_t*>(base + L.hc)[b * 256 + bin] = (uint16_t)n;
    }
    if (hmq[tid])  // the row histogram: integer atomics, so the sums do not depend on arrival order
        atomicAdd(reinterpret_cast<unsigned long long*>(base + L.hm) + b % kShards * 256 + tid, hmq[tid]);
}

// bin t of the row's histogram
__device__ __forceinline__ unsigned long long tp_mass(const uint8_t* base, const TpLayout& L, int t) {
    unsigned long long m = 0ull;
#pragma unroll
    for (int q = 0; q < kShards; ++q) m += reinterpret_cast<const unsigned long long*>(base + L.hm)[q * 256 + t];
    return m;
}

__device__ __forceinline__ double tp_uniform(float u) {  // in [0, 1)
    const double uu = (double)u;
    if (!(uu >= 0.0)) return 0.0;
    return uu >= 1.0 ? 1.0 - 1.0 / 16777216.0 : uu;
}

__global__ void __launch_bounds__(kTpThreads) k_tp_compact(int V, int NB, float top_p, const float* __restrict__ u,
                                                            uint8_t* __restrict__ scratch, TpLayout L) {
    __shared__ unsigned long long mq[256];
    __shared__ double suf[256 + 4];
    __shared__ int top[4];
    __shared__ unsigned wtot[kTpThreads / 64][2];
    const int b = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint8_t* base = scratch + (size_t)row * L.stride;
    const float* p = reinterpret_cast<const float*>(base + L.p);
    float* cv = reinterpret_cast<float*>(base + L.cv);
    int* ci = reinterpret_cast<int*>(base + L.ci);
    int i0, i1;
    tp_slice(V, NB, b, i0, i1);
    constexpr int PT = kTpHeld / kTpThreads;  // consecutive tokens of a thread
    float v[PT];
    auto load = [&](int c0) {
#pragma unroll
        for (int k = 0; k < PT; ++k) {
            const int i = c0 + tid * PT + k;
            v[k] = p[i < i1 ? i : i1 - 1];
        }
    };
    if (i0 < i1) load(i0);  // in flight during the plan
    mq[tid] = tp_mass(base, L, tid);
    const bool used = mq[tid] != 0ull;
    const double uu = tp_uniform(u[row]);
    __syncthreads();
    suffix_masses(mq, suf);
    const int cross = highest(used && suf[tid] > (double)top_p, top);
    const bool crossed = cross >= 0;
    int c1 = cross;
    if (!crossed) {  // everything is kept: from the lowest bin in use
        const int low = highest(mq[255 - tid] != 0ull, top);
        c1 = low < 0 ? 0 : 255 - low;
    }
    const double a1 = (crossed ? suf[c1] : suf[0]) - (double)mq[c1] * kMassUnit;
    const int c_hi = max(highest(used && suf[tid] > uu * a1, top), c1);  // r = u Z >= u * a1
    // this block's place among the candidates (block order = index order), and how many there are
    const uint16_t* hc = reinterpret_cast<const uint16_t*>(base + L.hc);
    unsigned before = 0u, all = 0u;
    for (int q = tid; q < NB; q += kTpThreads) {
        const unsigned k = hc[q * 256 + c1] - (c_hi < 255 ? hc[q * 256 + c_hi + 1] : 0u);
        all += k;
        if (q < b) before += k;
    }
    before = wave_join(before, SumOp{});
    all = wave_join(all, SumOp{});
    if (lane == 0) { wtot[wave][0] = before; wtot[wave][1] = all; }
    __syncthreads();
    unsigned off = 0u;
    all = 0u;
    for (int w = 0; w < kTpThreads / 64; ++w) {
        off += wtot[w][0];
        all += wtot[w][1];
    }
    if (b == 0 && tid == 0)
        *reinterpret_cast<TpMeta*>(base + L.meta) = TpMeta{a1, suf[0], c1, c_hi, (int)all, (int)crossed};
    for (int c0 = i0; c0 < i1; c0 += kTpHeld) {  // ordered compaction
        if (c0 > i0) load(c0);
        unsigned mask = 0u;
#pragma unroll
        for (int k = 0; k < PT; ++k) {
            const int d = tp_bin(v[k]);
            if (c0 + tid * PT + k < i1 && d >= c1 && d <= c_hi) mask |= 1u << k;
        }
        const unsigned n = (unsigned)__popc(mask);
        const unsigned incl = wave_scan(n);
        __syncthreads();
        if (lane == 63) wtot[wave][0] = incl;
        __syncthreads();
        unsigned to = off + incl - n;
        for (int w = 0; w < kTpThreads / 64; ++w) {
            if (w < wave) to += wtot[w][0];
            off += wtot[w][0];
        }
#pragma unroll
        for (int k = 0; k < PT; ++k)
            if (mask >> k & 1u) {
                cv[to] = v[k];
                ci[to++] = c0 + tid * PT + k;
            }
    }
}

// One select at a time through one loop, its digits through another: a launch starts with an empty instruction cache, and a
// single workgroup waits for every line of straight code.  Few candidates (the peaked rows) are ordered by comparing each
// with all, once for both decisions: 5 of them 12.5 us by digits.
__global__ void __launch_bounds__(kSampleThreads) k_tp_select(int V, float top_p, const float* __restrict__ u,
                                                               uint8_t* __restrict__ scratch, TpLayout L,
                                                               int64_t* __restrict__ out, float* __restrict__ kept_mass) {
    __shared__ SampleSmem sm;
    __shared__ unsigned long long row_mq[256];
    const int row = blockIdx.x, tid = threadIdx.x;
    uint8_t* base = scratch + (size_t)row * L.stride;
    const float* cv = reinterpret_cast<const float*>(base + L.cv);
    const int* ci = reinterpret_cast<const int*>(base + L.ci);
    const TpMeta M = *reinterpret_cast<const TpMeta*>(base + L.meta);
    const double uu = tp_uniform(u[row]);
    // the first candidates, before their number is known (cv has V places)
    const float v0 = cv[min(tid, V - 1)], v1 = cv[min(tid + kSampleThreads, V - 1)];
    const int token0 = ci[min(tid, V - 1)];
    if (tid < 256) row_mq[tid] = tp_mass(base, L, tid);
    const bool used = tid < 256 && row_mq[tid & 255] != 0ull;
    static_assert(kHeld == 2 * kSampleThreads, "two held candidates per thread");
    sm.val[tid] = v0;
    sm.val[tid + kSampleThreads] = v1;
    if (tid < kRanked) sm.token[tid] = token0;
    __syncthreads();
    suffix_masses(row_mq, sm.row_suf);
    const int n = M.n_cand, NT = n <= kHeld ? 256 : kSampleThreads;
    if (tid >= NT) return;  // whole waves: the barriers below count those that are left
    auto value = [&](int i) { return i < kHeld ? sm.val[i] : cv[i]; };

    // ranked: this thread's candidate, the mass of the larger ones, and how many equal ones come before it; then thread t
    // takes the t-th candidate of the descending order
    const bool ranked = n <= kRanked;
    double mass = 0.0;
    if (ranked) {
        if (tid < n) {
            unsigned long long q = 0ull;
            int at = 0, ties = 0;
#pragma unroll 4  // (one at a time each waits for its read: 21.5 us a draw, so 20.1)
            for (int j = 0; j < n; ++j) {
                const float w = sm.val[j];
                q += w > v0 ? mass_q(w) : 0ull;
                at += w > v0;
                ties += w == v0 && j < tid;
            }
            sm.ord_val[at + ties] = v0;
            sm.ord_mass[at + ties] = (M.c_hi < 255 ? sm.row_suf[M.c_hi + 1] : 0.0) + (double)q * kMassUnit + (double)(ties + 1) * (double)v0;
            sm.ord_at[at + ties] = tid;
        }
        __syncthreads();
        if (tid < n && sm.ord_val[tid] > 0.f) mass = sm.ord_mass[tid];  // (0: cannot be drawn)
    }
    // First position whose inclusive cumulative mass exceeds target.  Ranked: the masses of the larger ones are truncated sums, and
    // round otherwise than the inclusive ones, so neighbours may both or neither step over a target between them: the first
    // that is past it counts, and where there must be one, the last that can be drawn.
    int turn = 0;
    auto select = [&](double target, bool must) -> SelectOut {
        if (!ranked) return radix_select(value, n, NT, target, used, sm);
        int d = lowest(mass > target, sm.top[turn ^= 1]);
        if (d < 0 && must) {
            d = n - 1;
#pragma unroll 1
            while (d >= 0 && !(sm.ord_val[d] > 0.f)) --d;
        }
        if (d < 0) return SelectOut{0u, 0.0, 0, false};
        return SelectOut{__float_as_uint(sm.ord_val[d]), sm.ord_mass[d], sm.ord_at[d], true};
    };

    // nucleus cut-off.  In exact arithmetic the kept prefix ends at k, the first position whose
    // cumulative mass C exceeds p.  The reference decides in fp32 -- C is torch's CPU cumsum
    // (double accumulation, fp32 store) and position i is dropped iff fp32(fp32(C_i) - p_i) > p
    // (:18-19) -- which can drop k or keep positions after it when C lands within an fp32 ulp
    // of p; those boundary positions are re-decided by that formula.
    auto ref_dropped = [&](double C, float v) { return __fsub_rn((float)C, v) > top_p; };
    double Z = M.total, Ck = 0.0;
    SelectOut cut{0u, 0.0, 0, false}, got{0u, 0.0, 0, false};
    enum { CUT, MORE, DRAW };
    int extra = 0;
#pragma unroll 1
    for (int what = M.crossed ? CUT : DRAW;;) {
        // DRAW: first position whose inclusive mass exceeds r = u * Z (r < Z, so it is <= k*)
        got = select(what == CUT ? (double)top_p : what == MORE ? Z : uu * Z, what == CUT || (what == DRAW && !cut.crossed));
        if (what == DRAW) break;
        const int was = what;
        what = DRAW;
        if (got.crossed) {
            const float v = __uint_as_float(got.key);
            const double C = got.mass;
            const bool dropped = ref_dropped(C, v);
            if (was == CUT) {
                cut = got;
                Ck = C;
                Z = dropped ? Ck - (double)v : Ck;
                // positions after k that fp32 still keeps.  The one after k has fp32(fp32(C) - v) within 2^-23 C of C_k:
                // when C_k is further than that past p it is dropped, and so is every later one
                if (!dropped && !(Ck - (double)top_p > 1e-6 * fmax(1.0, M.total))) what = MORE;
            } else if (!dropped) {
                Z = C;
                if (++extra < 4) what = MORE;
            }
        }
        if (what == DRAW && cut.crossed && !(Z > 0.0)) Z = Ck;  // a first token alone beyond p is always kept (:19, C_0 - p_0 = 0)
    }
    int pos = -1;
#pragma unroll 1
    for (int k = got.crossed ? 0 : 1; k < 2 && pos < 0; ++k) {  // the cut-off's token: rounding at the very end
        const SelectOut& q = k == 0 ? got : cut;
        if (q.crossed) pos = ranked ? q.rank : nth_equal(value, n, NT, q.key, q.rank, sm);
    }
    if (tid == 0) {
        out[row] = pos < 0 ? 0 : pos < kRanked ? sm.token[pos] : ci[pos];
        if (kept_mass) kept_mass[row] = (float)Z;
    }
}

static int tp_blocks(int V) {
    const int nb = (V + 2047) / 2048, least = V / 65535 + 1;  // a block's counts fit 16 bits
    return std::max(nb < 1 ? 1 : (nb > 128 ? 128 : nb), least);
}

size_t sample_scratch_bytes(int rows, int V) { return (size_t)rows * tp_layout(V, tp_blocks(V)).stride; }

void sample_top_p(hipStream_t s, const float* x, int rows, int V, float temperature, float top_p, const float* u,
                  void* scratch, int64_t* out, float* kept_mass) {
    const int NB = tp_blocks(V);
    const TpLayout L = tp_layout(V, NB);
    uint8_t* sc = reinterpret_cast<uint8_t*>(scratch);
    if (temperature > 0.f)
        hipLaunchKernelGGL(k_tp_stats, dim3(NB, rows), dim3(kTpThreads), 0, s, x, V, temperature, NB, sc, L);
    else
        hipLaunchKernelGGL(k_tp_zero, dim3(rows), dim3(kTpThreads), 0, s, sc, L);
    hipLaunchKernelGGL(k_tp_hist, dim3(NB, rows), dim3(kTpThreads), 0, s, x, V, temperature, NB, sc, L);
    hipLaunchKernelGGL(k_tp_compact, dim3(NB, rows), dim3(kTpThreads), 0, s, V, NB, top_p, u, sc, L);
    hipLaunchKernelGGL(k_tp_select, dim3(rows), dim3(kSampleThreads), 0, s, V, top_p, u, sc, L, out, kept_mass);
}

}  // namespace pgmi
