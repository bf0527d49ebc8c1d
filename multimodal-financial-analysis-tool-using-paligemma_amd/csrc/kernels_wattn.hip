// kernels_wattn.hip -- grouped-query attention over a sliding window and, optionally, the sequence's first tokens; a
// logarithmic distance bias or a tanh cap on the scores; heads over their root mean squares; rotary positions; any head
// sizes.  Scores, weights, norms, positions and angles are fp32 (angles reduced in fp64).
//
//   k_append    norms and rotates the heads of a prefill's rows, writes the key / value rows into the cache
//   k_wattn     plain form, any size and both activation types: one workgroup per (row, head), online softmax
//   k_wattn_f   fp32 MFMA form: 16 (position, head) pairs per workgroup, its waves on every fourth 16-key tile
//   k_wattn_m   bf16 MFMA form: 64 (position, head) pairs per workgroup against 64-key tiles of one key/value head
//   k_wattn_d   one new token per sequence: keys split over workgroups, partials merged by k_wattn_dc
//   k_wattn_dm  the same on bf16 MFMA
#include <algorithm>

#include "act.h"
#include "decoder.h"

namespace pgmi {

namespace {

typedef short s4v __attribute__((ext_vector_type(4)));
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNone = -1e30f;  // running maximum before any key: finite, so exp2(-inf - kNone) is 0

// score modes
constexpr int SC_PLAIN = 0;  // scale, and a cap where sc.cap > 0
constexpr int SC_BIAS = 1;   // scale and distance bias
constexpr int SC_CAPPED = 2; // a cap so small that exp(+-cap) and sums of it fit fp32: no running maximum
constexpr float kCapFixed = 66.0f;  // nats: 2^95 times 2^20 keys times values in fp32

// score in powers of two: dot * c1 - r1 log2(1 + r2 dist)
__device__ __forceinline__ float biased(float dot, float c1, float r1, float r2, float dist) {
    return dot * c1 - r1 * __builtin_amdgcn_logf(fmaf(r2, dist, 1.0f));
}
// cap log2(e) tanh(x) from exp(2x): cap2 = cap log2(e), d2 = dot * 2 log2(e) scale / cap
__device__ __forceinline__ float capped(float d2, float cap2) {
    return fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(d2)), cap2);
}
// a head's score constants; fast() on the hardware's transcendentals, exact() on the library's
template <int SC>
struct Score {
    float c1, cap2, r1, r2;
    __device__ __forceinline__ Score(const WAttnScore& s, int h) {
        cap2 = s.cap * kLog2e;
        c1 = (SC == SC_CAPPED || (SC == SC_PLAIN && s.cap > 0.0f)) ? 2.0f * kLog2e * s.scale / s.cap : s.scale * kLog2e;
        r1 = SC == SC_BIAS ? bf2f(s.r1[h]) : 0.0f;
        r2 = SC == SC_BIAS ? bf2f(s.r2[h]) : 0.0f;
    }
    __device__ __forceinline__ float fast(float dot, float dist) const {
        if constexpr (SC == SC_BIAS) return biased(dot, c1, r1, r2, dist);
        else if constexpr (SC == SC_CAPPED) return capped(dot * c1, cap2);
        else return cap2 > 0.0f ? capped(dot * c1, cap2) : dot * c1;
    }
    __device__ __forceinline__ float exact(float dot, float dist) const {
        if constexpr (SC == SC_BIAS) return dot * c1 - r1 * (log1pf(r2 * dist) * kLog2e);
        else return cap2 > 0.0f ? cap2 * tanhf(dot * c1 * (0.5f / kLog2e)) : dot * c1;
    }
};

// n-th key a query at i sees, in order: the kept first tokens before the window, then the window
struct Keys {
    int kept, lo, n;
    __device__ __forceinline__ Keys(const WAttnScore& s, int i) {
        lo = max(0, i - s.window + 1);
        kept = min(s.keep, lo);
        n = kept + i - lo + 1;
    }
    __device__ __forceinline__ int at(int v) const { return v < kept ? v : v - kept + lo; }
};

__device__ __forceinline__ void angle(double turns, int pos, float& s, float& c) {
    double t = turns * (double)pos;
    t -= rint(t);
    sincospif(2.0f * (float)t, &s, &c);
}
// pair p of a head at position pos: (u, v) turned
__device__ __forceinline__ void rotate(const double* turns, int p, int pos, float& u, float& v) {
    float s, c;
    angle(turns[p], pos, s, c);
    const float x = u;
    u = x * c - v * s;
    v = v * c + x * s;
}

// ---------------------------------------------------------------- append
// LPH lanes per head of a row (8 elements each when V == 8: head sizes that are multiples of 8)
template <typename T, int LPH, int V>
__global__ void __launch_bounds__(256) k_append(WAttnArgs a) {
    const WAttnHeads& w = a.hd;
    const int row = blockIdx.x, sub = threadIdx.x % LPH;
    const int head = blockIdx.y * (256 / LPH) + threadIdx.x / LPH, NH = w.own_kv ? w.H + 2 * w.G : w.H;
    const SeqInfo q = a.seqs[a.row_seq[row]];
    const int pos = q.start + (row - q.off);
    const T* src = reinterpret_cast<const T*>(a.qkv) + (long)row * a.ldqkv;
    const int hd = head < NH ? head : NH - 1;
    T* dst;
    int n, np, rot = w.rot;
    bool norm = w.qk_norm;
    if (hd < w.H) {
        src += hd * w.d; n = w.d; np = w.dp;
        dst = reinterpret_cast<T*>(a.q) + ((long)row * w.H + hd) * w.dp;
    } else if (hd < w.H + w.G) {
        const int g = hd - w.H;
        src += w.H * w.d + g * w.d; n = w.d; np = w.dp;
        dst = reinterpret_cast<T*>(a.kc) + (((long)q.slot * w.G + g) * a.max_tokens + pos) * w.dp;
    } else {
        const int g = hd - w.H - w.G;
        src += (w.H + w.G) * w.d + g * w.e; n = w.e; np = w.ep;
        dst = reinterpret_cast<T*>(a.vc) + (((long)q.slot * w.G + g) * a.max_tokens + pos) * w.ep;
        norm = w.v_norm;
        rot = 0;
    }
    float ss = 0.0f;
    for (int i = sub * V; i < n; i += LPH * V) {
        if constexpr (V == 8) {
            float v[8];
            ld8(src + i, v);
#pragma unroll
            for (int t = 0; t < 8; ++t) ss = fmaf(v[t], v[t], ss);
        } else {
            const float v = ldf(src + i);
            ss = fmaf(v, v, ss);
        }
    }
    ss = lanes_join<LPH>(ss, SumOp{});
    const float inv = norm ? 1.0f / sqrtf(ss / (float)n + w.eps) : 1.0f;
    if (head >= NH) return;
    for (int i = sub * V; i < np; i += LPH * V) {
        if constexpr (V == 8) {
            float v[8];
            ld8(src + i, v);
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] *= inv;
#pragma unroll
            for (int t = 0; t < 8; t += 2)
                if (i + t < rot) rotate(w.turns, (i + t) / 2, pos, v[t], v[t + 1]);
            st8(dst + i, v);
        } else {
            float u = i < n ? ldf(src + i) * inv : 0.0f;
            if (i < rot) {
                float o = ldf(src + (i ^ 1)) * inv;
                if (i & 1) { rotate(w.turns, i / 2, pos, o, u); }
                else { rotate(w.turns, i / 2, pos, u, o); }
            }
            stf(dst + i, u);
        }
    }
}

template <typename T>
void append_t(hipStream_t s, const WAttnArgs& a) {
    const int NH = a.hd.own_kv ? a.hd.H + 2 * a.hd.G : a.hd.H;
    if (a.hd.d % 8 == 0 && a.hd.e % 8 == 0)
        hipLaunchKernelGGL((k_append<T, 16, 8>), dim3(a.rows, (NH + 15) / 16), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_append<T, 64, 1>), dim3(a.rows, (NH + 3) / 4), dim3(256), 0, s, a);
}

// ---------------------------------------------------------------- plain form
template <typename T, int SC>
__global__ void __launch_bounds__(256) k_wattn(WAttnArgs a) {
    extern __shared__ float sm[];
    const WAttnHeads& w = a.hd;
    float* qs = sm;              // [dp]
    float* p = qs + w.dp;        // [256]
    float* red = p + 256;        // [8]
    const int row = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const SeqInfo q = a.seqs[a.row_seq[row]];
    const int i = q.start + (row - q.off), g = h / (w.H / w.G);
    const T* qp = reinterpret_cast<const T*>(a.q) + ((long)row * w.H + h) * w.dp;
    for (int k = tid; k < w.dp; k += 256) qs[k] = ldf(qp + k);
    __syncthreads();
    const T* kc = reinterpret_cast<const T*>(a.kc) + ((long)q.slot * w.G + g) * a.max_tokens * w.dp;
    const T* vc = reinterpret_cast<const T*>(a.vc) + ((long)q.slot * w.G + g) * a.max_tokens * w.ep;
    const Score<SC> score(a.sc, h);
    const Keys keys(a.sc, i);
    float m = kNone, l = 0.0f;
    constexpr int EM = 8;  // value columns per thread: e <= 2048
    float acc[EM] = {};
    for (int j0 = 0; j0 < keys.n; j0 += 256) {
        float s = -INFINITY;
        if (j0 + tid < keys.n) {
            const int j = keys.at(j0 + tid);
            const T* kr = kc + (long)j * w.dp;
            float dot = 0.0f;
            for (int k = 0; k < w.d; ++k) dot = fmaf(qs[k], ldf(kr + k), dot);
            s = score.exact(dot, (float)(i - j));
        }
        float t = wave_max(s);
        if (lane == 0) red[wave] = t;
        __syncthreads();
        t = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        const float mn = fmaxf(m, t), alpha = exp2f(m - mn);
        const float e = exp2f(s - mn);
        p[tid] = e;
        const float ws = wave_sum(e);
        if (lane == 0) red[4 + wave] = ws;
        __syncthreads();
        l = l * alpha + red[4] + red[5] + red[6] + red[7];
        m = mn;
        const int n = min(256, keys.n - j0);
#pragma unroll
        for (int v = 0; v < EM; ++v) {
            const int col = tid + 256 * v;
            if (col < w.e) {
                float o = acc[v] * alpha;
                for (int k = 0; k < n; ++k) o = fmaf(p[k], ldf(vc + (long)keys.at(j0 + k) * w.ep + col), o);
                acc[v] = o;
            }
        }
        __syncthreads();
    }
    T* o = reinterpret_cast<T*>(a.o) + (long)row * a.ldo;
#pragma unroll
    for (int v = 0; v < EM; ++v) {
        const int col = tid + 256 * v;
        if (col < w.e) stf(o + h * w.e + col, acc[v] / l);
    }
    if (h == w.H - 1)
        for (int k = w.H * w.e + tid; k < a.ldo; k += 256) stf(o + k, 0.0f);
}

// ---------------------------------------------------------------- fp32 MFMA form
// Products and sums stay fp32 (16x16x4 MFMA, a fused multiply-add per term).  S^T = K Q^T puts a query on lane & 15 and keys
// 4 (lane >> 4) + r on accumulator r: the B operand of O^T = V^T P^T as it stands, a contraction slot per lane group.  Which
// slot is which dim or key is free, and which output row is which value column: every load is 16 bytes a lane, straight from
// the cache into registers.  Bound by the MFMA's rate and by the longest row's chain of tiles, so a tile of 16 pairs (500
// positions of 8 heads: 250 workgroups) with its keys dealt to four waves, long rows first.  The K of the wave's next tile is
// asked for between the two products, its V after them.  k_wattn, dims of 128: 500 positions of 8 heads 105 us, 1,024
// positions 312; here 24 and 45.
__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// The piece of work, of n pieces with the longest first, that this workgroup takes.  Workgroups b and b + 256 share a CU from the start,
// later ones come as others end: the longest 256 backwards, so that the second of a CU is the shorter the longer its first is, and
// the longest are alone where n < 512.  A group's neighbours are other key/value heads' equal pieces.  us, pieces by sequence
// and head, so this: fp32, 8 heads of 128 in 2 groups, 700 rows 39.9 / 31.9, 1,024 rows 68.9 / 45.0, 1,024 + 387 + 129 rows 72.4 / 53.2;
// bf16, 16 heads, 1,024 + 387 + 129 rows 32.0 / 25.8, 1,411 + 700 + 510 + 256 + 90 rows 51.6 / 47.0.
__device__ __forceinline__ int piece() {
    const int n = gridDim.x * gridDim.y, b = blockIdx.x + gridDim.x * blockIdx.y;
    return n > 256 && b < 256 ? 255 - b : b;
}

// PAD: heads narrower than D
template <int D, int SC, bool PAD>
__global__ void __launch_bounds__(256, D <= 128 ? 2 : 1) k_wattn_f(WAttnArgs a) {
    constexpr int QC = D / 16, VC = D / 64, PT = kWAttnRows / 16;
    __shared__ __attribute__((aligned(16))) float part[4][16][68];  // 64 value columns of the waves' sums
    __shared__ float ms[4][16], ls[4][16];
    const WAttnHeads& w = a.hd;
    const int pc = piece(), g = pc % w.G, at = a.ntile * PT - 1 - pc / w.G;  // the later positions first
    const ChunkInfo tl = a.tiles[at / PT];
    const SeqInfo sq = a.seqs[tl.seq];
    const int R = w.H / w.G, nrow = sq.len * R, row0 = tl.rel + at % PT * 16;
    if (row0 >= nrow) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int fr = min(row0 + li, nrow - 1), prow = fr / R, h = g * R + fr % R, i = sq.start + prow;
    const Score<SC> score(a.sc, h);
    const int window = a.sc.window, keep = a.sc.keep;
    // positions of the first and last pairs; keys they see: [lo, hi], and the kept ones before them: [0, kept)
    const int wfirst = sq.start + row0 / R, hi = sq.start + min(row0 + 15, nrow - 1) / R;
    const int lo = max(0, wfirst - window + 1), kept = min(keep, lo), nh = (kept + 15) / 16, nt = nh + (hi - lo) / 16 + 1;
    const float* kc = reinterpret_cast<const float*>(a.kc) + ((long)sq.slot * w.G + g) * a.max_tokens * w.dp;
    const float* vc = reinterpret_cast<const float*>(a.vc) + ((long)sq.slot * w.G + g) * a.max_tokens * w.ep;
    auto key0 = [&](int t) { return t < nh ? 16 * t : lo + 16 * (t - nh); };
    auto ld4 = [](const float* p, bool ok, const float* safe) {
        if constexpr (PAD) return __builtin_bit_cast(f32x4, ldg16_sel(p, ok, safe));
        else return *reinterpret_cast<const f32x4*>(p);
    };
    f32x4 q[QC], k[QC], v[4][VC], o[VC][4];  // v[r][c]: columns 64 c + 4 li .. of key 4 lg + r; o[c][x][r]: column 64 c + 16 lg + 4 r + x
    const float* qp = reinterpret_cast<const float*>(a.q) + ((long)(sq.off + prow) * w.H + h) * w.dp;
#pragma unroll
    for (int c = 0; c < QC; ++c) q[c] = ld4(qp + 16 * c + 4 * lg, 16 * c + 4 * lg < w.dp, qp);
    auto kload = [&](int t) {
        const float* p = kc + (long)min(key0(t) + li, hi) * w.dp;
#pragma unroll
        for (int c = 0; c < QC; ++c) k[c] = ld4(p + 16 * c + 4 * lg, 16 * c + 4 * lg < w.dp, kc);
    };
    auto vload = [&](int t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float* p = vc + (long)min(key0(t) + 4 * lg + r, hi) * w.ep;
#pragma unroll
            for (int c = 0; c < VC; ++c) v[r][c] = ld4(p + 64 * c + 4 * li, 64 * c + 4 * li < w.ep, vc);
        }
    };
#pragma unroll
    for (int c = 0; c < VC; ++c)
#pragma unroll
        for (int x = 0; x < 4; ++x) o[c][x] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = kNone, l = 0.0f;
    if (wave < nt) {
        kload(wave);
        vload(wave);
    }
    for (int t = wave; t < nt; t += 4) {
        const int j0 = key0(t), tn = min(t + 4, nt - 1);
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, s1 = s;
#pragma unroll
        for (int c = 0; c < QC; c += 2)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                s = mfma_f32(k[c][x], q[c][x], s);
                s1 = mfma_f32(k[c + 1][x], q[c + 1][x], s1);
            }
        kload(tn);
        __builtin_amdgcn_sched_barrier(0);
        const bool head = t < nh;  // kept keys: every row sees those before lo
        const bool whole = head ? j0 + 16 <= kept : j0 + 15 <= wfirst && (hi - j0 < window || j0 + 16 <= keep);
        const int end = head ? kept : i + 1;
        // (& and |: as && and || the compiler branches between the keys)
        auto sees = [&](int j) { return (j < end) & ((i - j < window) | (j < keep)); };
        float mt = m;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = j0 + 4 * lg + r;
            const float e = score.exact(s[r] + s1[r], (float)(i - j));
            s[r] = sees(j) ? e : -INFINITY;
            mt = fmaxf(mt, s[r]);
        }
        mt = rows_max(mt);
        const float alpha = exp2f(m - mt);
        m = mt;
        l *= alpha;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = exp2f(s[r] - m);
            l += s[r];  // this lane's keys; summed over the lane groups at the end
        }
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int c = 0; c < VC; ++c)
#pragma unroll
                for (int x = 0; x < 4; ++x) o[c][x] *= alpha;
        }
        float bad = 0.0f;
        if (!whole) {  // a weight of zero must not meet what is not finite
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < VC; ++c)
#pragma unroll
                    for (int x = 0; x < 4; ++x) bad = fmaf(v[r][c][x], 0.0f, bad);
        }
        if (!__any(bad != bad)) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < VC; ++c)
#pragma unroll
                    for (int x = 0; x < 4; ++x) o[c][x] = mfma_f32(v[r][c][x], s[r], o[c][x]);
        } else {
#pragma clang loop unroll(disable)
            for (int n = 0; n < 16; ++n) {
                const int j = j0 + n, from = n / 4 * 16 + li;
                const float p0 = __shfl(s[0], from, 64), p1 = __shfl(s[1], from, 64), p2 = __shfl(s[2], from, 64), p3 = __shfl(s[3], from, 64);
                const float p = n & 2 ? n & 1 ? p3 : p2 : n & 1 ? p1 : p0;
                if (!sees(j)) continue;
                const float* vp = vc + (long)j * w.ep;
#pragma unroll
                for (int c = 0; c < VC; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int col = 64 * c + 16 * lg + 4 * r;
                        const f32x4 f = ld4(vp + col, col < w.ep, vc);
                        const bool in = col < w.ep;
#pragma unroll
                        for (int x = 0; x < 4; ++x) o[c][x][r] = in ? fmaf(p, f[x], o[c][x][r]) : 0.0f;
                    }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        vload(tn);
        __builtin_amdgcn_sched_barrier(0);
    }
    l = rows_sum(l);
    if (lg == 0) { ms[wave][li] = m; ls[wave][li] = l; }
    __syncthreads();
    const float f = exp2f(m - fmaxf(fmaxf(ms[0][li], ms[1][li]), fmaxf(ms[2][li], ms[3][li])));
    // a thread per four value columns of a pair
    const int pr = tid >> 4, of = row0 + pr, oh = g * R + of % R;
    const float pm = fmaxf(fmaxf(ms[0][pr], ms[1][pr]), fmaxf(ms[2][pr], ms[3][pr]));
    float sum = 0.0f;
#pragma unroll
    for (int x = 0; x < 4; ++x) sum = fmaf(ls[x][pr], exp2f(ms[x][pr] - pm), sum);
    float* out = reinterpret_cast<float*>(a.o) + (long)(sq.off + of / R) * a.ldo;
#pragma unroll
    for (int c = 0; c < VC; ++c) {
        if (c) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(&part[wave][li][16 * lg + 4 * r]) = f32x4{o[c][0][r] * f, o[c][1][r] * f, o[c][2][r] * f, o[c][3][r] * f};
        __syncthreads();
        f32x4 t = *reinterpret_cast<const f32x4*>(&part[0][pr][(tid & 15) * 4]);
#pragma unroll
        for (int x = 1; x < 4; ++x) t += *reinterpret_cast<const f32x4*>(&part[x][pr][(tid & 15) * 4]);
        const int col = 64 * c + (tid & 15) * 4;
        if (of < nrow)
#pragma unroll
            for (int x = 0; x < 4; ++x)
                if (col + x < w.e) out[oh * w.e + col + x] = t[x] / sum;
    }
    if (of < nrow && oh == w.H - 1)
        for (int x = w.H * w.e + (tid & 15); x < a.ldo; x += 16) out[x] = 0.0f;
}

template <int D>
void run_f(hipStream_t s, const WAttnArgs& a) {
    const dim3 grid(a.ntile * (kWAttnRows / 16), a.hd.G);
    const bool pad = a.hd.dp != D || a.hd.ep != D;
    if (a.sc.r1 && pad) hipLaunchKernelGGL((k_wattn_f<D, SC_BIAS, true>), grid, dim3(256), 0, s, a);
    else if (a.sc.r1) hipLaunchKernelGGL((k_wattn_f<D, SC_BIAS, false>), grid, dim3(256), 0, s, a);
    else if (pad) hipLaunchKernelGGL((k_wattn_f<D, SC_PLAIN, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_wattn_f<D, SC_PLAIN, false>), grid, dim3(256), 0, s, a);
}

// ---------------------------------------------------------------- bf16 MFMA form
// Scores are computed transposed, S^T = K Q^T, so that a lane holds one query row (column lane & 15) and, after
// two 16-key tiles, exactly the 8 weights its B fragment of O^T = V^T P^T needs (the contraction order is free:
// slot 8g + i is key 4g + i of the first tile for i < 4, of the second for i >= 4).  V^T fragments are
// transposed LDS reads of the row-major V tile.
// Bound, where the chip is full, by LDS (a tile's K and V are read by each of its four waves, 128 KB, and V in halves) and by the
// score's vector operations; where it is not, by the longest tile's chain of barriers, LDS reads, two products and what is between
// them, which two teams halve (wattn_teams).  us, 1,300 + 511 + 235 + 2 rows of 16 heads of 128, capped scores: 51.3 before; sums in
// VGPRs, loads and masks without a branch each 46.2; two teams 39.6, tiles in the order of their keys 33.0.  32 rows a wave, which halves the LDS reads, beat this only for
// one sequence of 4,096 rows (64 against 77) and lost 20 to 40 % below 1,000.
constexpr size_t wattn_m_lds(int DQ, int DV, int teams) { return (size_t)teams * 64 * (DQ + 8 + DV + 8) * 2; }
template <int DQ, int DV, int SC, int TEAMS, bool PAD>
__global__ void __launch_bounds__(256 * TEAMS) k_wattn_m(WAttnArgs a) {
    const WAttnHeads& w = a.hd;
    constexpr int KT = 64;                 // keys per tile
    constexpr int KS = DQ + 8, VS = DV + 8;  // LDS row strides (elements)
    constexpr int KQ = KT * DQ / 8 / 256, VQ = KT * DV / 8 / 256;  // 16-byte pieces per thread
    extern __shared__ __attribute__((aligned(16))) uint8_t smem_wattn[];
    const int team = TEAMS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    uint16_t* Ks = reinterpret_cast<uint16_t*>(smem_wattn + (size_t)team * wattn_m_lds(DQ, DV, 1));
    uint16_t* Vs = Ks + KT * KS;
    const int R = w.H / w.G;
    // One sequence: every other key/value head backwards, so that a CU's two workgroups are not both long (2,048 rows 48.3 us, as
    // pieces 49.8); several: pieces
    const int pc = piece(), g = a.nseq > 1 ? pc % w.G : blockIdx.y;
    const ChunkInfo tl = a.tiles[a.nseq > 1 ? a.ntile - 1 - pc / w.G : g & 1 ? a.ntile - 1 - (int)blockIdx.x : blockIdx.x];
    const SeqInfo sq = a.seqs[tl.seq];
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int nrow = sq.len * R;
    // this lane's query row
    const int fr = tl.rel + wave * 16 + li;
    const bool ok = fr < nrow;
    const int frc = ok ? fr : nrow - 1;
    const int prow = frc / R, hh = frc % R, h = g * R + hh;
    const int i = sq.start + prow;
    auto ld = [](const uint16_t* p, bool in, const uint16_t* safe) {  // (the choice is a branch around every load)
        if constexpr (PAD) return ldg16_sel(p, in, safe);
        else return ldg16(p);
    };
    const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + ((long)(sq.off + prow) * w.H + h) * w.dp;
    short8 qf[DQ / 32];
#pragma unroll
    for (int c = 0; c < DQ / 32; ++c) {
        const int k = c * 32 + 8 * lg;
        qf[c] = __builtin_bit_cast(short8, ld(qp + k, k < w.dp, qp));
    }
    const Score<SC> score(a.sc, h);
    const float r1 = score.r1, r2 = score.r2, c1 = score.c1;
    const int window = a.sc.window, keep = a.sc.keep;
    // keys the tile's rows see: [lo, hi], and the kept ones before them: [0, kept)
    const int last = min(tl.rel + kWAttnRows, nrow) - 1;
    const int lo = max(0, sq.start + tl.rel / R - window + 1), hi = sq.start + last / R;
    const int kept = min(keep, lo);
    // positions of this wave's first and last rows
    const int wfirst = sq.start + min(tl.rel + wave * 16, nrow - 1) / R;
    const int wlast = sq.start + min(tl.rel + wave * 16 + 15, nrow - 1) / R;
    const uint16_t* kc = reinterpret_cast<const uint16_t*>(a.kc) + ((long)sq.slot * w.G + g) * a.max_tokens * w.dp;
    const uint16_t* vc = reinterpret_cast<const uint16_t*>(a.vc) + ((long)sq.slot * w.G + g) * a.max_tokens * w.ep;
    f32x4 o[DV / 16];
#pragma unroll
    for (int c = 0; c < DV / 16; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = SC == SC_CAPPED ? 0.0f : kNone, l = 0.0f;
    uint4 kr[KQ], vr[VQ];
    auto gload = [&](int j0) {
#pragma unroll
        for (int x = 0; x < KQ; ++x) {
            const int e = tid + 256 * x, r = e / (DQ / 8), k = (e % (DQ / 8)) * 8;
            const int j = min(j0 + r, hi);
            kr[x] = ld(kc + (long)j * w.dp + k, k < w.dp, kc);
        }
#pragma unroll
        for (int x = 0; x < VQ; ++x) {
            const int e = tid + 256 * x, r = e / (DV / 8), k = (e % (DV / 8)) * 8;
            const int j = min(j0 + r, hi);
            vr[x] = ld(vc + (long)j * w.ep + k, k < w.ep, vc);
        }
    };
    // tile t: the kept keys' first, then the window's; a team takes every TEAMS-th
    const int nh = (kept + KT - 1) / KT, nt = nh + (hi - lo) / KT + 1;
    auto key0 = [&](int t) { return t < nh ? KT * t : lo + KT * (t - nh); };
    if (team < nt) gload(key0(team));
    for (int t0 = 0; t0 < nt; t0 += TEAMS) {
        const int t = t0 + team, j0 = key0(t);
        __syncthreads();  // the previous tile's reads are done
#pragma unroll
        for (int x = 0; x < KQ; ++x) {
            const int e = tid + 256 * x, r = e / (DQ / 8), k = (e % (DQ / 8)) * 8;
            *reinterpret_cast<uint4*>(Ks + r * KS + k) = kr[x];
        }
#pragma unroll
        for (int x = 0; x < VQ; ++x) {
            const int e = tid + 256 * x, r = e / (DV / 8), k = (e % (DV / 8)) * 8;
            *reinterpret_cast<uint4*>(Vs + r * VS + k) = vr[x];
        }
        __syncthreads();
        if (t + TEAMS < nt) gload(key0(t + TEAMS));
        if (t >= nt || j0 > wlast || (j0 + KT <= wfirst - window + 1 && j0 >= keep)) continue;  // no row of this wave sees the tile
        f32x4 st[4];
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            st[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DQ / 32; ++c) {
                const short8 kf = *reinterpret_cast<const short8*>(Ks + (n * 16 + li) * KS + c * 32 + 8 * lg);
                st[n] = mfma16(kf, qf[c], st[n]);
            }
        }
        const bool head = t < nh;  // kept keys: every row sees those before lo
        const int end = head ? kept : i + 1;
        float mt = m;
        // 1 + r2 (i - j) for key j0 + 4 lg, less r2 per key after it
        const float x0 = fmaf(r2, (float)(i - j0 - 4 * lg), 1.0f);
        auto value = [&](float dot, int k) {
            if constexpr (SC == SC_BIAS) return fmaf(-r1, __builtin_amdgcn_logf(fmaf(-r2, (float)k, x0)), dot * c1);
            else return score.fast(dot, 0.0f);
        };
        if (head ? j0 + KT <= kept : j0 + KT - 1 <= wfirst && (wlast - j0 < window || j0 + KT <= keep)) {  // no mask
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) st[n][r] = value(st[n][r], n * 16 + r);
        } else {
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = j0 + n * 16 + 4 * lg + r;
                    const bool see = (j < end) & ((i - j < window) | (j < keep));  // (as && and || branches between the keys)
                    const float s = value(st[n][r], n * 16 + r);
                    st[n][r] = see ? s : -INFINITY;
                }
        }
        float alpha = 1.0f;
        if constexpr (SC != SC_CAPPED) {
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) mt = fmaxf(mt, st[n][r]);
            mt = rows_max(mt);
            alpha = __builtin_amdgcn_exp2f(m - mt);
            m = mt;
        }
        float ls = 0.0f;
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                st[n][r] = __builtin_amdgcn_exp2f(SC == SC_CAPPED ? st[n][r] : st[n][r] - m);
                ls += st[n][r];
            }
        l = l * alpha + ls;  // this lane's keys; summed over the lane groups at the end
        if (SC != SC_CAPPED && __any(alpha != 1.0f)) {
#pragma unroll
            for (int c = 0; c < DV / 16; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[c][r] *= alpha;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            short8 pf;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pf[r] = (short)f2bf(st[2 * u][r]);
                pf[4 + r] = (short)f2bf(st[2 * u + 1][r]);
            }
#pragma unroll
            for (int c = 0; c < DV / 16; ++c) {
                uint16_t* vp = Vs + (u * 32 + 4 * lg + (li >> 2)) * VS + c * 16 + 4 * (li & 3);
                const s4v lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*)(vp));
                const s4v hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*)(vp + 16 * VS));
                const short8 vf = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                o[c] = mfma16(vf, pf, o[c]);
            }
        }
    }
    if constexpr (TEAMS == 2) {  // the other team's sums, in its lanes' places
        f32x4* at = reinterpret_cast<f32x4*>(smem_wattn) + tid;
        float* ml = reinterpret_cast<float*>(at + (DV / 16) * 256 - tid) + tid;
        __syncthreads();  // the last tiles' reads are done
        if (team) {
#pragma unroll
            for (int c = 0; c < DV / 16; ++c) at[c * 256] = o[c];
            ml[0] = m;
            ml[256] = l;
        }
        __syncthreads();
        if (team) return;
        const float m2 = ml[0], mt = fmaxf(m, m2);
        const float f1 = SC == SC_CAPPED ? 1.0f : __builtin_amdgcn_exp2f(m - mt), f2 = SC == SC_CAPPED ? 1.0f : __builtin_amdgcn_exp2f(m2 - mt);
        l = l * f1 + ml[256] * f2;
#pragma unroll
        for (int c = 0; c < DV / 16; ++c) {
            const f32x4 o2 = at[c * 256];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[c][r] = o[c][r] * f1 + o2[r] * f2;
        }
    }
    l = rows_sum(l);
    if (!ok) return;
    const float inv = 1.0f / l;
    uint16_t* op = reinterpret_cast<uint16_t*>(a.o) + (long)(sq.off + prow) * a.ldo + h * w.e;
#pragma unroll
    for (int c = 0; c < DV / 16; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = c * 16 + 4 * lg + r;
            if (col < w.e) op[col] = f2bf(o[c][r] * inv);
        }
    if (h == w.H - 1 && lg == 0)
        for (int k = w.H * w.e; k < a.ldo; ++k) reinterpret_cast<uint16_t*>(a.o)[(long)(sq.off + prow) * a.ldo + k] = 0;
}

// the score mode of a layer on the hardware's transcendentals
int score_mode(const WAttnScore& sc) { return sc.r1 ? SC_BIAS : sc.cap > 0.0f && sc.cap <= kCapFixed ? SC_CAPPED : SC_PLAIN; }

template <int DQ, int DV, int SC, int TEAMS, bool PAD>
void run_mt(hipStream_t s, const WAttnArgs& a) {
    constexpr size_t lds = wattn_m_lds(DQ, DV, TEAMS);
    static_assert(TEAMS == 1 || (size_t)256 * (DV + 8) <= lds, "the other team's sums fit");
    static const bool once = [] {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_wattn_m<DQ, DV, SC, TEAMS, PAD>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    }();
    (void)once;
    hipLaunchKernelGGL((k_wattn_m<DQ, DV, SC, TEAMS, PAD>), dim3(a.ntile, a.hd.G), dim3(256 * TEAMS), lds, s, a);
}
template <int DQ, int DV, int SC>
void run_ms(hipStream_t s, const WAttnArgs& a) {
    const bool pad = a.hd.dp != DQ || a.hd.ep != DV;
    if (a.teams) pad ? run_mt<DQ, DV, SC, 2, true>(s, a) : run_mt<DQ, DV, SC, 2, false>(s, a);
    else pad ? run_mt<DQ, DV, SC, 1, true>(s, a) : run_mt<DQ, DV, SC, 1, false>(s, a);
}
template <int DQ, int DV>
void run_m(hipStream_t s, const WAttnArgs& a) {
    const int mode = score_mode(a.sc);
    if (mode == SC_BIAS) run_ms<DQ, DV, SC_BIAS>(s, a);
    else if (mode == SC_CAPPED) run_ms<DQ, DV, SC_CAPPED>(s, a);
    else run_ms<DQ, DV, SC_PLAIN>(s, a);
}
template <int DQ>
void run_mv(hipStream_t s, const WAttnArgs& a) {
    if (a.hd.ep <= 64) run_m<DQ, 64>(s, a);
    else if (a.hd.ep <= 96) run_m<DQ, 96>(s, a);
    else if (a.hd.ep <= 128) run_m<DQ, 128>(s, a);
    else run_m<DQ, 256>(s, a);
}

// ---------------------------------------------------------------- one token per sequence
constexpr int DK = 64;  // keys per tile

// grid (split, G, B).  RB: query heads of the group handled at once (registers).
// part record of (b, head, split): [ep] weighted values, then running maximum, then sum of weights
template <typename T, int RB, int SC>
__global__ void __launch_bounds__(256) k_wattn_d(WAttnDecodeArgs a) {
    extern __shared__ float sm[];
    const WAttnHeads& w = a.hd;
    const int R = w.H / w.G;
    float* qs = sm;                 // [R][dp] normalised queries
    float* ps = qs + R * w.dp;      // [RB][DK] scores, then weights
    float* st = ps + RB * DK;       // [RB][4]: running max, sum, alpha
    float* red = st + RB * 4;       // [256][8] cross-group reduction
    const int g = blockIdx.y, b = blockIdx.z, sp = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int slot = a.slot[b], i = a.pos[b];
    const Keys keys(a.sc, i);  // k0, k1, j below count the keys this query sees
    const int per = ((keys.n + a.nsplit - 1) / a.nsplit + DK - 1) / DK * DK;
    const int k0 = sp * per, k1 = min(keys.n, k0 + per);  // empty when k0 >= k1
    const T* qkv = reinterpret_cast<const T*>(a.qkv) + (long)b * a.ldqkv;
    const int rs = w.ep + 2;
    float* part = a.part + (((long)b * w.H + g * R) * a.nsplit + sp) * rs;
    if (k0 >= k1) {
        for (int r = tid; r < R; r += 256) {
            part[(long)r * a.nsplit * rs + w.ep] = kNone;
            part[(long)r * a.nsplit * rs + w.ep + 1] = 0.0f;
        }
        return;
    }
    T* kc = reinterpret_cast<T*>(a.kc) + ((long)slot * w.G + g) * a.max_tokens * w.dp;
    T* vc = reinterpret_cast<T*>(a.vc) + ((long)slot * w.G + g) * a.max_tokens * w.ep;
    // n elements of a head row by one wave, normed and rotated, rounded to T as the prefill form rounds them: put(k, v)
    auto head_row = [&](const T* src, int n, int np, bool norm, int rot, auto put) {
        float ss = 0.0f;
        for (int k = lane; k < n; k += 64) ss = fmaf(ldf(src + k), ldf(src + k), ss);
        const float inv = norm ? 1.0f / sqrtf(wave_sum(ss) / (float)n + w.eps) : 1.0f;
        for (int k = 2 * lane; k < np; k += 128) {  // np is even
            float u = k < n ? ldf(src + k) * inv : 0.0f, v = k + 1 < n ? ldf(src + k + 1) * inv : 0.0f;
            if (k < rot) rotate(w.turns, k / 2, i, u, v);
            put(k, u);
            put(k + 1, v);
        }
    };
    for (int r = wave; r < R; r += 4)
        head_row(qkv + (g * R + r) * w.d, w.d, w.dp, w.qk_norm, w.rot, [&](int k, float v) {
            T t;
            stf(&t, v);
            qs[r * w.dp + k] = ldf(&t);
        });
    if (k1 == keys.n && w.own_kv) {  // this workgroup's keys include the new one: write its cache rows
        if (wave == 0)
            head_row(qkv + w.H * w.d + g * w.d, w.d, w.dp, w.qk_norm, w.rot,
                     [&](int k, float v) { stf(kc + (long)i * w.dp + k, v); });
        else if (wave == 1)
            head_row(qkv + (w.H + w.G) * w.d + g * w.e, w.e, w.ep, w.v_norm, 0,
                     [&](int k, float v) { stf(vc + (long)i * w.ep + k, v); });
        __threadfence_block();
    }
    __syncthreads();
    // scores: LPK lanes share a key, 8 elements each per step
    int LPK = 1;
    while (LPK < 64 && LPK * 8 < w.dp) LPK <<= 1;
    const int kl = lane % LPK, kw = wave * (64 / LPK) + lane / LPK, kstep = 4 * (64 / LPK);
    // weighted values: CPV threads span the columns (8 each), the rest split the keys
    const int nch = w.ep / 8;
    int CPV = 1;
    while (CPV < 256 && CPV < nch) CPV <<= 1;
    const int vch = tid % CPV, vk = tid / CPV, vkn = 256 / CPV;
    for (int r0 = 0; r0 < R; r0 += RB) {
        const int nr = min(RB, R - r0);
        float acc[RB][8];
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int v = 0; v < 8; ++v) acc[r][v] = 0.0f;
        if (tid < RB) { st[tid * 4] = kNone; st[tid * 4 + 1] = 0.0f; }
        __syncthreads();
        for (int j0 = k0; j0 < k1; j0 += DK) {
            for (int kk = kw; kk < DK; kk += kstep) {
                const int j = j0 + kk;
                float dot[RB];
#pragma unroll
                for (int r = 0; r < RB; ++r) dot[r] = 0.0f;
                if (j < k1)
                    for (int c = kl * 8; c < w.dp; c += LPK * 8) {
                        float kv[8];
                        ld8(kc + (long)keys.at(j) * w.dp + c, kv);
#pragma unroll
                        for (int r = 0; r < RB; ++r) {
                            const float* q = qs + (r0 + (r < nr ? r : 0)) * w.dp + c;
#pragma unroll
                            for (int v = 0; v < 8; ++v) dot[r] = fmaf(q[v], kv[v], dot[r]);
                        }
                    }
#pragma unroll
                for (int r = 0; r < RB; ++r) dot[r] = lanes_join_n(dot[r], LPK, SumOp{});
                if (kl == 0) {
#pragma unroll
                    for (int r = 0; r < RB; ++r) {
                        const int h = g * R + r0 + (r < nr ? r : 0);
                        ps[r * DK + kk] = j < k1 ? Score<SC>(a.sc, h).exact(dot[r], (float)(i - keys.at(j))) : -INFINITY;
                    }
                }
            }
            __syncthreads();
            for (int r = wave; r < RB; r += 4) {
                const float s = ps[r * DK + lane];
                const float mo = st[r * 4], mn = fmaxf(mo, wave_max(s));
                const float e = exp2f(s - mn);
                ps[r * DK + lane] = e;
                const float sum = wave_sum(e);
                if (lane == 0) {
                    const float al = exp2f(mo - mn);
                    st[r * 4] = mn;
                    st[r * 4 + 1] = st[r * 4 + 1] * al + sum;
                    st[r * 4 + 2] = al;
                }
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                const float al = st[r * 4 + 2];
#pragma unroll
                for (int v = 0; v < 8; ++v) acc[r][v] *= al;
            }
            if (vch < nch) {
                const int n = min(DK, k1 - j0);
                for (int kk = vk; kk < n; kk += vkn) {
                    float vv[8];
                    ld8(vc + (long)keys.at(j0 + kk) * w.ep + vch * 8, vv);
#pragma unroll
                    for (int r = 0; r < RB; ++r) {
                        const float p = ps[r * DK + kk];
#pragma unroll
                        for (int v = 0; v < 8; ++v) acc[r][v] = fmaf(p, vv[v], acc[r][v]);
                    }
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            if (r < nr) {
#pragma unroll
                for (int v = 0; v < 8; ++v) red[tid * 8 + v] = acc[r][v];
                __syncthreads();
                float* pr = part + (long)(r0 + r) * a.nsplit * rs;
                for (int c = tid; c < w.ep; c += 256) {
                    float t = 0.0f;
                    for (int k = 0; k < vkn; ++k) t += red[(k * CPV + c / 8) * 8 + c % 8];
                    pr[c] = t;
                }
                if (tid == 0) {
                    pr[w.ep] = st[r * 4];
                    pr[w.ep + 1] = st[r * 4 + 1];
                }
                __syncthreads();
            }
        }
    }
}

// bf16 MFMA form, 16 query heads of a group per workgroup (grid (split, G * head blocks, B)).  A wave takes 32-key
// tiles: S^T = K Q^T with the key fragments straight from the cache, then O^T += V^T P^T as k_wattn_m, the values
// through the wave's own LDS rows; the four waves' running sums meet in LDS.
// VEC: head sizes that are multiples of 8 (up to 64 four waves to a SIMD: 136 registers and three, 16 sequences of 8 heads 143 us for 129).
// how a head lies: of odd sizes; of whole vectors, padded to DQ and DV; DQ and DV themselves (15.1 KB of code for those, 12.4 where
// nothing is chosen: one row over 1,000 keys 9.1 -> 7.2 us, 8 rows over up to 1,411 10.0 -> 8.5)
enum { ODD, VECTORS, WHOLE };
template <int DQ, int DV, int SC, int HEADS>
__global__ void __launch_bounds__(256, DQ <= 64 && DV <= 64 && HEADS != ODD ? 4 : 1) k_wattn_dm(WAttnDecodeArgs a) {
    const WAttnHeads& w = a.hd;
    constexpr bool VEC = HEADS != ODD, FULL = HEADS == WHOLE;
    const int dp = FULL ? DQ : w.dp, ep = FULL ? DV : w.ep, qd = FULL ? DQ : w.d, ve = FULL ? DV : w.e;
    auto ld = [](const uint16_t* p, bool in, const uint16_t* safe) {  // (the choice is a branch around every load)
        if constexpr (FULL) return ldg16(p);
        else return ldg16_sel(p, in, safe);
    };
    constexpr int VS = DV + 8;
    __shared__ __attribute__((aligned(16))) uint16_t Vs[4][32 * VS];
    __shared__ float sml[4][16][2];
    __shared__ __attribute__((aligned(16))) float2 turned[DQ / 2];  // cos and sin of the rotated pairs
    const int R = w.H / w.G, hb = blockIdx.y / w.G, g = blockIdx.y % w.G, b = blockIdx.z, sp = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lg = lane >> 4;
    const int slot = a.slot[b], i = a.pos[b];
    const Keys keys(a.sc, i);  // k0, k1, kend, j0 below count the keys this query sees
    const int per = ((keys.n + a.nsplit - 1) / a.nsplit + 127) / 128 * 128;
    const int k0 = sp * per, k1 = min(keys.n, k0 + per);
    const uint16_t* qkv = reinterpret_cast<const uint16_t*>(a.qkv) + (long)b * a.ldqkv;
    const int r0 = hb * 16, nr = min(16, R - r0), rs = ep + 2;
    float* part = a.part + (((long)b * w.H + g * R + r0) * a.nsplit + sp) * rs;
    if (k0 >= k1) {
        if (tid < nr) {
            part[(long)tid * a.nsplit * rs + ep] = kNone;
            part[(long)tid * a.nsplit * rs + ep + 1] = 0.0f;
        }
        return;
    }
    uint16_t* kc = reinterpret_cast<uint16_t*>(a.kc) + ((long)slot * w.G + g) * a.max_tokens * dp;
    uint16_t* vc = reinterpret_cast<uint16_t*>(a.vc) + ((long)slot * w.G + g) * a.max_tokens * ep;
    // A new key (position i) never passes through the cache here: its score and value come from its qkv row, in
    // wave 0 of the last split, which also writes its cache rows.  Cached keys end at kend.
    const bool own = w.own_kv && k1 == keys.n;
    const int kend = own ? k1 - 1 : k1;
    const int h = g * R + r0 + (li < nr ? li : 0);
    // the scores' and angles' few operands (each asked for where it was used, a trip to memory behind all others: 8 heads
    // at 1,000 keys 8.3 us, so 6.4), the first
    // tile's loads, then the query's: all in flight together
    const Score<SC> score(a.sc, h);
    const double turn = w.rot > 0 ? w.turns[min(tid, w.rot / 2 - 1)] : 0.0;
    asm volatile("" ::: "memory");
    uint4 vr[DV / 16], kr[2][DQ / 32];
    auto gload = [&](int j0) {
        const int jm = max(kend - 1, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint16_t* p = kc + (long)keys.at(min(j0 + t * 16 + li, jm)) * dp;
#pragma unroll
            for (int c = 0; c < DQ / 32; ++c) kr[t][c] = ld(p + c * 32 + 8 * lg, c * 32 + 8 * lg < dp, p);
        }
#pragma unroll
        for (int x = 0; x < DV / 16; ++x) {
            const int e = lane + 64 * x, r = e / (DV / 8), k = (e % (DV / 8)) * 8;
            vr[x] = ld(vc + (long)keys.at(min(j0 + r, jm)) * ep + k, k < ep, vc);
        }
    };
    if (k0 + wave * 32 < kend) gload(k0 + wave * 32);
    // this lane's dims 8 lg .. 8 lg + 7 of every 32 of its query and of the new key, and 4 lg .. of every 16 of the new value
    float qr[DQ / 32][8], knr[DQ / 32][8], vnr[DV / 16][4];
    auto raw = [&](const uint16_t* src, int n, float (&q)[DQ / 32][8]) {
#pragma unroll
        for (int c = 0; c < DQ / 32; ++c) {
            const int k = c * 32 + 8 * lg;
            if constexpr (VEC) {
                ld8(src + (k < n ? k : 0), q[c]);
#pragma unroll
                for (int v = 0; v < 8; ++v) q[c][v] = k < n ? q[c][v] : 0.0f;
            } else {
#pragma unroll
                for (int v = 0; v < 8; ++v) q[c][v] = k + v < n ? bf2f(src[k + v]) : 0.0f;
            }
        }
    };
    raw(qkv + h * qd, qd, qr);
    // (by the one wave that uses them: every wave asked for them and cut their pads, 40 sequences of 16 heads of 80 53 us a layer, so 49)
    const bool mine = own && wave == 0;
    const uint16_t* vn = qkv + (w.H + w.G) * qd + g * ve;
    if (mine) {
        raw(qkv + w.H * qd + g * qd, qd, knr);
#pragma unroll
        for (int c = 0; c < DV / 16; ++c) {
            const int k = c * 16 + 4 * lg;
            if constexpr (VEC) {
                ld4(vn + (k < ve ? k : 0), vnr[c]);
#pragma unroll
                for (int r = 0; r < 4; ++r) vnr[c][r] = k < ve ? vnr[c][r] : 0.0f;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) vnr[c][r] = k + r < ve ? bf2f(vn[k + r]) : 0.0f;
            }
        }
    }
    // every head turns by the same angles: a thread per pair, once (by every lane for its own dims, each turn loaded behind its
    // own check, and the new key and value asked for only then: 8 sequences of 16 heads 13.3 us, now 9.8)
    if (tid < w.rot / 2) {
        float s, c;
        angle(turn, i, s, c);
        turned[tid] = make_float2(c, s);
    }
    if (w.rot > 0) __syncthreads();
    // such a head row, normed and rotated, as bf16
    auto head_row = [&](const float (&q)[DQ / 32][8], short8 (&f)[DQ / 32]) {
        float ss = 0.0f;
        float inv = 1.0f;
        if (w.qk_norm) {
#pragma unroll
            for (int c = 0; c < DQ / 32; ++c)
#pragma unroll
                for (int v = 0; v < 8; ++v) ss = fmaf(q[c][v], q[c][v], ss);
            ss = rows_sum(ss);
            inv = 1.0f / sqrtf(ss / (float)qd + w.eps);
        }
        auto put = [&](auto turns) {
            float2 r[DQ / 32][4];  // (all asked for at once; past the rotated pairs whatever is there, and not taken)
            if constexpr (decltype(turns)::value)
#pragma unroll
                for (int c = 0; c < DQ / 32; ++c)
#pragma unroll
                    for (int v = 0; v < 4; ++v) r[c][v] = turned[c * 16 + 4 * lg + v];
#pragma unroll
            for (int c = 0; c < DQ / 32; ++c)
#pragma unroll
                for (int v = 0; v < 8; v += 2) {
                    float x = q[c][v] * inv, y = q[c][v + 1] * inv;
                    if constexpr (decltype(turns)::value) {
                        const float u = x * r[c][v / 2].x - y * r[c][v / 2].y, z = y * r[c][v / 2].x + x * r[c][v / 2].y;
                        const bool in = c * 32 + 8 * lg + v < w.rot;
                        x = in ? u : x;
                        y = in ? z : y;
                    }
                    f[c][v] = (short)f2bf(x);
                    f[c][v + 1] = (short)f2bf(y);
                }
        };
        if (w.rot > 0) put(std::true_type{});
        else put(std::false_type{});
    };
    short8 qf[DQ / 32];
    head_row(qr, qf);
    f32x4 o[DV / 16];
#pragma unroll
    for (int c = 0; c < DV / 16; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = SC == SC_CAPPED ? 0.0f : kNone, l = 0.0f;
    if (mine) {
        short8 kf[DQ / 32];
        head_row(knr, kf);
        float dot = 0.0f;
#pragma unroll
        for (int c = 0; c < DQ / 32; ++c)
#pragma unroll
            for (int v = 0; v < 8; ++v) dot = fmaf(bf2f((uint16_t)qf[c][v]), bf2f((uint16_t)kf[c][v]), dot);
        dot = rows_sum(dot);
        const float s = score.fast(dot, 0.0f);
        float p = 1.0f;
        if constexpr (SC == SC_CAPPED) p = __builtin_amdgcn_exp2f(s);
        else m = s;
        l = lg == 0 ? p : 0.0f;  // summed over the lane groups below
        float vss = 0.0f;
#pragma unroll
        for (int c = 0; c < DV / 16; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                o[c][r] = vnr[c][r];
                vss = fmaf(vnr[c][r], vnr[c][r], vss);
            }
        float vinv = 1.0f;
        if (w.v_norm) {
            vss = rows_sum(vss);
            vinv = 1.0f / sqrtf(vss / (float)ve + w.eps);
        }
#pragma unroll
        for (int c = 0; c < DV / 16; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[c][r] = rbf(o[c][r] * vinv) * p;
        if (li == 0) {
#pragma unroll
            for (int c = 0; c < DQ / 32; ++c)
                if (c * 32 + 8 * lg < dp) *reinterpret_cast<short8*>(kc + (long)i * dp + c * 32 + 8 * lg) = kf[c];
        }
        for (int k = lane; k < ep; k += 64) vc[(long)i * ep + k] = k < ve ? f2bf(bf2f(vn[k]) * vinv) : 0;
    }
    for (int j0 = k0 + wave * 32; j0 < kend; j0 += 128) {
        f32x4 st[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            st[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DQ / 32; ++c) st[t] = mfma16(__builtin_bit_cast(short8, kr[t][c]), qf[c], st[t]);
        }
        float mt = m;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = j0 + t * 16 + 4 * lg + r;
                const float s = score.fast(st[t][r], SC == SC_BIAS ? (float)(i - keys.at(j)) : 0.0f);
                st[t][r] = j < kend ? s : -INFINITY;
                if constexpr (SC != SC_CAPPED) mt = fmaxf(mt, st[t][r]);
            }
        float alpha = 1.0f;
        if constexpr (SC != SC_CAPPED) {
            mt = rows_max(mt);
            alpha = __builtin_amdgcn_exp2f(m - mt);
            m = mt;
            l *= alpha;
        }
        short8 pf;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(st[t][r] - m);
                l += p;
                pf[4 * t + r] = (short)f2bf(p);
            }
#pragma unroll
        for (int x = 0; x < DV / 16; ++x) {
            const int e = lane + 64 * x, r = e / (DV / 8), k = (e % (DV / 8)) * 8;
            *reinterpret_cast<uint4*>(&Vs[wave][r * VS + k]) = vr[x];
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's own rows: no barrier
        if (j0 + 128 < kend) gload(j0 + 128);
#pragma unroll
        for (int c = 0; c < DV / 16; ++c) {
            if constexpr (SC != SC_CAPPED) {
#pragma unroll
                for (int r = 0; r < 4; ++r) o[c][r] *= alpha;
            }
            uint16_t* vp = &Vs[wave][(4 * lg + (li >> 2)) * VS + c * 16 + 4 * (li & 3)];
            const s4v lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*)(vp));
            const s4v hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4v*)(vp + 16 * VS));
            const short8 vf = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
            o[c] = mfma16(vf, pf, o[c]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    l = rows_sum(l);
    if (lg == 0) { sml[wave][li][0] = m; sml[wave][li][1] = l; }
    __syncthreads();
    float M = kNone;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, sml[w][li][0]);
    const float f = __builtin_amdgcn_exp2f(m - M);
    float* os = reinterpret_cast<float*>(&Vs[0][0]);  // [wave][head][DV + 4], in place of the value rows
    constexpr int OS = DV + 4;
    static_assert(4 * 16 * OS * 4 <= 4 * 32 * VS * 2, "the sums fit the value rows");
#pragma unroll
    for (int c = 0; c < DV / 16; ++c)
        *reinterpret_cast<float4*>(os + (wave * 16 + li) * OS + c * 16 + 4 * lg) =
            make_float4(o[c][0] * f, o[c][1] * f, o[c][2] * f, o[c][3] * f);
    __syncthreads();
    for (int e = tid; e < nr * ep; e += 256) {
        const int r = e / ep, c = e % ep;
        float t = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) t += os[(w * 16 + r) * OS + c];
        part[(long)r * a.nsplit * rs + c] = t;
    }
    if (tid < nr) {
        float mm = kNone, ll = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) mm = fmaxf(mm, sml[w][tid][0]);
#pragma unroll
        for (int w = 0; w < 4; ++w) ll += sml[w][tid][1] * __builtin_amdgcn_exp2f(sml[w][tid][0] - mm);
        part[(long)tid * a.nsplit * rs + ep] = mm;
        part[(long)tid * a.nsplit * rs + ep + 1] = ll;
    }
}

// merge a head's partials: grid (H, B), nsplit <= 64.  A thread's values of the first AHEAD splits are asked for ahead of their weights,
// also an empty split's, which were never written and are not taken (each behind its weight: 9 trips to memory, 8 sequences of 16 heads 5.2 us, now 4.8)
template <typename T>
__global__ void __launch_bounds__(256) k_wattn_dc(WAttnDecodeArgs a) {
    __shared__ float wt[64];
    constexpr int AHEAD = 16;
    const int h = blockIdx.x, b = blockIdx.y, rs = a.hd.ep + 2, n = a.nsplit, lane = threadIdx.x & 63, E = a.hd.e;
    const float* p = a.part + ((long)b * a.hd.H + h) * n * rs;
    const float* pl = p + (long)min(lane, n - 1) * rs + a.hd.ep;
    const float ml = pl[0], ll = pl[1];
    float q[AHEAD];
    auto load = [&](int c, int s0) {
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) q[s] = p[(long)min(s0 + s, n - 1) * rs + min(c, E - 1)];
    };
    load(threadIdx.x, 0);
    asm volatile("" ::: "memory");
    {
        const float m = lane < n ? ml : kNone, l = lane < n ? ll : 0.0f;
        const float M = wave_max(l > 0.0f ? m : kNone);
        const float w = l > 0.0f ? exp2f(m - M) : 0.0f;
        const float L = wave_sum(l * w);
        if (threadIdx.x < 64) wt[lane] = w / L;
    }
    __syncthreads();
    T* o = reinterpret_cast<T*>(a.o) + (long)b * a.ldo;
    for (int c = threadIdx.x; c < E; c += 256) {
        float t = 0.0f;
        for (int s0 = 0; s0 < n; s0 += AHEAD) {
            if (s0 > 0 || c >= 256) load(c, s0);
#pragma unroll
            for (int s = 0; s < AHEAD; ++s) {
                const float w = s0 + s < n ? wt[s0 + s] : 0.0f;
                t = w > 0.0f ? fmaf(q[s], w, t) : t;
            }
        }
        stf(o + h * E + c, t);
    }
    if (h == a.hd.H - 1)
        for (int k = a.hd.H * E + threadIdx.x; k < a.ldo; k += 256) stf(o + k, 0.0f);
}

template <typename T, int RB, int SC>
void run_d(hipStream_t s, const WAttnDecodeArgs& a) {
    const WAttnHeads& w = a.hd;
    const size_t lds = (size_t)(w.H / w.G * w.dp + RB * DK + RB * 4 + 256 * 8) * sizeof(float);
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_wattn_d<T, RB, SC>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((k_wattn_d<T, RB, SC>), dim3(a.nsplit, w.G, a.B), dim3(256), lds, s, a);
    hipLaunchKernelGGL((k_wattn_dc<T>), dim3(w.H, a.B), dim3(256), 0, s, a);
}

template <int DQ, int DV>
void run_dm(hipStream_t s, const WAttnDecodeArgs& a) {
    const WAttnHeads& w = a.hd;
    const dim3 grid(a.nsplit, w.G * ((w.H / w.G + 15) / 16), a.B);
    const int mode = score_mode(a.sc);
    auto go = [&](auto heads) {
        constexpr int HEADS = decltype(heads)::value;
        if (mode == SC_BIAS) hipLaunchKernelGGL((k_wattn_dm<DQ, DV, SC_BIAS, HEADS>), grid, dim3(256), 0, s, a);
        else if (mode == SC_CAPPED) hipLaunchKernelGGL((k_wattn_dm<DQ, DV, SC_CAPPED, HEADS>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((k_wattn_dm<DQ, DV, SC_PLAIN, HEADS>), grid, dim3(256), 0, s, a);
    };
    if (w.d == DQ && w.e == DV) go(std::integral_constant<int, WHOLE>{});
    else if (w.d % 8 == 0 && w.e % 8 == 0) go(std::integral_constant<int, VECTORS>{});
    else go(std::integral_constant<int, ODD>{});
    if (!a.parts_only) hipLaunchKernelGGL((k_wattn_dc<uint16_t>), dim3(w.H, a.B), dim3(256), 0, s, a);
}
template <int DQ>
void run_dmv(hipStream_t s, const WAttnDecodeArgs& a) {
    if (a.hd.ep <= 64) run_dm<DQ, 64>(s, a);
    else if (a.hd.ep <= 128) run_dm<DQ, 128>(s, a);
    else run_dm<DQ, 256>(s, a);
}

template <typename T, int SC>
void decode_sc(hipStream_t s, const WAttnDecodeArgs& a) {
    const int R = a.hd.H / a.hd.G;
    if (R <= 1) run_d<T, 1, SC>(s, a);
    else if (R <= 2) run_d<T, 2, SC>(s, a);
    else if (R <= 4) run_d<T, 4, SC>(s, a);
    else run_d<T, 8, SC>(s, a);
}
template <typename T>
void decode_t(hipStream_t s, const WAttnDecodeArgs& a) {
    if (a.sc.r1) decode_sc<T, SC_BIAS>(s, a);
    else decode_sc<T, SC_PLAIN>(s, a);
}

template <typename T>
void plain_t(hipStream_t s, const WAttnArgs& a) {
    const size_t lds = (size_t)(a.hd.dp + 256 + 8) * sizeof(float);
    const dim3 grid(a.rows, a.hd.H);
    if (a.sc.r1) hipLaunchKernelGGL((k_wattn<T, SC_BIAS>), grid, dim3(256), lds, s, a);
    else hipLaunchKernelGGL((k_wattn<T, SC_PLAIN>), grid, dim3(256), lds, s, a);
}

}  // namespace

void wattn_append(hipStream_t s, Act act, const WAttnArgs& a) {
    if (act == ACT_F32) append_t<float>(s, a);
    else append_t<uint16_t>(s, a);
}

void wattn_prefill(hipStream_t s, Act act, const WAttnArgs& a) {
    const int dp = a.hd.dp, ep = a.hd.ep;
    if (act == ACT_F32) {
        const int n = std::max(dp, ep);
        if (n > 256) plain_t<float>(s, a);
        else if (n <= 64) run_f<64>(s, a);
        else if (n <= 128) run_f<128>(s, a);
        else run_f<256>(s, a);
    } else if (dp > 256 || ep > 256) {
        plain_t<uint16_t>(s, a);
    } else if (dp <= 64) {
        run_mv<64>(s, a);
    } else if (dp <= 96) {
        run_mv<96>(s, a);
    } else if (dp <= 128) {
        run_mv<128>(s, a);
    } else {
        run_mv<256>(s, a);
    }
}

int wattn_decode_splits(int B, int G, const WAttnScore& sc, int max_tokens) {
    const int span = (int)std::max(1L, std::min((long)sc.window + sc.keep, (long)max_tokens));
    const int tiles = (span + 127) / 128;
    int n = (1024 + B * G - 1) / (B * G);
    return std::max(1, std::min(std::min(n, tiles), 64));
}

size_t wattn_decode_floats(int B, int H, int ep, int nsplit) { return (size_t)B * H * nsplit * (ep + 2); }

void wattn_decode(hipStream_t s, Act act, const WAttnDecodeArgs& a) {
    const int dp = a.hd.dp, ep = a.hd.ep;
    if (act == ACT_F32) decode_t<float>(s, a);
    else if (dp > 256 || ep > 256) decode_t<uint16_t>(s, a);
    else if (dp <= 64) run_dmv<64>(s, a);
    else if (dp <= 128) run_dmv<128>(s, a);
    else run_dmv<256>(s, a);
}

}  // namespace pgmi
