// kernels_matmul.hip -- matrix products of the layered decoders: any M and N, K a multiple of 8.
//
// bf16 activations run on the prefill GEMM kernels (kernels_gemm.hip: LDS-DMA panel, warp-specialised and 8-phase
// forms), a few instantiations chosen by shape; fp32 activations on tile_f32.h's exact split over the same matrix units.
// Weights are bf16 [N][ldw] in both.
#define PGMI_GEMM_KERNELS_ONLY
#include "kernels_gemm.hip"

#include <algorithm>

#include "act.h"
#include "decoder.h"
#include "plan.h"
#include "tile_f32.h"

namespace pgmi {

namespace {

// ---------------------------------------------------------------- fp32
struct F32Args {
    const float* A;
    int lda;
    const uint16_t* W;
    int ldw, M, N, K;
    const uint16_t* bias;
    float* out;
    int ldo;  // columns; N .. ldo-1 are written as zeros
    int per;  // 64-deep steps of a K slice, one slab [M][ldo] each
};

// grid (row tiles x column tiles, K slices), the row tiles of a column tile adjacent.  NB = 2: gate and up columns, silu(gate)
// up stored.
template <int WM, int WN, int TM, int TN, int NB>
__global__ void __launch_bounds__(64 * WM * WN) k_matmul_f32(F32Args a) {
    constexpr int BM = 16 * WM * TM, BN = 16 * WN * TN;
    const int n_mt = (a.M + BM - 1) / BM, m0 = blockIdx.x % n_mt * BM, n0 = blockIdx.x / n_mt * BN;
    const int k0 = blockIdx.y * a.per * 64, k1 = min(a.K, k0 + a.per * 64);
    float* out = a.out + (long)blockIdx.y * a.M * a.ldo;
    tile_f32<WM, WN, TM, TN, NB>(
        a.A, a.lda, a.W, a.ldw, (long)a.N * a.ldw, a.N, a.ldo, n0, k0, k1, [&](int m) { return min(m0 + m, a.M - 1); },
        [&](int n) {
            if constexpr (NB == 2) return 0.0f;
            else return a.bias ? bf2f(a.bias[min(n, a.N - 1)]) : 0.0f;
        },
        [&](int m, int n, float v, float u, float b) {
            if (m0 + m >= a.M) return;
            if constexpr (NB == 2) v = siluf_(v) * u;
            else if (a.bias) v += b;
            out[(long)(m0 + m) * a.ldo + n] = n < a.N ? v : 0.0f;
        });
}

template <int WM, int WN, int TM, int TN, int NB>
void run_f32(hipStream_t s, const F32Args& a, int split) {
    constexpr int BM = 16 * WM * TM, BN = 16 * WN * TN;
    constexpr size_t lds = tile_f32_lds(BM, BN, NB);
    static const bool once = [] {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(&k_matmul_f32<WM, WN, TM, TN, NB>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    }();
    (void)once;
    hipLaunchKernelGGL((k_matmul_f32<WM, WN, TM, TN, NB>), dim3((a.M + BM - 1) / BM * ((a.ldo + BN - 1) / BN), split),
                       dim3(64 * WM * WN), lds, s, a);
}

// zeros in columns N .. ldo-1 (the GEMM kernels write columns < N only)
__global__ void k_zero_cols(uint16_t* __restrict__ out, int M, int N, int ldo) {
    const int w = ldo - N;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < (long)M * w; i += gridDim.x * 256L)
        out[i / w * ldo + N + i % w] = 0;
}

// ---------------------------------------------------------------- bf16
template <auto KERN>
void lds_attr(size_t lds) {
    static bool done = false;
    if (!done && lds > 64 * 1024) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(KERN), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        done = true;
    }
}

struct Job {
    hipStream_t s;
    const uint16_t* A;
    int lda;
    const uint16_t* W;
    int ldw, M, N, K;
    EpiArgs ea;
    float* ws;
    int split;
    long up;
    int per() const {
        const int nkt = (K + 63) / 64;
        return (nkt + split - 1) / split;
    }
};

// 32 TM x 64 tiles (dual: 32 + 32 columns)
template <int TM, int EPI, bool SPLIT>
void run_p(const Job& j) {
    constexpr int NB = epi_dual(EPI) ? 2 : 1, TN = NB == 2 ? 1 : 2, ST = 4;
    constexpr int BM = 32 * TM, BN = 2 * TN * 16;
    constexpr size_t lds = (size_t)ST * (BM + NB * BN) * 128;
    const int n_mt = (j.M + BM - 1) / BM, n_nt = (j.N + BN - 1) / BN;
    lds_attr<&k_gemm_p<4, 2, TM, TN, NB, ST, EPI, SPLIT>>(lds);
    hipLaunchKernelGGL((k_gemm_p<4, 2, TM, TN, NB, ST, EPI, SPLIT>), dim3(n_mt * n_nt, j.split), dim3(256), lds, j.s, j.A,
                       j.lda, j.W, j.ldw, j.M, j.N, j.K, j.per(), j.ea, j.ws, j.up, n_mt, 0);
}

// 128 x 128 tiles, loader waves (dual: 128 x 64 + 64)
template <int EPI, bool SPLIT>
void run_w128(const Job& j) {
    constexpr int NB = epi_dual(EPI) ? 2 : 1, TN = NB == 2 ? 1 : 2, ST = 4;
    constexpr int BM = 128, BN = 4 * TN * 16;
    constexpr size_t lds = (size_t)ST * (BM + NB * BN) * 128;
    const int n_mt = (j.M + BM - 1) / BM, n_nt = (j.N + BN - 1) / BN;
    lds_attr<&k_gemm_w<8, 2, 4, TN, NB, ST, 4, EPI, SPLIT>>(lds);
    hipLaunchKernelGGL((k_gemm_w<8, 2, 4, TN, NB, ST, 4, EPI, SPLIT>), dim3(n_mt * n_nt, j.split), dim3(64 * 12), lds, j.s,
                       j.A, j.lda, j.W, j.ldw, j.M, j.N, j.K, j.per(), j.ea, j.ws, j.up, n_mt, n_mt == 1 ? 1 << 30 : 0);
}

// 32 TM x 256 tiles, 8 phases (dual: 128 + 128 columns); K % 64 == 0
template <int TM, int EPI, bool SPLIT>
void run_8p(const Job& j) {
    constexpr int BM = 32 * TM, BN = epi_dual(EPI) ? 128 : 256;
    constexpr size_t lds = lds_8p(TM);
    const int n_mt = (j.M + BM - 1) / BM, n_nt = (j.N + BN - 1) / BN;
    lds_attr<&k_gemm_8p<TM, EPI, SPLIT>>(lds);
    hipLaunchKernelGGL((k_gemm_8p<TM, EPI, SPLIT>), dim3(n_mt * n_nt, j.split), dim3(512), lds, j.s, j.A, j.lda, j.W, j.ldw,
                       j.M, j.N, j.K, j.per(), j.ea, j.ws, j.up, n_mt, 0);
}

long tiles(int M, int N, int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); }

// The form with the least predicted time (plan.h, whose forms are the same kernels but for the height of their ring).
// slab_bytes > 0: into slabs, K cut as the form gains from it; the pass that follows reads every slab, 0.25 us per MB past the
// first one, which it reads of a whole product too (gemm_plan.hip's readers take bf16 rows where a product is whole, behind
// fixed work of their own: another price).  Before, K slices were counted in 64 x 64 tiles and three tile shapes had fixed borders.  1,540 rows,
// us before / now: 2048 columns of K = 16384 123 / 97 (three slices), 6144 of 2048 48.3 / 41.0, 2560 of 2048 39.4 / 30.6,
// 4096 of 128 12.2 / 10.5.
template <int EPI, bool SPLIT>
void run_plan(Job& j, size_t slab_bytes) {
    const float mb = 4e-6f * (float)j.M * (float)j.N;
    const TileChoice t = choose_form(j.M, j.N, j.K, epi_dual(EPI), slab_bytes ? 8 : 1, [&](const TileForm& f, int split) {
        if (f.cfg == R288w || f.cfg == W288n || f.cfg == W64x64 || f.cfg == W128x64) return -1.0f;  // not instantiated here
        if (split > 1 && (size_t)split * j.M * j.N * sizeof(float) > slab_bytes) return -1.0f;
        return 0.25f * mb * (float)(split - 1);
    });
    j.split = t.split;
    switch (t.form->cfg) {
        case P32x64s4: run_p<1, EPI, SPLIT>(j); break;
        case P96x64s4: run_p<3, EPI, SPLIT>(j); break;
        case W128x128: run_w128<EPI, SPLIT>(j); break;
        case E128: run_8p<4, EPI, SPLIT>(j); break;
        case E160: run_8p<5, EPI, SPLIT>(j); break;
        case E192: run_8p<6, EPI, SPLIT>(j); break;
        case E224: run_8p<7, EPI, SPLIT>(j); break;
        case E256: run_8p<8, EPI, SPLIT>(j); break;
        default: run_p<2, EPI, SPLIT>(j); break;
    }
}

// K slices for a product whose t tiles alone leave CUs idle
int pick_split(long t, int want, int M, int N, int K, size_t out_bytes) {
    const int nkt = (K + 63) / 64;
    int split = 1;
    while (t * split < want && split < 8 && nkt / (split * 2) >= 4) split *= 2;
    while (split > 1 && (size_t)split * M * N * sizeof(float) > out_bytes) split /= 2;
    if (split > 1) {  // every slice non-empty
        const int per = (nkt + split - 1) / split;
        split = (nkt + per - 1) / per;
    }
    return split;
}

}  // namespace

int matmul_rt(hipStream_t s, Act act, const void* A, int lda, const uint16_t* W, int ldw, int M, int N, int K,
              RtOut mode, const uint16_t* bias, void* out, int ldo, size_t out_bytes) {
    if (M <= 0 || N <= 0) return 1;
    if (act == ACT_F32) {
        const bool plain = mode == RT_F32 || mode == RT_SLABS;
        F32Args f{reinterpret_cast<const float*>(A), lda, W, ldw, M, N, K, plain ? nullptr : bias, reinterpret_cast<float*>(out),
                  plain ? N : ldo, (K + 63) / 64};
        // 64 x 128 tiles of 8 waves once they fill the chip, else 32 x 64 tiles of 4 waves, which more workgroups share.
        // Measured, us: 500 x 1024, K = 4096: 20.9 (4 slices) against 22.1; 500 x 4096, K = 1024: 20.9 / 26.7;
        // 300 x 1024, K = 1024: 17.2 / 10.4
        int split = 1;
        auto cut = [&](int bm, int bn, int want) {
            const long t = tiles(M, f.ldo, bm, bn);
            if (mode == RT_SLABS) split = pick_split(t, want, M, N, K, out_bytes);
            f.per = ((K + 63) / 64 + split - 1) / split;
            return t * split;
        };
        if (cut(64, 128, 256) >= 256) {
            if (mode == RT_SWIGLU) run_f32<2, 4, 2, 2, 2>(s, f, 1);
            else run_f32<2, 4, 2, 2, 1>(s, f, split);
        } else {
            cut(32, 64, 512);
            if (mode == RT_SWIGLU) run_f32<1, 4, 2, 1, 2>(s, f, 1);
            else run_f32<1, 4, 2, 1, 1>(s, f, split);
        }
        return split;
    }
    Job j{s, reinterpret_cast<const uint16_t*>(A), lda, W, ldw, M, N, K, {}, nullptr, 1, 0};
    if (mode == RT_F32 || mode == RT_SLABS) {
        j.ws = reinterpret_cast<float*>(out);
        run_plan<EPI_STORE, true>(j, mode == RT_SLABS ? out_bytes : 0);
        return j.split;
    }
    j.ea.out = reinterpret_cast<uint16_t*>(out);
    j.ea.ldo = ldo;
    j.ea.bias = bias;
    if (mode == RT_SWIGLU) {
        j.up = (long)N * ldw;
        run_plan<EPI_SWIGLU, false>(j, 0);
    } else if (bias) {
        run_plan<EPI_BIAS, false>(j, 0);
    } else {
        run_plan<EPI_STORE, false>(j, 0);
    }
    if (ldo > N && ldo - N < 8)
        hipLaunchKernelGGL(k_zero_cols, dim3(256), dim3(256), 0, s, reinterpret_cast<uint16_t*>(out), M, N, ldo);
    return 1;
}

}  // namespace pgmi
