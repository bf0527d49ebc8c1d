// gemm_plan.hip -- the plan of a prefill product (kernels_gemm.hip): chosen by predicted time (plan.h), or forced by the
// tuning hooks (host code only).
#include <algorithm>

#include "launch.h"
#include "plan.h"

namespace pgmi {

static_assert(kNumCfg == kGemmCfgs, "launch.h kGemmCfgs");

static int g_force_cfg = -1, g_force_split = 0;  // tuning override (pgmi_tune_gemm)

void gemm_force_plan(int cfg, int split) {
    g_force_cfg = cfg;
    g_force_split = split;
}

// per-shape plan overrides (tuning hook pgmi_tune_gemm_shape): in-situ sweeps of one GEMM of a
// forward while the others keep their measured plans
struct ShapePlan {
    int M, N, K;
    bool dual;
    int cfg, split;
};
static ShapePlan g_shape_plans[16];
static int g_n_shape_plans = 0;

int gemm_force_shape(int M, int N, int K, int dual, int cfg, int split) {
    for (int i = 0; i < g_n_shape_plans; ++i)
        if (g_shape_plans[i].M == M && g_shape_plans[i].N == N && g_shape_plans[i].K == K &&
            g_shape_plans[i].dual == (dual != 0)) {
            g_shape_plans[i] = g_shape_plans[--g_n_shape_plans];
            break;
        }
    if (cfg < 0) return 0;
    if (g_n_shape_plans >= 16) return -1;
    g_shape_plans[g_n_shape_plans++] = {M, N, K, dual != 0, cfg, split < 1 ? 1 : split};
    return 0;
}

static bool rope_form(int cfg) {
    return cfg == P32x64s4 || cfg == P64x64s4 || cfg == P96x64s4 || cfg == W64x64 || cfg == W128x64 || cfg == W128x128;
}

Plan gemm_plan(int M, int N, int K, bool dual, After after, size_t ws_bytes) {
    if (g_force_cfg >= 0) return {(Cfg)g_force_cfg, !dual && g_force_split > 0 ? g_force_split : 1};
    for (int i = 0; i < g_n_shape_plans; ++i) {
        const ShapePlan& o = g_shape_plans[i];
        if (o.M == M && o.N == N && o.K == K && o.dual == dual) return {(Cfg)o.cfg, dual ? 1 : o.split};
    }
    // lock-step decode batches as GEMMs (M <= 16 rows; in isolation: gate|up 64x128 tiles 24.2 us, down 64x64
    // split 8 18.1 us)
    if (M <= 16 && dual) return {P64x128, 1};
    if (M <= 16 && K >= 8192) return {P64x64, 8};
    const float mb = 4e-6f * M * N;
    const bool slabs = !dual && N % 4 == 0;  // the slabs' readers take 4 outputs per thread
    const TileChoice t = choose_form(M, N, K, dual, slabs ? 8 : 1, [&](const TileForm& f, int s) {
        if (dual && f.cfg == W288n) return -1.0f;
        if (s > 1 && (size_t)s * M * N * sizeof(float) > ws_bytes) return -1.0f;
        // reading slabs: 0.25 us per MB past what a norm kernel's fixed 5 us hide, less of few rows, whose workgroups are
        // all there at once (288 x 2048 of 8 slices 6.2 us; 1056 x 2048 unsplit 5.2, of 2 slices 8.3; 2048 x 1152
        // unsplit 5.4, of 3 slices 10.8)
        const float read = s > 1 ? std::max(0.0f, 0.25f * mb * s - 2.0f) * std::min(1.0f, M / 700.0f) : 0.0f;
        if (after == AFTER_NORM) return read;
        if (after == AFTER_OWN) return s > 1 ? read + 4.6f : 0.0f;
        // RoPE in the epilogue: 288 rows + 1.5 us (+ 3.3 where the waves that multiply also load), 1056 + 4; k_rope_kv 6.3 at
        // 288, 8.1 at 2304
        if (s == 1 && rope_form(f.cfg)) return 0.8f + 0.003f * M + (f.cfg >= W64x64 ? 0.0f : 2.6f);
        return read + 6.0f + 0.001f * M;
    });
    return {(Cfg)t.form->cfg, t.split};
}

}  // namespace pgmi
