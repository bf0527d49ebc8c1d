// plan.h -- the tiles and the K slices of a bf16 product C[M,N] = A . W^T, chosen by predicted time (host only).
//
// A form's time is c + R (a + b n): n the 64-deep k-tiles of a slice, R the rounds of its workgroups over the chip, of
// which a round that is not full takes lo + (1 - lo) of its share (the workgroups that are there run faster, not in
// proportion).  c, a, b and lo (us) were set on MI355X from launches with cold weights: M 32 .. 4608 at 27 (N, K) of this
// library's layers, K slices.  tools/plan_fit.py times such launches, holds the constants against them and fits them again;
// 19,281 of its times are in profiles/gemm_plan_sweep.csv.gz.  Over these the constants are off by 8 % (E128) to 24 % (W64x64)
// of a time on average, and the form chosen, the price of its slabs included, is 2.2 % (layered decoders) to 3.2 % slower than
// the best of 702 shapes' measured forms, 16 to 22 % over the tenth of the shapes where it does worst: K of 64 and 128, few
// tiles of long K, and rows that are no multiple of 128 bytes (K = 4304), whose k-tiles take 1.3 to 1.5 b where those of both
// operands are (the vision tower's activations lie 4,352 apart).
// What it replaced, plans listed for the shapes of one photo of each size and of eight with one rule for all others:
// 576 rows, 16384 gate and up columns of K = 2048: 110 us, here 74; 640: 110 / 90; 1280: 190 / 143; 512 rows of q|k|v
// (3456 columns of K = 1152): 25 / 11; prompts of 2 .. 7 photos 1.21 - 1.33x faster, of one with another text 1.1 - 1.2x.
// (One listed plan was better: 256 rows, 1152 columns of K = 4304, P96x64s4 in four slices 12.5 us, here P64x64s4 in three
// 13.3; the tower of one 224 px photo 1,442 -> 1,461 us, the photo's whole call 3,759 -> 3,727.)
#pragma once
#include <stddef.h>

#include <algorithm>

namespace pgmi {

// Tile configurations (wave grid, per-wave MFMA tiles).  BM = WGM*TM*16, BN = WGN*TN*16.  The rule takes those of kTileForms
// below and, up to 16 rows, P64x64 and P64x128; the others are there for the tuning hooks (pgmi_tune_gemm*), which name a
// configuration by its number here.
enum Cfg : int {
    C288x64 = 0,   // 6x1 waves, 3x4 tiles  (text rows: M = 288 = 18 x 16)
    C288x32 = 1,   // 6x1 waves, 3x2 tiles
    C256x64 = 2,   // 4x1 waves, 4x4 tiles  (vision rows: M = 256)
    C256x32 = 3,   // 4x1 waves, 4x2 tiles
    C128x128 = 4,  // 2x2 waves, 4x4 tiles  (large M)
    C128x64 = 5,   // 2x2 waves, 4x2 tiles
    // panel GEMM (k_gemm_p, LDS-DMA ring): BM x BN output columns (dual gate/up: BN/2 columns x 2)
    P288w = 6,     // TM 9,  BN 128, 3 slots
    P256w = 7,     // TM 8,  BN 128, 3 slots
    P352w = 8,     // TM 11, BN 128, 2 slots  (448 px text rows: M = 1056 = 3 x 352)
    P288n = 9,     // TM 9,  BN 64,  3 slots
    P256n = 10,    // TM 8,  BN 64,  3 slots
    P128w = 11,    // TM 4,  BN 128, 3 slots
    P288t = 12,    // TM 9,  BN 32,  4 slots  (2x2 waves, 1 column fragment each)
    P256t = 13,    // 4x1 waves, TM 4, BN 32, 4 slots
    P64x64 = 14,   // TM 2, BN 64,  6 slots   (small GEMMs: every CU busy, little A per CU)
    P128x64 = 15,  // TM 4, BN 64,  6 slots
    P64x128 = 16,  // TM 2, BN 128, 6 slots
    P128x128 = 17, // TM 4, BN 128, 5 slots
    P64x64d = 18,  // TM 2, BN 64,  10 slots
    P128x64d = 19, // 4x1 waves, TM 2, BN 64, 6 slots
    // 8 waves (2 per SIMD: one wave's LDS-DMA issue stalls overlap its partner's MFMAs)
    Q288w = 20,    // 2x4 waves, TM 9,  BN 128, 3 slots
    Q352w = 21,    // 2x4 waves, TM 11, BN 128, 2 slots
    Q256w = 22,    // 2x4 waves, TM 8,  BN 128, 3 slots
    Q288x256 = 23, // 2x4 waves, TM 9,  BN 256, 2 slots
    // shallow rings (2-3 workgroups per CU: more k-tiles in flight per CU for the small GEMMs)
    P64x64s3 = 24, // TM 2, BN 64, 3 slots
    P64x64s4 = 25, // TM 2, BN 64, 4 slots
    P32x64s4 = 26, // TM 1, BN 64, 4 slots
    P64x32s4 = 27, // TM 2, BN 32, 4 slots
    P96x64s4 = 28, // TM 3, BN 64, 4 slots (M = 288 = 3 x 96)
    P96x64s3 = 29, // TM 3, BN 64, 3 slots
    // warp-specialised (k_gemm_w): compute waves + 4 LDS-DMA loader waves
    W288w = 30,    // 2x4 compute waves, TM 9,  BN 128, 3 slots
    W288n = 31,    // 2x4 compute waves, TM 9,  BN 64,  3 slots
    W64x64 = 32,   // 2x2 compute waves, TM 2,  BN 64,  6 slots
    W352w = 33,    // 2x4 compute waves, TM 11, BN 128, 2 slots
    W128x128 = 34, // 2x4 compute waves, TM 4,  BN 128, 4 slots
    W128x64 = 35,  // 2x2 compute waves, TM 4,  BN 64,  5 slots
    // 8-phase (k_gemm_8p): 2x4 waves, BN 256 (dual: 128 gate + 128 up), two K-tile buffers
    E256 = 36,     // TM 8: 256 rows
    E192 = 37,     // TM 6: 192 rows
    // k_gemm_w's in-wave reload mode (W288w's tiles; bit-identical results)
    R288w = 38,    // 2x4 compute waves, TM 9, BN 128 (dual 64 + 64), 3 slots
    // 8-phase, further heights
    E128 = 39,     // TM 4: 128 rows
    E160 = 40,     // TM 5: 160 rows
    E224 = 41,     // TM 7: 224 rows
    kNumCfg = 42,
};

struct Plan {
    Cfg cfg;
    int split;
};

struct TileForm {
    int cfg;
    int bm, bn;       // rows and columns of a tile (gate and up: bn / 2 of each)
    int per_cu;       // workgroups of one round on a CU
    bool whole_k;     // needs K % 64 == 0 and a k-tile
    float c, a, b, lo;
};

// (W288n's gate and up tiles are R288w's, and R288w is the faster of the two)
constexpr TileForm kTileForms[] = {
    {R288w, 288, 128, 1, false, 4.32f, 7.07f, 0.935f, 0.50f},
    {W288n, 288, 64, 1, false, 3.30f, 7.59f, 0.637f, 0.69f},
    {P32x64s4, 32, 64, 3, false, 3.05f, 2.62f, 0.440f, 0.21f},
    {P64x64s4, 64, 64, 1, false, 3.69f, 1.22f, 0.210f, 0.74f},
    {P96x64s4, 96, 64, 1, false, 5.11f, 1.14f, 0.260f, 0.72f},
    {W64x64, 64, 64, 1, false, 3.17f, 5.21f, 0.192f, 0.66f},
    {W128x64, 128, 64, 1, false, 1.69f, 5.85f, 0.333f, 0.78f},
    {W128x128, 128, 128, 1, false, 2.63f, 6.42f, 0.464f, 0.82f},
    {E128, 128, 256, 1, true, 3.00f, 6.66f, 0.798f, 0.77f},
    {E160, 160, 256, 1, true, 4.75f, 6.63f, 0.954f, 0.81f},
    {E192, 192, 256, 1, true, 2.61f, 7.00f, 1.138f, 0.95f},
    {E224, 224, 256, 1, true, 8.85f, 4.83f, 1.293f, 0.76f},
    {E256, 256, 256, 1, true, 1.78f, 12.13f, 1.373f, 0.85f},
};

struct TileChoice {
    const TileForm* form;
    int split;
    float us;
};

inline long form_tiles(const TileForm& f, int M, int N, bool dual) {
    const int bn = dual ? f.bn / 2 : f.bn;
    return (long)((M + f.bm - 1) / f.bm) * ((N + bn - 1) / bn);
}

// (K = 0, the epilogue of empty sums, is planned as one k-tile)
inline int k_tiles(int K) { return std::max(1, (K + 63) / 64); }

inline float form_us(const TileForm& f, int M, int N, int K, int split, bool dual) {
    const int nkt = k_tiles(K), per = (nkt + split - 1) / split;
    const long t = form_tiles(f, M, N, dual) * ((nkt + per - 1) / per), slots = 256L * f.per_cu;
    const long rest = t % slots;
    const float r = (float)(t / slots) + (rest ? f.lo + (1.0f - f.lo) * (float)rest / (float)slots : 0.0f);
    return f.c + r * (f.a + f.b * (float)per);
}

// the least form_us + extra(form, slices) over the forms and slices, of four k-tiles or more on average (the last one takes what
// is left); extra < 0: not to be taken
template <class Extra>
TileChoice choose_form(int M, int N, int K, bool dual, int max_split, Extra extra) {
    TileChoice best{nullptr, 1, 0.0f};
    const int nkt = k_tiles(K);
    for (const TileForm& f : kTileForms) {
        if (f.whole_k && (K % 64 != 0 || K < 64)) continue;
        for (int s = 1; s <= max_split && (s == 1 || nkt / s >= 4); ++s) {
            if ((nkt + (nkt + s - 1) / s - 1) / ((nkt + s - 1) / s) != s) continue;  // a slice would be empty
            const float x = extra(f, s);
            if (x < 0.0f) continue;
            const float us = form_us(f, M, N, K, s, dual) + x;
            if (!best.form || us < best.us) best = {&f, s, us};
        }
    }
    return best;
}

// Bytes for the K slabs of a layered decoder's step of these rows, `one` slab of the widest product being rows x n fp32: four of them
// up to 160 MB, as many as the rule above gains from; at the least one, and 32 MB for steps of few rows.
inline size_t slab_least(int rows, int n) { return std::max((size_t)rows * n * 4, (size_t)32 << 20); }
inline size_t slab_room(int rows, int n) {
    return std::max(slab_least(rows, n), std::min((size_t)rows * n * 16, (size_t)160 << 20));
}
// takes the room, or where the device does not have it the least, by alloc(bytes): the bytes taken, 0 if neither is there
template <class Alloc>
size_t take_slabs(int rows, int n, Alloc alloc) {
    const size_t room = slab_room(rows, n), least = slab_least(rows, n);
    if (alloc(room)) return room;
    return least < room && alloc(least) ? least : 0;
}

// what follows a product: its own epilogue (K slices need k_splitk_epi's launch), a residual + norm kernel that reads
// slabs as readily as rows, or RoPE + KV append (in the epilogue of some forms, else k_rope_kv)
enum After { AFTER_OWN, AFTER_NORM, AFTER_ROPE };
Plan gemm_plan(int M, int N, int K, bool dual, After after, size_t ws_bytes);

}  // namespace pgmi
