// common.h -- shared device helpers for libpgmi (gfx950 / CDNA4 only).
//
// bf16 is carried as raw uint16 bit patterns; all arithmetic is fp32 with an
// explicit round-to-nearest-even back to bf16 exactly where the reference's bf16
// PyTorch modules round (their bf16 outputs).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pgmi {

typedef uint16_t bf16_t;
typedef short short8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

struct alignas(16) u16x8 { uint16_t v[8]; };

__device__ __forceinline__ float bf2f(uint16_t b) {
    return __uint_as_float(((uint32_t)b) << 16);
}

// round-to-nearest-even f32 -> bf16: one v_cvt_pk_bf16_f32 on gfx950 (the integer form
// u + 0x7FFF + ((u >> 16) & 1) took four VALU ops per element; same result for finite inputs, and a
// NaN stays a NaN -- MI355X_MICROARCH.md, correctness boundaries)
__device__ __forceinline__ uint16_t f2bf(float f) {
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}

__device__ __forceinline__ float rbf(float f) { return bf2f(f2bf(f)); }

// gelu(approximate="tanh") in fp32 (torch: 0.5*x*(1+tanh(sqrt(2/pi)*(x+0.044715*x^3)))), as the
// identity 0.5*(1+tanh(u)) = 1/(1+exp(-2u)): one v_exp_f32 and one v_rcp_f32 (a few fp32 ulp, far
// below the bf16 rounding that follows every use) instead of the library tanhf, whose branches and
// division made the GELU epilogues of the fc1 / gate|up GEMMs cost up to a third of the kernel.
// exp(-2u) overflowing to +inf gives x * 0 = -0 (gelu of a large negative x).
__device__ __forceinline__ float gelu_tanh(float x) {
    const float k = 0.7978845608028654f;
    const float u = k * (x + 0.044715f * x * x * x);
    const float e = __builtin_amdgcn_exp2f(u * -2.8853900817779268f);  // exp(-2u) = 2^(-2u log2 e)
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// Values joined across lanes by the vector unit's own lane moves (DPP within 16 lanes, the row swaps past them): a step is one or two
// instructions.  By ds_bpermute (what __shfl_xor becomes) it is a round trip through LDS of some 100 cycles, six of them for a
// wave's sum, which nothing hides in a kernel of a few us (a small model's step 296 -> 280 us, a reply 1,071 -> 1,050).  op is
// commutative, so the tree is the butterfly's and its results are __shfl_xor's to the bit.
// (8-byte values: both halves.)
typedef int i32x2 __attribute__((ext_vector_type(2)));
template <int CTRL, typename T>
__device__ __forceinline__ T lane_move(T v) {
    if constexpr (sizeof(T) == 8) {
        i32x2 h = __builtin_bit_cast(i32x2, v);
        h.x = lane_move<CTRL>((int)h.x);
        h.y = lane_move<CTRL>((int)h.y);
        return __builtin_bit_cast(T, h);
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
    }
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppRor4 = 0x124, kDppRor8 = 0x128;
// with lane ^ 16, with lane ^ 32: the swapped pair is (the lower row's, the upper row's) in both rows
template <typename T, typename Op>
__device__ __forceinline__ T join_xor16(T v, Op op) {
    if constexpr (sizeof(T) == 8) {
        const i32x2 u = __builtin_bit_cast(i32x2, v);
        const auto x = __builtin_amdgcn_permlane16_swap((unsigned)u.x, (unsigned)u.x, false, false);
        const auto y = __builtin_amdgcn_permlane16_swap((unsigned)u.y, (unsigned)u.y, false, false);
        return op(__builtin_bit_cast(T, i32x2{(int)x[0], (int)y[0]}), __builtin_bit_cast(T, i32x2{(int)x[1], (int)y[1]}));
    } else {
        const unsigned u = __builtin_bit_cast(unsigned, v);
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        return op(__builtin_bit_cast(T, (unsigned)r[0]), __builtin_bit_cast(T, (unsigned)r[1]));
    }
}
template <typename T, typename Op>
__device__ __forceinline__ T join_xor32(T v, Op op) {
    if constexpr (sizeof(T) == 8) {
        const i32x2 u = __builtin_bit_cast(i32x2, v);
        const auto x = __builtin_amdgcn_permlane32_swap((unsigned)u.x, (unsigned)u.x, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap((unsigned)u.y, (unsigned)u.y, false, false);
        return op(__builtin_bit_cast(T, i32x2{(int)x[0], (int)y[0]}), __builtin_bit_cast(T, i32x2{(int)x[1], (int)y[1]}));
    } else {
        const unsigned u = __builtin_bit_cast(unsigned, v);
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return op(__builtin_bit_cast(T, (unsigned)r[0]), __builtin_bit_cast(T, (unsigned)r[1]));
    }
}
// all 64 lanes, from lane ^ 32 down to lane ^ 1 (behind ^ 8 a row's halves are alike: a turn by 4 is ^ 4)
template <typename T, typename Op>
__device__ __forceinline__ T wave_join(T v, Op op) {
    v = join_xor16(join_xor32(v, op), op);
    v = op(v, lane_move<kDppRor8>(v));
    v = op(v, lane_move<kDppRor4>(v));
    v = op(v, lane_move<kDppXor2>(v));
    return op(v, lane_move<kDppXor1>(v));
}
// groups of N lanes (a power of two), from lane ^ 1 up to lane ^ N / 2 (behind ^ 2 four lanes are alike: a mirrored half row is ^ 4)
template <int N, typename T, typename Op>
__device__ __forceinline__ T lanes_join(T v, Op op) {
    if constexpr (N > 1) v = op(v, lane_move<kDppXor1>(v));
    if constexpr (N > 2) v = op(v, lane_move<kDppXor2>(v));
    if constexpr (N > 4) v = op(v, lane_move<kDppHalfMirror>(v));
    if constexpr (N > 8) v = op(v, lane_move<kDppRor8>(v));
    if constexpr (N > 16) v = join_xor16(v, op);
    if constexpr (N > 32) v = join_xor32(v, op);
    return v;
}
// groups of n lanes, n a power of two known to the whole wave
template <typename T, typename Op>
__device__ __forceinline__ T lanes_join_n(T v, int n, Op op) {
    if (n > 1) v = op(v, lane_move<kDppXor1>(v));
    if (n > 2) v = op(v, lane_move<kDppXor2>(v));
    if (n > 4) v = op(v, lane_move<kDppHalfMirror>(v));
    if (n > 8) v = op(v, lane_move<kDppRor8>(v));
    if (n > 16) v = join_xor16(v, op);
    if (n > 32) v = join_xor32(v, op);
    return v;
}
// inclusive sums over the wave's lanes (lanes that a move finds nothing for add 0)
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T lane_before(T v) {
    if constexpr (sizeof(T) == 8) {
        const i32x2 h = __builtin_bit_cast(i32x2, v);
        return __builtin_bit_cast(T, i32x2{lane_before<CTRL, ROWS>((int)h.x), lane_before<CTRL, ROWS>((int)h.y)});
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROWS, 0xF, false));
    }
}
template <typename T>
__device__ __forceinline__ T wave_scan(T v) {
    v += lane_before<0x111, 0xF>(v);  // the lane before, in a row of 16
    v += lane_before<0x112, 0xF>(v);
    v += lane_before<0x114, 0xF>(v);
    v += lane_before<0x118, 0xF>(v);
    v += lane_before<0x142, 0xA>(v);  // a row's last lane to the next row: rows 1 and 3
    v += lane_before<0x143, 0xC>(v);  // lane 31 to rows 2 and 3
    return v;
}
// a bf16 that lane `lane` of the wave holds in an int, in every lane.  That lane has to be on: behind a branch it was not in, the register
// that it is read from may not be the one it was written to
__device__ __forceinline__ float of_lane(int bf, int lane) { return __uint_as_float((unsigned)__builtin_amdgcn_readlane(bf, lane) << 16); }
struct SumOp {
    template <typename T>
    __device__ __forceinline__ T operator()(T a, T b) const { return a + b; }
};
struct MaxOp {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};

__device__ __forceinline__ float wave_sum(float v) { return wave_join(v, SumOp{}); }
__device__ __forceinline__ float wave_max(float v) { return wave_join(v, MaxOp{}); }
// over the 4 lanes of one place in a row of 16: ^ 16, then ^ 32
__device__ __forceinline__ float rows_sum(float v) { return join_xor32(join_xor16(v, SumOp{}), SumOp{}); }
__device__ __forceinline__ float rows_max(float v) { return join_xor32(join_xor16(v, MaxOp{}), MaxOp{}); }

// 8 bf16 (16 B) dot 8 bf16 with fp32 accumulation via v_dot2_f32_bf16
__device__ __forceinline__ float dot8(const uint4 a, const uint4 b, float acc) {
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a.x), __builtin_bit_cast(bf16x2, b.x), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a.y), __builtin_bit_cast(bf16x2, b.y), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a.z), __builtin_bit_cast(bf16x2, b.z), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a.w), __builtin_bit_cast(bf16x2, b.w), acc, false);
    return acc;
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint4 ldg_nt(const void* p) {
    u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

// Read as one vector: of a uint4 read word by word, joined again for a matrix instruction and carried around a loop, hipcc (ROCm 7.2)
// has given words to another value while they were needed (few-row experts' weights: its IR was right, its registers not)
__device__ __forceinline__ uint4 ldg16(const void* p) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}

// 16-B load whose lane may be out of range: the load is ALWAYS issued (from `safe` when !ok) and
// the value zeroed afterwards -- a conditional load (ok ? load : 0) makes hipcc branch around the
// load and wait vmcnt(0) for it, one dependent round trip per element.  Its words are read and chosen one by one, unlike ldg16's (as
// one vector residual + router spills 18 registers); in the disassembly of its users no matrix instruction's words are overwritten
__device__ __forceinline__ uint4 ldg16_sel(const void* p, bool ok, const void* safe) {
    const uint4 v = *reinterpret_cast<const uint4*>(ok ? p : safe);
    return ok ? v : make_uint4(0, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma16(const short8 a, const short8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

}  // namespace pgmi
