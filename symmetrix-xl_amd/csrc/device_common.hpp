// Shared helpers of the HIP kernels (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <string>

namespace smx {

constexpr int kWave = 64;
// Edge ids are int32 (the reference's cardinality guard,
// mace_kokkos_runtime.cpp:199); the margin keeps strided int loops over edge
// ranges (stride <= 4096) from overflowing.
constexpr long long kMaxEdges = 2147483647LL - 4096;
// The tiled plan indexes the graph's edges with 64 bits (each tile's kernels
// see 32-bit offsets relative to the tile's first edge); its bound keeps a
// one-thread-per-edge launch under the 2^32 work-items of a dispatch.
constexpr long long kMaxWideEdges = (1LL << 32) - (1LL << 20);
constexpr int kXcds = 8;

inline void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}
#define SMX_HIP(call) ::smx::hip_check((call), #call)
#define SMX_LAUNCH_CHECK(name) ::smx::hip_check(hipGetLastError(), name)

// MI355X dispatches workgroups round-robin over its 8 XCDs, each with its own
// L2.  Remap so that XCD x processes one contiguous range of the logical
// index space: neighbouring receivers share neighbours, so their features stay
// in that XCD's L2.  The map is a bijection on [0, n).
__device__ __forceinline__ int xcd_remap(int b, int n) {
    const int q = n / kXcds, r = n % kXcds;
    const int x = b % kXcds, j = b / kXcds;
    return x * q + (x < r ? x : r) + j;
}

// Butterfly sum over the first `width` lanes of a wave (width a power of two
// <= 64); every participating lane ends with the total.
template <int WIDTH>
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = WIDTH / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, WIDTH);
    return v;
}

// v + v[lane permuted by the DPP control CTRL] on the rows in ROW_MASK
// (other rows add 0)
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v) {
    const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false);
    return v + __int_as_float(moved);
}

// Sum over each row of 16 lanes with DPP (quad permutes, half-row and row
// mirrors); every lane of a row holds its row's sum.
__device__ __forceinline__ float row_total(float v) {
    v = dpp_add<0xb1, 0xf>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4e, 0xf>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x141, 0xf>(v);  // row_half_mirror
    return dpp_add<0x140, 0xf>(v);  // row_mirror
}

// Sum over the first WIDTH (32 or 64) lanes of a wave with DPP row
// operations (quad permutes, half-row and row mirrors, then the row
// broadcasts 15 and 31), returned wave-uniform from the last lane.
template <int WIDTH>
__device__ __forceinline__ float wave_total(float v) {
    static_assert(WIDTH == 32 || WIDTH == 64, "DPP reduction over 32 or 64 lanes");
    v = dpp_add<0xb1, 0xf>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4e, 0xf>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x141, 0xf>(v);  // row_half_mirror: sums of 8
    v = dpp_add<0x140, 0xf>(v);  // row_mirror: every lane of a row holds the row sum
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    if constexpr (WIDTH == 64) {
        v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
    } else {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 31));
    }
}

template <int WIDTH>
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = WIDTH / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, WIDTH);
    return v;
}

// FP32 matrix products on bf16 MFMAs: an FP32 value as three bf16 parts, each
// the rounding of what the ones before it left.  Three parts hold a normal
// value exactly; the MFMA takes parts below 2^-126 as zero, so values below
// about 2^-102 lose their last bits (2^-16 of a sum at inputs of 2^-112).  The first two are
// kept finite, so that values up to FLT_MAX, which round to infinity in bf16,
// stay finite too, and an infinity or NaN is the third part alone: it meets
// only the other operand's first part and gives what an FP32 product gives.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

// largest bf16, and the largest that a second part can be
constexpr float kSplitMax = 0x1.fep127f, kSplitMax2 = 0x1p120f;

struct SplitOperand {
    bf16x8 part[3];
};

// (pairs by hand: one v_cvt_pk_bf16_f32 rounds two values, and a part's value
// is its bits in the upper half)
__device__ __forceinline__ SplitOperand split_operand(f32x8 x) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    SplitOperand o;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        u32x4 bits;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const float big = p == 0 ? kSplitMax : kSplitMax2;
            const f32x2 v = p == 2 ? f32x2{x[2 * h], x[2 * h + 1]}
                                   : f32x2{__builtin_amdgcn_fmed3f(x[2 * h], -big, big),
                                           __builtin_amdgcn_fmed3f(x[2 * h + 1], -big, big)};
            bits[h] = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
            if (p < 2) {
                x[2 * h] -= __uint_as_float(bits[h] << 16);
                x[2 * h + 1] -= __uint_as_float(bits[h] & 0xffff0000u);
            }
        }
        o.part[p] = __builtin_bit_cast(bf16x8, bits);
    }
    return o;
}

// acc + a b over 32 channels (v_mfma_f32_16x16x32_bf16) from the parts, the
// smallest products first.  A second part is at most 2^-8 and a third 2^-17 of
// its value: the products left out (2 with 3, 3 with 2, 3 with 3) are at most
// about 2^-24 |a b|, the size of an FP32 product's own rounding.
typedef float acc4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ acc4 split_product(const SplitOperand& a, const SplitOperand& b, acc4 acc) {
    constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.part[pa[q]], b.part[pb[q]], acc, 0, 0, 0);
    return acc;
}

inline unsigned blocks_for(std::int64_t n, int per_block) {
    return static_cast<unsigned>((n + per_block - 1) / per_block);
}

}  // namespace smx
