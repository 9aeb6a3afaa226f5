// Wave-wide sums of eight values per lane, shared by the symmetric pair kernels.
#pragma once
#include "halma_common.h"

namespace halma {

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    // lanes whose source lies outside their row of 16 read 0 (never used below)
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf,
                                                      true));
}

// a double from another lane of the row, half by half
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// v[0..7] per lane -> the sum over all 64 lanes of v[k], for k = source index of the lane:
// k = 4*bit5 + 2*bit4 + bit3 of the lane id, valid in the lanes with lane % 8 == 0.
// A fixed binary tree of depth 6 per total: recursive halving over lane bits 5 and 4 with
// the CDNA4 half-wave and row swaps (v_permlane32_swap / v_permlane16_swap: each lane
// ends with its half's pair sum of v[k] or v[k + 4], then of w[k] or w[k + 2]), over
// bit 3 with a row rotation by 8, then lane + (lane + 4), + (lane + 2), + (lane + 1)
// within the row (DPP row shifts).  The first kF32 levels are FP32, the others FP64, so a
// caller adds its own terms times 2^kF32 in FP32.  The last three levels in FP64, whose
// roundings no other sum averages out, take 8 issue slots per eight sources more than in FP32
// and halve the symmetric kernel's error (kF32 = 3: 26 slots); the first three take 12 more.
__device__ __forceinline__ double swap_add32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    return static_cast<double>(__uint_as_float(r[0])) +
           static_cast<double>(__uint_as_float(r[1]));
}

__device__ __forceinline__ double swap_add16(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap(
        static_cast<unsigned>(__double2loint(a)), static_cast<unsigned>(__double2loint(b)), false,
        false);
    const auto h = __builtin_amdgcn_permlane16_swap(
        static_cast<unsigned>(__double2hiint(a)), static_cast<unsigned>(__double2hiint(b)), false,
        false);
    return __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0])) +
           __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
}

template <int kF32>
__device__ __forceinline__ double reduce8(const float v[8], int lane) {
    const bool h3 = (lane & 8) != 0;
    double t;
    if constexpr (kF32 == 0) {
        double w[4], u[2];
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = swap_add32(v[k], v[k + 4]);
#pragma unroll
        for (int k = 0; k < 2; ++k) u[k] = swap_add16(w[k], w[k + 2]);
        t = (h3 ? u[1] : u[0]) + dpp_move<0x128>(h3 ? u[0] : u[1]);  // row_ror:8
    } else {
        static_assert(kF32 == 2 || kF32 == 3, "FP32 levels");
        float w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const auto r = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(v[k]), __float_as_uint(v[k + 4]), false, false);
            w[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
        float u[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const auto r = __builtin_amdgcn_permlane16_swap(
                __float_as_uint(w[k]), __float_as_uint(w[k + 2]), false, false);
            u[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
        const float keep = h3 ? u[1] : u[0], other = dpp_move<0x128>(h3 ? u[0] : u[1]);
        t = kF32 == 2 ? static_cast<double>(keep) + static_cast<double>(other)
                      : static_cast<double>(keep + other);
    }
    t += dpp_move<0x104>(t);  // row_shl:4
    t += dpp_move<0x102>(t);  // row_shl:2
    t += dpp_move<0x101>(t);  // row_shl:1
    return t;
}

}  // namespace halma
