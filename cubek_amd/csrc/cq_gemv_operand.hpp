// What the kernels of the products with quantized weights on the matrix cores share (cq_kernels_gemv_quads.hip,
// cq_kernels_gemv_batch.hip): codes to operands of the matrix instructions, and the store of y.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/cubek_quant_device.hpp"
#include "cq_internal.hpp"

namespace cq {
namespace {

namespace dev = cubek_quant::device;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kCodeE4M3 = 100, kCodeE5M2 = 101, kCodeE2M1x2 = 102;  // the native encodings; else bits per field

constexpr uint32_t values_per_unit(int code) { return code <= 8 ? 128u / static_cast<uint32_t>(code) : (code == kCodeE2M1x2 ? 32u : 16u); }

// The 4-bit fields of f16 tensors pair up as (0, 4), (1, 5), (2, 6), (3, 7): one mask plants two digits in two
// halves, without shifting them together; x is brought into the same order.
template <dev::Float kF, int kCode>
constexpr bool kCrossPairs = kF == dev::Float::F16 && kCode == 4;

// Eight consecutive values (kVals of a unit / 8 such groups) of a lane's unit as the matrix instruction takes them.
template <dev::Float kF, int kCode, bool kShort>
__device__ __forceinline__ u32x4 operand(const u32x4& unit, uint32_t m, float scale) {
    uint32_t p[8];
    if constexpr (kCrossPairs<kF, kCode> && kShort) {
        const uint32_t w = unit[m];
        const _Float16 sh = static_cast<_Float16>(scale);
        const f16x2 s2 = {sh, sh};
        const f16x2 off0 = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-1032.0f)};
        const f16x2 off1 = {static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)};
        const f16x2 sixteenth = {static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t v = h ? w >> 8 : w;
            const uint32_t a = (v & 0x000f000fu) ^ 0x64086408u;  // 1024 + digit
            const uint32_t b = (v & 0x00f000f0u) ^ 0x64806480u;  // 1024 + 16 * digit
            const f16x2 qa = __builtin_bit_cast(f16x2, a) + off0;                                            // exact
            const f16x2 qb = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, b), sixteenth, off1);      // exact
            p[2 * h] = __builtin_bit_cast(uint32_t, s2 * qa);
            p[2 * h + 1] = __builtin_bit_cast(uint32_t, s2 * qb);
        }
        return u32x4{p[0], p[1], p[2], p[3]};
    } else if constexpr (kCode == 4) {
        if constexpr (kShort)
            dev::dequantize_symmetric_packed_value_pairs_tame<kF, 4>(unit[m], scale, p);
        else
            dev::dequantize_symmetric_packed_value_pairs<kF, 4>(unit[m], scale, p);
        if constexpr (kCrossPairs<kF, kCode>)
            return u32x4{__builtin_amdgcn_perm(p[2], p[0], 0x05040100u), __builtin_amdgcn_perm(p[2], p[0], 0x07060302u),
                         __builtin_amdgcn_perm(p[3], p[1], 0x05040100u), __builtin_amdgcn_perm(p[3], p[1], 0x07060302u)};
        else
            return u32x4{p[0], p[1], p[2], p[3]};
    } else if constexpr (kCode == 8) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (kShort)
                dev::dequantize_symmetric_packed_value_pairs_tame<kF, 8>(unit[2 * m + j], scale, p + 2 * j);
            else
                dev::dequantize_symmetric_packed_value_pairs<kF, 8>(unit[2 * m + j], scale, p + 2 * j);
        }
        return u32x4{p[0], p[1], p[2], p[3]};
    } else if constexpr (kCode == kCodeE2M1x2) {
        dev::dequantize_symmetric_native_value_pairs<kF, dev::Native::E2M1x2>(unit[m], scale, p);
        return u32x4{p[0], p[1], p[2], p[3]};
    } else {
        constexpr dev::Native kNative = kCode == kCodeE4M3 ? dev::Native::E4M3 : dev::Native::E5M2;
        dev::dequantize_symmetric_native_value_pairs<kF, kNative>(unit[2 * m], scale, p);
        dev::dequantize_symmetric_native_value_pairs<kF, kNative>(unit[2 * m + 1], scale, p + 2);
        return u32x4{p[0], p[1], p[2], p[3]};
    }
}

__device__ __forceinline__ void store_y(int dtype, void* y, uint64_t i, float v) {
    if (dtype == CQ_F32)
        static_cast<float*>(y)[i] = v;
    else if (dtype == CQ_F16)
        static_cast<_Float16*>(y)[i] = static_cast<_Float16>(v);
    else
        static_cast<__bf16*>(y)[i] = static_cast<__bf16>(v);
}

}  // namespace
}  // namespace cq
