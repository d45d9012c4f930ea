// What the kernels of the products with quantized weights share (cq_kernels_gemv.hip, cq_kernels_gemv_quads.hip,
// cq_kernels_gemv_batch.hip): codes to operands of the matrix instructions, and the store of y.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

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

// The 4-bit fields of f16 tensors come out of a word's bytes as (0, 2), (4, 6), (1, 3), (5, 7).  Where x is laid out by the kernel it is brought
// into the same order (`crossed`), else the bytes are put in order first, half the work of reordering x in every step.
template <dev::Float kF, int kCode>
constexpr bool kPairsCross = kF == dev::Float::F16 && kCode == 4;
__device__ __forceinline__ u32x4 crossed(u32x4 p) {
    return u32x4{__builtin_amdgcn_perm(p[1], p[0], 0x05040100u), __builtin_amdgcn_perm(p[3], p[2], 0x05040100u),
                 __builtin_amdgcn_perm(p[1], p[0], 0x07060302u), __builtin_amdgcn_perm(p[3], p[2], 0x07060302u)};
}

// Scales of less than this size take the short dequantization (their bits as a number, sign apart): where digit * s - bias * s
// is exact.  A sum does not see the sign of a zero product, so unlike a stored value zero and negative scales may go that way.
template <dev::Float kF, int kCode>
constexpr uint32_t kShortBelow = kPairsCross<kF, kCode> ? 0x45800000u : 0x71800000u;  // 4096, so that 8 * s is a number of f16; 2^100

// Eight consecutive values (kVals of a unit / 8 such groups) of a lane's unit as the matrix instruction takes them; kCrossed: in the
// order of crossed().
//
// 4 bits of f16: a byte 0x0d read as an e4m3 number is d * 2^-9 for every d in 0..15, so one conversion gives two digits and one packed FMA
// their values, rounded once: 44 cycles of VALU for eight, 50 by digits planted under the exponent of 1024, which take a
// subtraction and a product.
template <dev::Float kF, int kCode, bool kShort, bool kCrossed = false>
__device__ __forceinline__ u32x4 operand(const u32x4& unit, uint32_t m, float scale) {
    static_assert(!kCrossed || kPairsCross<kF, kCode>, "other pairs come in order");
    uint32_t p[8];
    if constexpr (kPairsCross<kF, kCode> && kShort) {
        const uint32_t w = unit[m];
        const _Float16 sh = static_cast<_Float16>(scale);
        const f16x2 s2 = {sh, sh}, bias = s2 * f16x2{static_cast<_Float16>(-8.0f), static_cast<_Float16>(-8.0f)};  // exact
        uint32_t first = (w & 0x0f0f0f0fu) ^ 0x08080808u, second = ((w >> 4) & 0x0f0f0f0fu) ^ 0x08080808u;  // digits 0, 2, 4, 6; 1, 3, 5, 7
        if constexpr (!kCrossed) {
            const uint32_t even = first, odd = second;
            first = __builtin_amdgcn_perm(odd, even, 0x05010400u), second = __builtin_amdgcn_perm(odd, even, 0x07030602u);
        }
        const auto values = [&](uint32_t digits, auto high) {
            return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(digits, 512.0f, high.value)), s2, bias));
        };
        return u32x4{values(first, std::false_type{}), values(first, std::true_type{}), values(second, std::false_type{}), values(second, std::true_type{})};
    } else if constexpr (kCode == 4) {
        if constexpr (kShort)
            dev::dequantize_symmetric_packed_value_pairs_tame<kF, 4>(unit[m], scale, p);
        else
            dev::dequantize_symmetric_packed_value_pairs<kF, 4>(unit[m], scale, p);
        const u32x4 in_order = {p[0], p[1], p[2], p[3]};
        return kCrossed ? crossed(in_order) : in_order;
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

inline uint32_t log2_of(uint32_t v) {
    uint32_t l = 0;
    while ((1u << l) < v) l++;
    return l;
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
