// y = dequantize(W) * x for one to four vectors, W read once in its packed form, where cq_kernels_gemv.hip's and
// cq_kernels_gemv_batch.hip's kernels leave compute units idle or lanes empty (quads_split() says where): the quantized-input arm of the
// reference's matmul (crates/cubek-matmul/src/base.rs:309-317; scale lookup components/global/memory/layout.rs:371-455).
// Every weight enters the product as cq_dequantize would store it (crates/cubek-quant/src/dequantize.rs:20-79); products
// accumulate in f32.
//
// One workgroup per compute unit takes an equal share of the rows, and its waves four rows at a time, or shares of the columns of
// four rows where rows are few.  All of x is staged in LDS once per workgroup, behind the first loads of codes, and the codes of a
// wave's next steps are always on their way, across the ends of rows, so that there is one start-up per launch and no barrier between
// it and the end.  A step is sixteen 16-byte units of each of four rows: 256 bytes of a row side by side, which memory serves as well as whole
// KiB (the loads alone, [28672, 8192] 4 bits: 24.2 us, as gemv_stream_kernel's), where the 64 bytes of 16 x 16 x 32 instructions are not.
//
// Bound by the issue of the dequantization's instructions where weights of 4 bits fill the chip ([28672, 8192] bf16 29.9 us, without its loads 27.1, with x in
// registers instead of LDS as long, the loads alone 24.1; 12.3 M instructions of four cycles are 83 % of the cycles of the launch without loads; a 4 x 4 x 4
// matrix instruction takes nine cycles of the same unit, so one vector costs what v_dot2 does and four cost no more), by memory and the
// one start-up elsewhere.  Two steps ahead: three and four hold more registers than they hide (31.1, 31.9 against 30.2 us).
#include <hip/hip_runtime.h>

#include "cq_gemv_operand.hpp"
#include "cq_launch_rules.hpp"

namespace cq {
namespace {

// D (4 x 4 per block) += A (4 x 4) * B (4 x 4), sixteen blocks side by side: lane (i, b) = (lane % 4, lane / 4) holds row i of
// A and column i of B of block b, four values each, and column i of D in four registers.
template <dev::Float kF>
__device__ __forceinline__ f32x4 mfma4(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, f32x4 c) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 a = {a0, a1}, b = {b0, b1};
    if constexpr (kF == dev::Float::BF16) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
    } else {
        typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
        return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
    }
}

constexpr int kDepth = 2;

__device__ __forceinline__ uint32_t bits_of(float v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ float float_of(uint32_t v) { return __builtin_bit_cast(float, v); }

template <int kCtrl>
__device__ __forceinline__ float ror_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kCtrl, 0xf, 0xf, true));
}

template <dev::Float kF, class FS, int kCode, uint32_t kWaves>
__global__ __launch_bounds__(64 * kWaves) void gemv_quads_kernel(
    const char* __restrict__ words, const char* __restrict__ scales, const char* __restrict__ x, uint32_t rows, uint32_t units_per_row,
    uint32_t row_bytes, uint32_t scale_row_bytes, uint32_t scale_step, uint32_t packed, uint32_t quads_per, uint32_t pieces_inverse,
    uint32_t x_stride_bytes, uint32_t block_rows, void* __restrict__ y, uint64_t y_stride) {
    const uint32_t vectors = packed & 31u, units_per_block_log2 = (packed >> 5) & 31u, slots_log2 = (packed >> 10) & 7u,
                   shares_log2 = (packed >> 13) & 7u;
    const int y_dtype = static_cast<int>(packed >> 16);
    const uint32_t base = quads_per & 255u, extra = quads_per >> 8;
    constexpr bool kPacked = kCode <= 8;
    constexpr uint32_t kM = values_per_unit(kCode) / 8;
    extern __shared__ char lds[];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t i = lane & 3u, b = lane >> 2;
    const uint32_t steps = (units_per_row + 15u) / 16u;
    const uint32_t rot = slots_log2 == 2 ? 1u : 4u;
    const uint32_t ring = (16u << slots_log2) - 1u;
    const uint32_t quad0 = blockIdx.x * base + min(blockIdx.x, extra), nq = base + (blockIdx.x < extra ? 1u : 0u);
    const uint32_t shares = 1u << shares_log2, share = wave & (shares - 1u), slot = wave >> shares_log2;
    const uint32_t per = (steps + shares - 1u) >> shares_log2;
    const uint32_t first = min(share * per, steps), len = min(per, steps - first);
    const uint32_t wave_slots = kWaves >> shares_log2;
    const uint32_t mine = slot < nq ? (nq - slot + wave_slots - 1u) / wave_slots : 0u;
    const uint32_t total = mine * len;

    // x: piece m of unit (step, column b) of vector v at ((step * kM + m) * kN + v / 4) * (16 << slots_log2) + (column * kV + v % 4, rotated by m)
    const uint32_t pieces = steps * 16u * kM, staged = pieces << slots_log2;
    const auto x_from = [&](uint32_t at) {
        const uint32_t v = __umulhi(at, pieces_inverse), p = at - v * pieces;
        return *reinterpret_cast<const u32x4*>(x + static_cast<uint64_t>(min(v, vectors - 1u)) * x_stride_bytes + min(p, units_per_row * kM - 1u) * 16u);
    };
    const auto x_to = [&](uint32_t at, u32x4 val) {
        const uint32_t v = __umulhi(at, pieces_inverse), p = at - v * pieces, u = p / kM, m = p % kM;
        if (u >= units_per_row) val = u32x4{0, 0, 0, 0};
        if constexpr (kPairsCross<kF, kCode>) val = crossed(val);
        const uint32_t at_lds = (((u >> 4) * kM + m) << (4u + slots_log2)) + ((((u & 15u) << slots_log2) + v + m * rot) & ring);
        *reinterpret_cast<u32x4*>(lds + at_lds * 16u) = val;
    };
    constexpr uint32_t kThreads = 64 * kWaves;
    u32x4 x_first[2];
#pragma unroll
    for (uint32_t k = 0; k < 2; k++) x_first[k] = x_from(min(threadIdx.x + k * kThreads, staged - 1u));
    __builtin_amdgcn_sched_barrier(0);
    float* const part = reinterpret_cast<float*>(lds + staged * 16u);  // [quad][share][four vectors][row][vector]
    uint32_t x_lane[kM];
#pragma unroll
    for (uint32_t m = 0; m < kM; m++)
        x_lane[m] = (m << (8u + slots_log2)) + ((((b << slots_log2) + (i & ((1u << slots_log2) - 1u))) + m * rot) & ring) * 16u;
    const uint32_t step_bytes = kM << (8u + slots_log2);

    struct Chunk {
        u32x4 w;
        FS s;
    };
    Chunk c[kDepth];
    uint32_t left = total, load_step = first, load_quad = slot;
    const char *wq = words, *sq = scales;
    // a lane's distances from the quad's first row: in whole steps, and in the row's last step, where lanes past the row's end
    // read its last unit again
    const uint32_t b_last = min(b, (units_per_row - 1u) & 15u);
    const uint32_t w_b = b * 16u, w_b_last = b_last * 16u;
    const uint32_t s_b = (b >> units_per_block_log2) * scale_step, s_b_last = (b_last >> units_per_block_log2) * scale_step;
    uint32_t w_lane = 0, s_lane = 0, w_last = 0, s_last = 0;
    const auto go_to = [&](uint32_t q) {
        const uint32_t row0 = (quad0 + q) * 4u, r = min(row0 + i, rows - 1u);
        wq = words + static_cast<uint64_t>(row0) * row_bytes;
        const uint32_t w_row = (r - row0) * row_bytes;
        uint32_t sr0 = row0, sr = r;
        if (block_rows != 1) sr0 = row0 / block_rows, sr = r / block_rows;
        sq = scales + static_cast<uint64_t>(sr0) * scale_row_bytes;
        const uint32_t s_row = (sr - sr0) * scale_row_bytes;
        w_lane = w_row + w_b, w_last = w_row + w_b_last;
        s_lane = s_row + s_b, s_last = s_row + s_b_last;
    };
    if (total != 0) go_to(slot);
    const auto load = [&](Chunk& k) {
        const bool last = load_step == steps - 1u;
        const char* const wf = wq + load_step * 256u;
        const char* const sf = sq + static_cast<uint64_t>((load_step * 16u) >> units_per_block_log2) * scale_step;
        k.w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wf + (last ? w_last : w_lane)));
        k.s = *reinterpret_cast<const FS*>(sf + (last ? s_last : s_lane));
        __builtin_amdgcn_sched_barrier(0);
        if (left > 1) {
            load_step++;
            if (load_step == first + len) {
                load_step = first, load_quad += wave_slots;
                go_to(load_quad);
            }
            left--;
        } else {  // past the wave's last step: one address instead of nothing
            w_lane = w_last = s_lane = s_last = 0;
        }
    };
    f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    uint32_t work_step = first, work_quad = slot;
    const auto work = [&](const Chunk& k) {
        u32x4 w = k.w;
        FS stored = k.s;
        if (work_step * 16u + 16u > units_per_row) {  // wave-uniform: units past the row's end count nothing
            const bool past = work_step * 16u + b >= units_per_row;
            asm volatile("");  // (a branch, not a selection in every step)
            w = past ? u32x4{0, 0, 0, 0} : w;
            stored = past ? static_cast<FS>(1.0f) : stored;
        }
        const char* const x_step = lds + work_step * step_bytes;
        const float s = dev::round_to<kF>(dev::widen(stored));
        // ordinary scales all take the short dequantization
        if (!kPacked || __builtin_amdgcn_ballot_w64((bits_of(s) & 0x7fffffffu) >= kShortBelow<kF, kCode>) == 0) {
#pragma unroll
            for (uint32_t m = 0; m < kM; m++) {
                const u32x4 xb = *reinterpret_cast<const u32x4*>(x_step + x_lane[m]);
                const u32x4 p = operand<kF, kCode, true, kPairsCross<kF, kCode>>(w, m, s);
                acc[0] = mfma4<kF>(p[0], p[1], xb[0], xb[1], acc[0]);
                acc[1] = mfma4<kF>(p[2], p[3], xb[2], xb[3], acc[1]);
            }
        } else {
#pragma unroll 1
            for (uint32_t m = 0; m < kM; m++) {  // one copy of the general code: its operands are picked out
                u32x4 word = {0, 0, 0, 0};
                uint32_t x_at = 0;
#pragma unroll
                for (uint32_t t = 0; t < kM; t++)
                    if (m == t) {
                        word = kM == 4 ? u32x4{w[t], 0, 0, 0} : u32x4{w[2 * t & 3], w[(2 * t + 1) & 3], 0, 0};
                        x_at = x_lane[t];
                    }
                const u32x4 xb = *reinterpret_cast<const u32x4*>(x_step + x_at);
                const u32x4 p = operand<kF, kCode, false, kPairsCross<kF, kCode>>(word, 0, s);
                acc[0] = mfma4<kF>(p[0], p[1], xb[0], xb[1], acc[0]);
                acc[0] = mfma4<kF>(p[2], p[3], xb[2], xb[3], acc[0]);
            }
        }
        work_step++;
        if (work_step == first + len) {  // wave-uniform: the share of these rows is done, and the sixteen blocks' sums meet
            const f32x4 d = acc[0] + acc[1];
            const float d0 = d[0], d1 = d[1], d2 = d[2], d3 = d[3];  // (a bit cast of the element expression itself reads element 0)
            // two rows' sums fold into the halves of one register, then all four into its rows of 16 lanes, in the order 0, 2, 1, 3
            const auto s01 = __builtin_amdgcn_permlane32_swap(bits_of(d0), bits_of(d1), false, false);
            const auto s23 = __builtin_amdgcn_permlane32_swap(bits_of(d2), bits_of(d3), false, false);
            const float h01 = float_of(s01[0]) + float_of(s01[1]), h23 = float_of(s23[0]) + float_of(s23[1]);
            const auto q = __builtin_amdgcn_permlane16_swap(bits_of(h01), bits_of(h23), false, false);
            float v = float_of(q[0]) + float_of(q[1]);
            v = ror_add<0x124>(v);
            v = ror_add<0x128>(v);
            const uint32_t r16 = lane >> 4, r = (r16 >> 1) | ((r16 & 1u) << 1);
            if ((lane & 12u) == 0) part[((work_quad << shares_log2) + share) * 16u + r * 4u + i] = v;
            acc[0] = acc[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            work_step = first, work_quad += wave_slots;
        }
    };
    if (total != 0) {
#pragma unroll
        for (int d = 0; d < kDepth; d++) load(c[d]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t k = 0; k < 2; k++)
        if (threadIdx.x + k * kThreads < staged) x_to(threadIdx.x + k * kThreads, x_first[k]);
    if (staged > 2 * kThreads) {
        for (uint32_t at = threadIdx.x + 2 * kThreads; at < staged; at += 4 * kThreads) {
            u32x4 val[4];
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) val[k] = x_from(min(at + k * kThreads, staged - 1u));
#pragma unroll
            for (uint32_t k = 0; k < 4; k++)
                if (at + k * kThreads < staged) x_to(at + k * kThreads, val[k]);
        }
    }
    __syncthreads();
    if (total != 0) {
        for (uint32_t t = 0; t < total; t += kDepth) {
#pragma unroll
            for (int d = 0; d < kDepth; d++) {
                if (d == 0 || t + d < total) work(c[d]);
                load(c[d]);
            }
        }
    }
    __syncthreads();
    const uint32_t my_rows = min(nq * 4u, rows - quad0 * 4u);
    const uint32_t full = (steps + per - 1u) / per;  // shares that have steps
    for (uint32_t at = threadIdx.x; at < my_rows << slots_log2; at += kThreads) {
        const uint32_t v = at & ((1u << slots_log2) - 1u), r = at >> slots_log2;
        const float* const from = part + ((r >> 2) << shares_log2) * 16u + (r & 3u) * 4u + v;
        float sum = 0.0f;
        for (uint32_t s = 0; s < full; s += 4) {
            float t[4];
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) t[k] = from[min(s + k, full - 1u) * 16u];
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) sum += s + k < full ? t[k] : 0.0f;
        }
        if (v < vectors) store_y(y_dtype, y, v * y_stride + quad0 * 4u + r, sum);
    }
}

template <dev::Float kF, class FS, int kCode, uint32_t kWaves>
void launch_waves(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) {
    constexpr uint32_t kVals = values_per_unit(kCode), kM = kVals / 8;
    const uint32_t units = a.cols / kVals, steps = (units + 15) / 16, quads = (a.rows + 3) / 4;
    const uint32_t block_log2 = a.block_rows == 0 ? 31u : log2_of(a.block_cols / kVals);
    const uint32_t packed = a.vectors | block_log2 << 5 | log2_of(a.vectors) << 10 | q.shares_log2 << 13 | static_cast<uint32_t>(a.y_dtype) << 16;
    hipLaunchKernelGGL((gemv_quads_kernel<kF, FS, kCode, kWaves>), dim3(q.grid), dim3(64 * kWaves), q.lds, s, static_cast<const char*>(a.words),
                       static_cast<const char*>(a.scales), static_cast<const char*>(a.x), a.rows, units, static_cast<uint32_t>(a.word_pitch * 4),
                       static_cast<uint32_t>(a.scale_stride_row * sizeof(FS)), static_cast<uint32_t>(a.scale_stride_col * sizeof(FS)), packed,
                       quads / q.grid | (quads % q.grid) << 8, static_cast<uint32_t>((1ull << 32) / (steps * 16 * kM)) + 1,
                       static_cast<uint32_t>(a.x_stride * 2), a.block_rows == 0 ? 1u : a.block_rows, a.y, a.y_stride);
}

template <dev::Float kF, class FS, int kCode>
void launch_code(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) {
    if (q.waves == 16)
        launch_waves<kF, FS, kCode, 16>(s, a, q);
    else
        launch_waves<kF, FS, kCode, 8>(s, a, q);
}

template <dev::Float kF, class FS>
hipError_t launch_codes(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) {
    if (a.native == 1)
        launch_code<kF, FS, kCodeE4M3>(s, a, q);
    else if (a.native == 2)
        launch_code<kF, FS, kCodeE5M2>(s, a, q);
    else if (a.native == 3)
        launch_code<kF, FS, kCodeE2M1x2>(s, a, q);
    else if (a.bits == 4)
        launch_code<kF, FS, 4>(s, a, q);
    else
        launch_code<kF, FS, 8>(s, a, q);
    return hipGetLastError();
}

}  // namespace

// One object per type of x and of the scales (CQ_GEMV_PART names the one being compiled), so that a process loads the
// code of the kind it uses.
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 0
hipError_t gemv_quads_bf16_f32(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) { return launch_codes<dev::Float::BF16, float>(s, a, q); }
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 1
hipError_t gemv_quads_bf16_bf16(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) { return launch_codes<dev::Float::BF16, __bf16>(s, a, q); }
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 2
hipError_t gemv_quads_bf16_f16(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) { return launch_codes<dev::Float::BF16, _Float16>(s, a, q); }
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 3
hipError_t gemv_quads_f16_f32(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) { return launch_codes<dev::Float::F16, float>(s, a, q); }
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 4
hipError_t gemv_quads_f16_bf16(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) { return launch_codes<dev::Float::F16, __bf16>(s, a, q); }
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 5
hipError_t gemv_quads_f16_f16(hipStream_t s, const GemvArgs& a, const QuadsSplit& q) { return launch_codes<dev::Float::F16, _Float16>(s, a, q); }
#endif

}  // namespace cq
