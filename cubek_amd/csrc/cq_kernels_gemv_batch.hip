// Y = X * dequantize(W)^T for up to sixteen right-hand vectors at once, on the matrix cores: the quantized-input arm of
// the reference's matmul (crates/cubek-matmul/src/base.rs:309-317; scale lookup
// components/global/memory/layout.rs:371-455) for a decode step of a batch.  Every weight enters the product as
// cq_dequantize would store it, F(F(scale) * F(code)) (crates/cubek-quant/src/dequantize.rs:20-79, through
// include/cubek_quant_device.hpp); products accumulate in f32.
//
// A 16 x 16 x 32 matrix instruction wants, in lane (i, g) = (lane % 16, lane / 16), eight values of row i of W and
// the same eight columns of vector i of x, and the columns of the four g may be any 32 that both operands agree on.
// Read straight into registers in that order, an instruction touches 64 bytes of each of 16 rows, and such loads cost
// about 75 cycles of a compute unit each, codes, scales and x alike (28672 x 8192, 4 bits: 47 - 60 us however deep
// they were issued ahead).  So everything goes through LDS with direct loads of whole lines, a stage of eight 16-byte
// units per row (128 bytes) at a time, and the next stage is on its way while one is worked on.  The places of a
// stage are rotated from row to row on their way in, so that the 16 lanes of a read fall on 16 different groups of banks.
//
// Bound by instructions beside the loads where a weight of 4 bits fills the chip: 2.4 per bf16 weight for the
// dequantization, 0.5 for the rest; at 4 cycles each they issue for more than half of the time ([28672, 8192], blocks of 32:
// 34 us for 4 vectors, 38 us for 16; a read of the bytes 21 us), the matrix instructions for a tenth beside them.  With 8
// bits and e4m3 bytes ([28672, 8192] 8 bits, 16 vectors 57 us), and in launches of a few rounds ([14336, 4096] f16, 8 vectors
// 10 us), they issue for 35 - 43 %, and the waves spend about half of theirs waiting for a stage; few rows ([1024, 28672],
// 64 workgroups, 28 us) are a chain of stages on a quarter of the chip.
//
// Products of up to four vectors go through it only where its groups of 16 rows fill the chip (quads_split()).  Against the kernels of
// two to four vectors a launch before it, us: [28672, 8192] 4 bits bf16 2 vectors 35.0 -> 34.1, 16
// vectors 140 -> 39, f16 2 vectors 54 -> 31, 8 bits 57 -> 51, e4m3 56 -> 50; [14336, 4096] bf16 2 vectors 12.5 -> 11.7, f16
// blocks of 128 20.0 -> 10.5 (9.95 since its codes are put in order instead of x); [1024, 28672] 2 vectors 30 -> 17.8, 16 vectors 141 -> 28.6.  The one size that lost is
// [8192, 28672] in e4m3 bytes with 3 vectors, 54.2 -> 56.5.
#include <hip/hip_runtime.h>

#include "cq_gemv_operand.hpp"
#include "cq_launch_rules.hpp"

namespace cq {
namespace {

template <dev::Float kF>
__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (kF == dev::Float::BF16) {
        typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    } else {
        typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
}

#define CQ_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))


constexpr uint32_t kU = 8;  // units of a row per stage
// LDS of a stage: the codes and scales of a wave's 16 rows; the vectors' values (whole loads of 1 KiB)
constexpr uint32_t kCodeBytes = 16 * kU * 16, kWaveBytes = kCodeBytes + 16 * kU * 4;
template <int kCode>
__host__ __device__ constexpr uint32_t x_bytes(uint32_t vectors) {
    return (vectors * 2u * kU * values_per_unit(kCode) + 1023u) & ~1023u;
}

// kG groups of 16 rows per workgroup times kS shares of the row's stages (every kS-th one): kG * kS waves.  The waves
// of a share use its x together; the shares' sums meet in LDS at the end.
//
// kWholeLines: the rows start on lines of 128 bytes, and the codes, of which a stage takes whole lines, are streamed past the caches.  Rows that do
// not: a stage reads parts of lines, whose rest the next one wants from the caches (streaming -> plain loads, us: f16 4 bits [2788, 4256] 5 vectors
// 6.4 -> 5.6, [3590, 14752] 16 19.4 -> 17.6, 8 bits [20000, 6752] 8 44.0 -> 40.8; whole lines [28672, 8192] 8 bits 16 54.7 -> 59.2, 4 bits 36.9 -> 38.9,
// [14336, 4096] f16 8 10.1 -> 9.7).  gemv_batch_streams() names the rows of parts that stream all the same.  A kernel of its own for each: with both
// behind a branch in every stage whole lines lost 1 - 5 % (4 bits [8192, 28672] 2 vectors 30.8 -> 32.0, e4m3 [12288, 11904] 4 26.7 -> 28.0, 4 bits
// [14439, 4352] 16 13.2 -> 13.6) and parts of lines 2 %; but in 4 x 2 parts of lines are 2 - 4 % slower without it (1536 groups and more, on
// the mean of 148 products; [19104, 8128] 8 bits 16 54.5 -> 57.2), whose waves it keeps closer together, and there it stays.
template <dev::Float kF, class FS, int kCode, int kG, int kS, bool kWholeLines>
__global__ __launch_bounds__(64 * kG * kS, 4) void gemv_batch_kernel(
    const char* __restrict__ words, const char* __restrict__ scales, const char* __restrict__ x, void* __restrict__ y, int y_dtype,
    uint32_t rows, uint32_t units_per_row, uint32_t units_per_block_log2, uint32_t block_rows, uint64_t row_bytes,
    uint64_t scale_row_bytes, uint32_t scale_step, uint32_t vectors, uint32_t x_stride_bytes, uint64_t y_stride) {
    constexpr bool kPacked = kCode <= 8;
    constexpr uint32_t kM = values_per_unit(kCode) / 8;  // matrix instructions, and pieces of eight values of x, per unit
    static_assert(kM == 2 || kM == 4, "units of 16 or 32 values");
    constexpr uint32_t kQ = kU / 4;                      // a lane's units of a stage
    constexpr uint32_t kPieces = kU * kM;                // a vector's pieces of a stage
    constexpr uint32_t kCodeLoads = kCodeBytes / 1024, kScaleLoads = kU / 4, kXLoads = (16 * kPieces / 64 + kG - 1) / kG;
    extern __shared__ char lds[];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t grp = wave % kG, share = wave / kG;
    const uint32_t i = lane & 15u, g = lane >> 4;
    const uint32_t x_size = x_bytes<kCode>(vectors);
    const uint32_t buffer = kS * x_size + kG * kS * kWaveBytes;
    char* const x_img = lds + share * x_size;
    char* const code_img = lds + kS * x_size + wave * kWaveBytes;
    const uint32_t row0 = min((blockIdx.x * kG + grp) * 16u, rows - 1u);
    const bool idle = (blockIdx.x * kG + grp) * 16u >= rows;  // goes through the motions on the last row
    const uint32_t stages = (units_per_row + kU - 1u) / kU, steps = (stages + kS - 1) / kS;
    // scales of a row per stage: 2^slots_log2
    const uint32_t slots_log2 = 3u - min(units_per_block_log2, 3u);
    const uint32_t scale_loads = max(1u, (16u << slots_log2) / 64u);
    const uint32_t my_x_loads = (x_size / 1024u - grp + kG - 1u) / kG;

    // Where a lane's pieces of a stage come from: distances from bases that are uniform (the dispatch sees to it that they
    // fit).  Codes: place p of row s holds unit (p - rot) % kU, rot = s / 2 (two rows lie side by side across the
    // banks).  x: place p of vector v's blocks of 16 pieces holds piece (p - v) % 16.  Rows past the last one are the last
    // one again and never stored.
    const char* const wbase = words + row0 * row_bytes;
    const char* const sbase = scales + (row0 / block_rows) * scale_row_bytes;
    constexpr uint32_t kRowsPerLoad = 64 / kU;
    uint32_t code_row[kCodeLoads], code_unit[kCodeLoads], scale_row[kScaleLoads], x_at[kXLoads], x_piece[kXLoads];
#pragma unroll
    for (uint32_t t = 0; t < kCodeLoads; t++) {
        const uint32_t s = kRowsPerLoad * t + lane / kU;
        code_unit[t] = (lane - (s >> 1)) & (kU - 1u);
        code_row[t] = (min(row0 + s, rows - 1u) - row0) * static_cast<uint32_t>(row_bytes);
    }
#pragma unroll
    for (uint32_t n = 0; n < kScaleLoads; n++)
        scale_row[n] = (min(row0 + min((64u * n + lane) >> slots_log2, 15u), rows - 1u) / block_rows - row0 / block_rows) * static_cast<uint32_t>(scale_row_bytes);
    const uint32_t scale_slot = lane & ((1u << slots_log2) - 1u);
#pragma unroll
    for (uint32_t n = 0; n < kXLoads; n++) {
        const uint32_t pl = 64u * (grp + kG * n) + lane, v = min(pl / kPieces, vectors - 1u), in = pl % kPieces;
        x_piece[n] = (in & ~15u) | ((in - v) & 15u);
        x_at[n] = v * x_stride_bytes;
    }
    [[maybe_unused]] const bool whole_lines = ((reinterpret_cast<uintptr_t>(words) | row_bytes) & 127u) == 0;
    const auto load = [&](uint32_t stage, uint32_t into) {
        const uint32_t unit0 = stage * kU, block0 = unit0 >> units_per_block_log2;
        const bool partial = unit0 + kU > units_per_row;  // wave-uniform: units past the end are the last one again
        const uint32_t last_unit = units_per_row - 1u - unit0, last_block = ((units_per_row - 1u) >> units_per_block_log2) - block0;
        const char* const wfrom = wbase + static_cast<uint64_t>(unit0) * 16u;
        const char* const sfrom = sbase + static_cast<uint64_t>(block0) * scale_step;
        const char* const xfrom = x + static_cast<uint64_t>(unit0) * kM * 16u;
#pragma unroll
        for (uint32_t t = 0; t < kCodeLoads; t++) {
            const uint32_t unit = partial ? min(code_unit[t], last_unit) : code_unit[t];
            const u32x4* const p = reinterpret_cast<const u32x4*>(wfrom + (code_row[t] + unit * 16u));
            if (kWholeLines || (kG == 4 && whole_lines))
                __builtin_amdgcn_global_load_lds(p, CQ_LDS_PTR(code_img + into + t * 1024u), 16, 0, 2 /* nt */);
            else
                __builtin_amdgcn_global_load_lds(p, CQ_LDS_PTR(code_img + into + t * 1024u), 16, 0, 0);
        }
        const uint32_t slot = partial ? min(scale_slot, last_block) : scale_slot;
#pragma unroll
        for (uint32_t n = 0; n < kScaleLoads; n++)
            if (n < scale_loads) {
                const char* const p = sfrom + (scale_row[n] + slot * scale_step);
                if constexpr (sizeof(FS) == 4)
                    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t*>(p), CQ_LDS_PTR(code_img + into + kCodeBytes + n * 256u), 4, 0, 0);
                else
                    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint16_t*>(p), CQ_LDS_PTR(code_img + into + kCodeBytes + n * 256u), 2, 0, 0);
            }
#pragma unroll
        for (uint32_t n = 0; n < kXLoads; n++)
            if (n < my_x_loads) {
                const uint32_t piece = partial ? min(x_piece[n], last_unit * kM + kM - 1u) : x_piece[n];
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const u32x4*>(xfrom + (x_at[n] + piece * 16u)), CQ_LDS_PTR(x_img + into + (grp + kG * n) * 1024u),
                                                 16, 0, 0);
            }
    };

    const uint32_t col = min(i, vectors - 1u);  // columns past the vectors repeat the last one
    f32x4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    const auto work = [&](uint32_t stage, uint32_t from) {
        const char* const x_mine = x_img + from + col * (kPieces * 16u);
        const char* const codes = code_img + from + i * (kU * 16u);
        const char* const slots = code_img + from + kCodeBytes + (i << (slots_log2 + 2u));
        // everything a stage needs is asked of LDS at once, in the order of use (a word per scale: 16-bit ones alone in theirs)
        FS stored[kQ];
        u32x4 w[kQ], xb[kQ][kM];
#pragma unroll
        for (uint32_t q = 0; q < kQ; q++)
            stored[q] = *reinterpret_cast<const FS*>(slots + ((4u * q + g) >> (3u - slots_log2)) * 4u);
#pragma unroll
        for (uint32_t q = 0; q < kQ; q++) {
            w[q] = *reinterpret_cast<const u32x4*>(codes + ((4u * q + g + (i >> 1)) & (kU - 1u)) * 16u);
#pragma unroll
            for (uint32_t m = 0; m < kM; m++) {
                const uint32_t p = (4u * q + g) * kM + m;
                xb[q][m] = *reinterpret_cast<const u32x4*>(x_mine + (p >> 4) * 256u + ((p + col) & 15u) * 16u);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (stage * kU + kU > units_per_row) {  // wave-uniform: units past the row's end count nothing
#pragma unroll
            for (uint32_t q = 0; q < kQ; q++) {
                const bool past = stage * kU + 4u * q + g >= units_per_row;
                w[q] = past ? u32x4{0, 0, 0, 0} : w[q];
                stored[q] = past ? static_cast<FS>(1.0f) : stored[q];
#pragma unroll
                for (uint32_t m = 0; m < kM; m++) xb[q][m] = past ? u32x4{0, 0, 0, 0} : xb[q][m];
            }
        }
        float sc[kQ];
        uint32_t largest = 0;
#pragma unroll
        for (uint32_t q = 0; q < kQ; q++) {
            sc[q] = dev::round_to<kF>(dev::widen(stored[q]));
            if (kPacked) largest = max(largest, __builtin_bit_cast(uint32_t, sc[q]) & 0x7fffffffu);
        }
        if (!kPacked || __builtin_amdgcn_ballot_w64(largest >= kShortBelow<kF, kCode>) == 0) {  // ordinary scales all are
#pragma unroll
            for (uint32_t q = 0; q < kQ; q++)
#pragma unroll
                for (uint32_t m = 0; m < kM; m++) acc[m % 2] = mfma<kF>(operand<kF, kCode, true>(w[q], m, sc[q]), xb[q][m], acc[m % 2]);
        } else {
#pragma unroll 1
            for (uint32_t qm = 0; qm < kQ * kM; qm++) {  // one copy of the general code: its operands are picked out
                u32x4 word = {0, 0, 0, 0}, b = xb[0][0];
                float scale = sc[0];
#pragma unroll
                for (uint32_t k = 0; k < kQ * kM; k++)
                    if (qm == k) {
                        b = xb[k / kM][k % kM], scale = sc[k / kM];
                        word = kM == 4 ? u32x4{w[k / kM][k % kM], 0, 0, 0} : u32x4{w[k / kM][2 * (k % kM)], w[k / kM][2 * (k % kM) + 1], 0, 0};
                    }
                acc[0] = mfma<kF>(operand<kF, kCode, false>(word, 0, scale), b, acc[0]);
            }
        }
    };
    load(min(share, stages - 1u), 0);
    for (uint32_t n = 0; n < steps; n++) {
        const uint32_t from = (n & 1u) * buffer;
        // Stage n is there, and everybody has read the stage before it, whose place the next load takes.  The reads are waited
        // for here and not only where their values are used: nothing else keeps those uses in front of the barrier.
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (n + 1 < steps) load(min((n + 1) * kS + share, stages - 1u), buffer - from);
        if (n * kS + share < stages) work(n * kS + share, from);
    }
    f32x4 sum = acc[0] + acc[1];  // sum[r] = (row 4 g + r, vector i)
    if constexpr (kS > 1) {
        __syncthreads();
        float* const part = reinterpret_cast<float*>(lds);  // [share][group][register][lane]
#pragma unroll
        for (uint32_t r = 0; r < 4; r++)
            if (share != 0) part[(((share - 1) * kG + grp) * 4u + r) * 64u + lane] = sum[r];
        __syncthreads();
        if (share != 0) return;
#pragma unroll
        for (uint32_t s = 0; s + 1 < kS; s++)
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) sum[r] += part[((s * kG + grp) * 4u + r) * 64u + lane];
    }
#pragma unroll
    for (uint32_t r = 0; r < 4; r++)
        if (i < vectors && !idle && row0 + 4u * g + r < rows) store_y(y_dtype, y, i * y_stride + row0 + 4u * g + r, sum[r]);
}

template <dev::Float kF, class FS, int kCode, int kG, int kS, bool kWholeLines>
void launch_shape(hipStream_t s, const GemvArgs& a) {
    constexpr uint32_t kVals = values_per_unit(kCode);
    hipLaunchKernelGGL((gemv_batch_kernel<kF, FS, kCode, kG, kS, kWholeLines>), dim3((a.rows + 16 * kG - 1) / (16 * kG)),
                       dim3(64 * kG * kS), 2 * (kS * x_bytes<kCode>(a.vectors) + kG * kS * kWaveBytes), s,
                       static_cast<const char*>(a.words), static_cast<const char*>(a.scales), static_cast<const char*>(a.x), a.y, a.y_dtype,
                       a.rows, a.cols / kVals, a.block_rows == 0 ? 31u : log2_of(a.block_cols / kVals), a.block_rows == 0 ? 1u : a.block_rows,
                       a.word_pitch * 4, a.scale_stride_row * sizeof(FS), static_cast<uint32_t>(a.scale_stride_col * sizeof(FS)), a.vectors,
                       static_cast<uint32_t>(a.x_stride * 2), a.y_stride);
}

template <dev::Float kF, class FS, int kCode, bool kWholeLines>
void launch_code(hipStream_t s, const GemvArgs& a) {
    const uint32_t units = a.cols / values_per_unit(kCode), x = x_bytes<kCode>(a.vectors);
    static_assert(kU == 8, "the stages of gemv_batch_shape()");
    switch (gemv_batch_shape((a.rows + 15) / 16, x, 2 * 8 * (x + kWaveBytes), units, kCode == kCodeE4M3 || kCode == kCodeE5M2)) {
        case GemvShape::k1x8: return launch_shape<kF, FS, kCode, 1, 8, kWholeLines>(s, a);
        case GemvShape::k1x4: return launch_shape<kF, FS, kCode, 1, 4, kWholeLines>(s, a);
        case GemvShape::k2x4: return launch_shape<kF, FS, kCode, 2, 4, kWholeLines>(s, a);
        case GemvShape::k4x2: return launch_shape<kF, FS, kCode, 4, 2, kWholeLines>(s, a);
    }
}

template <dev::Float kF, class FS, bool kWholeLines>
hipError_t launch_codes(hipStream_t s, const GemvArgs& a) {
    if (a.native == 1)
        launch_code<kF, FS, kCodeE4M3, kWholeLines>(s, a);
    else if (a.native == 2)
        launch_code<kF, FS, kCodeE5M2, kWholeLines>(s, a);
    else if (a.native == 3)
        launch_code<kF, FS, kCodeE2M1x2, kWholeLines>(s, a);
    else if (a.bits == 4)
        launch_code<kF, FS, 4, kWholeLines>(s, a);
    else
        launch_code<kF, FS, 8, kWholeLines>(s, a);
    return hipGetLastError();
}

}  // namespace

// One object per type of x and of the scales (CQ_GEMV_PART names the one being compiled) and for either kind of rows
// (CQ_GEMV_LINES), so that a process loads the code of the kind it uses.
#if !defined(CQ_GEMV_LINES) || CQ_GEMV_LINES == 1
#define CQ_GEMV_BATCH_LINES(NAME, F, FS) hipError_t gemv_batch_lines_##NAME(hipStream_t s, const GemvArgs& a) { return launch_codes<dev::Float::F, FS, true>(s, a); }
#else
#define CQ_GEMV_BATCH_LINES(NAME, F, FS)
#endif
#if !defined(CQ_GEMV_LINES) || CQ_GEMV_LINES == 0
#define CQ_GEMV_BATCH_PARTS(NAME, F, FS) hipError_t gemv_batch_parts_##NAME(hipStream_t s, const GemvArgs& a) { return launch_codes<dev::Float::F, FS, false>(s, a); }
#else
#define CQ_GEMV_BATCH_PARTS(NAME, F, FS)
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 0
CQ_GEMV_BATCH_LINES(bf16_f32, BF16, float)
CQ_GEMV_BATCH_PARTS(bf16_f32, BF16, float)
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 1
CQ_GEMV_BATCH_LINES(bf16_bf16, BF16, __bf16)
CQ_GEMV_BATCH_PARTS(bf16_bf16, BF16, __bf16)
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 2
CQ_GEMV_BATCH_LINES(bf16_f16, BF16, _Float16)
CQ_GEMV_BATCH_PARTS(bf16_f16, BF16, _Float16)
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 3
CQ_GEMV_BATCH_LINES(f16_f32, F16, float)
CQ_GEMV_BATCH_PARTS(f16_f32, F16, float)
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 4
CQ_GEMV_BATCH_LINES(f16_bf16, F16, __bf16)
CQ_GEMV_BATCH_PARTS(f16_bf16, F16, __bf16)
#endif
#if !defined(CQ_GEMV_PART) || CQ_GEMV_PART == 5
CQ_GEMV_BATCH_LINES(f16_f16, F16, _Float16)
CQ_GEMV_BATCH_PARTS(f16_f16, F16, _Float16)
#endif

}  // namespace cq
