// Abs-max along one axis: out[.., 0, ..] = max_k |in[.., k, ..]|, the MaxAbs
// reduction a caller of the reference runs in front of quantize to build scales
// (crates/cubek-reduce/src/instructions/maxabs.rs:47-96, entry point
// crates/cubek-reduce/src/lib.rs:93-131).  NaN elements are ignored; abs and max
// are exact, so any evaluation order gives the same bits.
//
// A contiguous tensor is viewed as [outer, L, inner] around the reduced axis.
//   inner == 1 (innermost axis):  rows of L contiguous elements
//        rows that are 1..64 chunks long (power of two): lane groups + DPP butterfly
//        other rows of up to 512 chunks: lane groups with up to eight loads per lane
//        few long ones: a workgroup per row; others: one wave per (row, slice) with 16-byte lane-strided loads
//        rows that are not whole chunks: the same, over the aligned chunks inside each row
//   inner of at least one 16-byte chunk (a ragged end overlaps the chunk before it):
//        wide or many: one lane per (outer, inner chunk) walking L with stride `inner`
//        narrow, few:  one workgroup per (outer, tile of chunk columns, slice of L);
//                      its lanes form a [row phase][chunk column] grid, so a step
//                      reads whole rows of the tile, and combine through LDS
//        short axes: one launch of the tile kernel
// When the outputs alone give too few workgroups to fill the GPU, L is cut into
// slices whose partial maxima go to a caller-provided workspace ([slice][output])
// and a second kernel folds them (the same tile kernel over the partials).
// Partials are f32, except that those of the contiguous one-lane-per-column kernel
// are typed like the tensor (a maximum is a number of it), so that twice as many
// slices of a 16-bit tensor fit.  Strided tensors with a contiguous last dimension
// of whole chunks have kernels of their own on the same plan; anything else (less than a
// chunk of columns, strided last dimension) takes a one-wave-per-output (long axis) or
// one-thread-per-output fallback.
#include "cq_device.hpp"
#include "cq_internal.hpp"
#include "cq_launch_rules.hpp"
#include "cq_magic_div.hpp"

namespace cq {
namespace {

constexpr int kThreads = 256;

template <class F>
__device__ __forceinline__ float chunk_absmax(u32x4 raw, float acc) {
    float v[F::kPerChunk];
    F::unpack(raw, v);
#pragma unroll
    for (int i = 0; i < F::kPerChunk; i++) acc = fmaxf(acc, fabsf(v[i]));
    return acc;
}

// ---- rows, short: kGroup lanes per row ---------------------------------------
template <class F, int kGroup, int kUnroll>
__global__ __launch_bounds__(kThreads) void reduce_rows_grouped_kernel(const u32x4* __restrict__ in,
                                                                       void* __restrict__ out,
                                                                       uint64_t num_chunks) {
    const uint64_t first = static_cast<uint64_t>(blockIdx.x) * (kThreads * kUnroll) + threadIdx.x;
    u32x4 raw[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
        uint64_t c = first + static_cast<uint64_t>(u) * kThreads;
        raw[u] = stream_load(in + (c < num_chunks ? c : num_chunks - 1));
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
        const uint64_t c = first + static_cast<uint64_t>(u) * kThreads;
        float amax = group_max<kGroup>(chunk_absmax<F>(raw[u], 0.0f));
        if (c < num_chunks && (c % kGroup) == 0) F::store(out, c / kGroup, amax);
    }
}

// ---- rows of a few chunks that are not a power of two: kGroup lanes per row --------------------
// `loads` (uniform, at most kRowLoads) chunks per lane, all in flight at once; the last one of a row again for lanes past it.
// One straight piece of code per number of loads: with the loads behind conditions one by one, the compiler waited for each
// f32 load before the next and kept 238 registers (f32 [42651, 328] 28.8 us, [8192, 512] 9.2, [100000, 24] 6.0).
// Bound by HBM.  With a wave per row most of its lanes had nothing to load: f32 [42651, 328] 12.8 -> 9.5 us, [8192, 512]
// 4.8 -> 4.5, [100000, 24] 21.2 -> 4.3; bf16 [42651, 656] 14.2 -> 9.7, [8192, 1024] 4.9 -> 4.6, [100000, 48] 26.0 -> 4.4.
constexpr uint32_t kRowLoads = 8;
template <class F, int kGroup, uint32_t kLoads>
__device__ __forceinline__ float row_share_absmax(const u32x4* row, uint32_t lane, uint32_t chunks_per_row) {
    u32x4 raw[kLoads];
#pragma unroll
    for (uint32_t u = 0; u < kLoads; u++) {
        const uint32_t c = lane + u * kGroup;
        raw[u] = stream_load(row + (c < chunks_per_row ? c : chunks_per_row - 1));
    }
    __builtin_amdgcn_sched_barrier(0);  // every load ahead of the arithmetic
    float amax = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < kLoads; u++) amax = chunk_absmax<F>(raw[u], amax);
    return amax;
}
template <class F, int kGroup>
__global__ __launch_bounds__(kThreads) void reduce_rows_lanes_kernel(const u32x4* __restrict__ in, void* __restrict__ out, uint64_t rows,
                                                                     uint32_t chunks_per_row, uint32_t loads) {
    const uint64_t row = (static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x) / kGroup;
    const uint32_t lane = threadIdx.x % kGroup;
    const u32x4* const p = in + (row < rows ? row : rows - 1) * chunks_per_row;
    float amax = 0.0f;
    switch (loads) {
        case 1: amax = row_share_absmax<F, kGroup, 1>(p, lane, chunks_per_row); break;
        case 2: amax = row_share_absmax<F, kGroup, 2>(p, lane, chunks_per_row); break;
        case 3: amax = row_share_absmax<F, kGroup, 3>(p, lane, chunks_per_row); break;
        case 4: amax = row_share_absmax<F, kGroup, 4>(p, lane, chunks_per_row); break;
        case 5: amax = row_share_absmax<F, kGroup, 5>(p, lane, chunks_per_row); break;
        case 6: amax = row_share_absmax<F, kGroup, 6>(p, lane, chunks_per_row); break;
        case 7: amax = row_share_absmax<F, kGroup, 7>(p, lane, chunks_per_row); break;
        case kRowLoads: amax = row_share_absmax<F, kGroup, kRowLoads>(p, lane, chunks_per_row); break;
    }
    amax = group_max<kGroup>(amax);
    if (lane == 0 && row < rows) F::store(out, row, amax);
}

// Lanes per row for `chunks` chunks in at most kRowLoads loads: the fewest idle slots, more lanes on a tie.
inline uint32_t row_lanes(uint64_t chunks) {
    uint32_t best = kWave;
    for (uint32_t g = kWave; g >= 1; g /= 2) {
        const uint64_t loads = (chunks + g - 1) / g;
        if (loads > kRowLoads) break;
        if (loads * g < (chunks + best - 1) / best * best) best = g;
    }
    return best;
}

// The same for rows with edges, which are dealt out to the lanes too.
inline uint32_t ragged_row_lanes(uint64_t chunks) { return row_lanes(chunks) < 8 ? 8 : row_lanes(chunks); }

// ---- rows that start anywhere -------------------------------------------------------------------
// A row of `len` elements at any element: its whole aligned chunks, and the fewer than two chunks' worth of elements beside
// them.  Every access is aligned, so nothing is read twice and nothing outside the row.
template <class F>
struct RowSpan {
    const char* begin;
    const u32x4* body;   // the first aligned chunk inside the row
    uint32_t len, head, chunks;  // elements; elements in front of the body; whole chunks inside (at least one: len >= 2 chunks)
    __device__ __forceinline__ RowSpan(const void* in, uint64_t row, uint32_t row_len) : len(row_len) {
        begin = static_cast<const char*>(in) + row * row_len * F::kBytes;
        const uint32_t off = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(begin)) & 15u;
        head = off == 0 ? 0 : (16 - off) / F::kBytes;
        body = reinterpret_cast<const u32x4*>(begin + head * F::kBytes);
        chunks = (len - head) / F::kPerChunk;
    }
    // the elements beside the body, dealt out to kLanes lanes
    template <int kLanes>
    __device__ __forceinline__ float edges(uint32_t lane) const {
        float amax = 0.0f;
        const uint32_t tail = head + chunks * F::kPerChunk;  // elements from here on
#pragma unroll
        for (uint32_t u = 0; u < (2 * F::kPerChunk + kLanes - 1) / kLanes; u++) {
            const uint32_t i = lane + u * kLanes;
            const uint32_t e = i < F::kPerChunk ? i : tail + i - F::kPerChunk;
            const bool mine = i < F::kPerChunk ? e < head : e < len;
            amax = fmaxf(amax, fabsf(F::load(begin, mine ? e : 0)));  // the row's first element again where there is none
        }
        return amax;
    }
};

// Short ones: kGroup lanes per row, all loads in flight at once (reduce_rows_lanes_kernel).
template <class F, int kGroup>
__global__ __launch_bounds__(kThreads) void reduce_ragged_rows_lanes_kernel(const void* __restrict__ in, void* __restrict__ out, uint64_t rows,
                                                                            uint32_t len, uint32_t loads) {
    const uint64_t row = (static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x) / kGroup;
    const uint32_t lane = threadIdx.x % kGroup;
    const RowSpan<F> r(in, row < rows ? row : rows - 1, len);
    float amax = r.template edges<kGroup>(lane);
    switch (loads) {
#define CQ_CASE(N) case N: amax = fmaxf(amax, row_share_absmax<F, kGroup, N>(r.body, lane, r.chunks)); break;
        CQ_CASE(1) CQ_CASE(2) CQ_CASE(3) CQ_CASE(4) CQ_CASE(5) CQ_CASE(6) CQ_CASE(7) CQ_CASE(8)
#undef CQ_CASE
    }
    static_assert(kRowLoads == 8, "the cases above");
    amax = group_max<kGroup>(amax);
    if (lane == 0 && row < rows) F::store(out, row, amax);
}

// Long ones: kLanes lanes (a wave, or a workgroup of 1024) per row and slice of it; slice 0 takes the elements beside the
// body.  kPartial as in reduce_rows_wave_kernel.
template <class F, int kLanes, bool kPartial>
__global__ __launch_bounds__(kLanes > kThreads ? kLanes : kThreads) void reduce_rows_span_kernel(const void* __restrict__ in, void* __restrict__ out,
                                                                                                 uint64_t rows, uint32_t len, uint32_t slices,
                                                                                                 uint64_t pitch) {
    constexpr int kT = kLanes > kThreads ? kLanes : kThreads;
    constexpr uint32_t kUnroll = 4;
    const uint32_t lane = threadIdx.x % kLanes;
    const uint64_t job = static_cast<uint64_t>(blockIdx.x) * (kT / kLanes) + threadIdx.x / kLanes;
    if (job >= rows * slices) return;  // whole waves (kLanes of 64) leave together; a workgroup of one job never does
    const uint64_t row = job / slices;
    const uint32_t slice = static_cast<uint32_t>(job % slices);
    const RowSpan<F> r(in, row, len);
    const uint32_t per_slice = (r.chunks + slices - 1) / slices;
    const uint32_t begin = slice * per_slice;
    const uint32_t end = begin + per_slice < r.chunks ? begin + per_slice : r.chunks;
    float amax = slice == 0 ? r.template edges<kLanes>(lane) : 0.0f;
    for (uint32_t c0 = begin + lane; c0 < end; c0 += kLanes * kUnroll) {
        u32x4 raw[kUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; u++) {
            const uint32_t c = c0 + u * kLanes;
            raw[u] = stream_load(r.body + (c < end ? c : end - 1));
        }
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; u++) amax = chunk_absmax<F>(raw[u], amax);
    }
    amax = group_max<64>(amax);
    if constexpr (kLanes > kWave) {
        __shared__ float wave_max[kLanes / kWave];
        if (threadIdx.x % kWave == 0) wave_max[threadIdx.x / kWave] = amax;
        __syncthreads();
        amax = group_max<kLanes / kWave>(wave_max[threadIdx.x % (kLanes / kWave)]);
    }
    if (lane == 0) {
        if constexpr (kPartial)
            static_cast<float*>(out)[static_cast<uint64_t>(slice) * pitch + row] = amax;
        else
            F::store(out, row, amax);
    }
}

// ---- rows, long: one wave per (row, slice) --------------------------------------
// kPartial: write f32 partials [slice][row] with row pitch `pitch`; otherwise the
// final value typed F.
template <class F, bool kPartial>
__global__ __launch_bounds__(kThreads) void reduce_rows_wave_kernel(const u32x4* __restrict__ in,
                                                                    void* __restrict__ out, uint64_t rows,
                                                                    uint64_t chunks_per_row, uint32_t slices,
                                                                    uint64_t pitch) {
    constexpr int kUnroll = 4;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t job = static_cast<uint64_t>(blockIdx.x) * (kThreads / kWave) + threadIdx.x / kWave;
    if (job >= rows * slices) return;  // whole waves leave together
    const uint64_t row = job / slices;
    const uint32_t slice = static_cast<uint32_t>(job % slices);
    const uint64_t per_slice = (chunks_per_row + slices - 1) / slices;
    const uint64_t begin = slice * per_slice;
    const uint64_t end = begin + per_slice < chunks_per_row ? begin + per_slice : chunks_per_row;
    const u32x4* p = in + row * chunks_per_row;
    float amax = 0.0f;
    for (uint64_t c0 = begin + lane; c0 < end; c0 += kWave * kUnroll) {
        u32x4 raw[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint64_t c = c0 + static_cast<uint64_t>(u) * kWave;
            raw[u] = stream_load(p + (c < end ? c : end - 1));  // re-reading a chunk is harmless for max
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) amax = chunk_absmax<F>(raw[u], amax);
    }
    amax = group_max<64>(amax);
    if (lane == 0) {
        if constexpr (kPartial)
            static_cast<float*>(out)[static_cast<uint64_t>(slice) * pitch + row] = amax;
        else
            F::store(out, row, amax);
    }
}

// (Ragged rows, one wave or thread per output of single elements -> these kernels, us: axis 0 bf16 [43625, 2348] 386 -> 44.7,
// [7995, 5226] 119 -> 20.6, f16 [120, 1553] 13.4 -> 3.7; axis 1 f16 [2996, 29565] 202 -> 29.8, f32 [6153, 15671] 133 -> 63.)
// The chunks of kN columns along `inner`.  kRagged: `inner` is not a whole number of chunks, or the tensor does not start on
// one: accesses of 16 bytes at any element (global memory takes them), and the last chunk lies over the one before it, so
// that it ends with the row: its columns are reduced twice, to the same bits, and stored twice.
template <class F, bool kRagged>
struct ColumnChunks {
    uint64_t row_bytes;
    uint64_t at;  // bytes from a row's start to the lane's chunk
    __device__ __forceinline__ ColumnChunks(uint64_t inner, uint64_t j) : row_bytes(inner * F::kBytes), at(j * 16) {
        if (kRagged && at + 16 > row_bytes) at = row_bytes - 16;
    }
    __device__ __forceinline__ const char* rows(const void* in, uint64_t first) const { return static_cast<const char*>(in) + first * row_bytes + at; }
    __device__ __forceinline__ const u32x4* row(const char* p, uint64_t l) const { return reinterpret_cast<const u32x4*>(p + l * row_bytes); }
    __device__ __forceinline__ void store(char* outputs, u32x4 v) const {
        if constexpr (kRagged)
            __builtin_memcpy(outputs + at, &v, 16);
        else
            *reinterpret_cast<u32x4*>(outputs + at) = v;
    }
};

// ---- columns, wide: one lane per (slice of L, outer, inner chunk) ---------------------
// Writes one chunk typed F per lane: the result, or a partial [slice][output] (maxima are F numbers, so the partials lose
// nothing in 16 bits, and their traffic, written and read again, is halved).
// Bound by HBM; kColsUnroll loads of 16 bytes per lane in flight.  `per_slice`: rows_per_slice().
constexpr int kColsUnroll = 8;
template <class F, bool kRagged>
__global__ __launch_bounds__(kThreads) void reduce_cols_kernel(const u32x4* __restrict__ in, void* __restrict__ out,
                                                               uint64_t outer, uint64_t len, uint64_t inner,
                                                               uint32_t slices, uint64_t per_slice, uint64_t pitch) {
    constexpr int kN = F::kPerChunk;
    constexpr int kUnroll = kColsUnroll;
    const uint64_t inner_chunks = (inner + kN - 1) / kN;
    const uint64_t cols = outer * inner_chunks;  // output chunks
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= cols * slices) return;
    const uint32_t slice = static_cast<uint32_t>(t / cols);
    const uint64_t col = t % cols;
    const uint64_t o = col / inner_chunks, j = col % inner_chunks;
    const uint64_t begin = slice * per_slice;
    const uint64_t end = begin + per_slice < len ? begin + per_slice : len;
    const ColumnChunks<F, kRagged> at(inner, j);
    const char* p = at.rows(in, o * len);
    float amax[kN];
#pragma unroll
    for (int i = 0; i < kN; i++) amax[i] = 0.0f;
    for (uint64_t l0 = begin; l0 < end; l0 += kUnroll) {
        u32x4 raw[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint64_t l = l0 + u < end ? l0 + u : end - 1;
            raw[u] = stream_load(at.row(p, l));
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            float v[kN];
            F::unpack(raw[u], v);
#pragma unroll
            for (int i = 0; i < kN; i++) amax[i] = fmaxf(amax[i], fabsf(v[i]));
        }
    }
    at.store(static_cast<char*>(out) + (static_cast<uint64_t>(slice) * pitch + o * inner) * F::kBytes, F::pack(amax));  // values are F numbers: packing is exact
}

// ---- columns, few outputs: one workgroup per (outer, column tile, slice of L) ----------
// Lanes form a [kT / kCW row phases][kCW chunk columns] grid.  FIn is the type read
// (F32 when folding partials), FOut the type of the final result.  kAhead: the next loads go out before the previous ones are
// folded (reduce_loads_ahead() says where).
enum TileOut { kTileFinalPacked = 0, kTilePartial = 1, kTileFinalChecked = 2 };

template <class FIn, class FOut, int kCW, int kT, int kMode, bool kRagged, bool kAhead>
__global__ __launch_bounds__(kT) void reduce_tile_kernel(const u32x4* __restrict__ in, void* __restrict__ out,
                                                         uint64_t len, uint64_t inner, uint32_t col_tiles,
                                                         uint32_t slices, uint64_t pitch, uint64_t count) {
    static_assert(kCW >= 1 && kCW <= kWave && kT % kWave == 0, "a tile row fits in one wave");
    constexpr int kN = FIn::kPerChunk;
    constexpr int kRH = kT / kCW;
    constexpr int kUnroll = 4;
    constexpr int kWaves = kT / kWave;
    const uint64_t job = blockIdx.x;
    // column tiles vary fastest: workgroups in flight together read whole rows, which
    // spreads their requests over all memory channels
    const uint32_t tile = static_cast<uint32_t>(job % col_tiles);
    const uint32_t slice = static_cast<uint32_t>((job / col_tiles) % slices);
    const uint64_t o = job / col_tiles / slices;
    const uint32_t cx = threadIdx.x % kCW, ry = threadIdx.x / kCW;
    const uint64_t j = static_cast<uint64_t>(tile) * kCW + cx;
    const uint64_t per_slice = (len + slices - 1) / slices;
    const uint64_t begin = slice * per_slice;
    const uint64_t end = begin + per_slice < len ? begin + per_slice : len;
    const uint64_t inner_chunks = (inner + kN - 1) / kN;
    const ColumnChunks<FIn, kRagged> at(inner, j < inner_chunks ? j : inner_chunks - 1);
    const char* p = at.rows(in, o * len);
    float amax[kN];
#pragma unroll
    for (int i = 0; i < kN; i++) amax[i] = 0.0f;
    const auto load = [&](u32x4 (&raw)[kUnroll], uint64_t l0) {
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint64_t l = l0 + static_cast<uint64_t>(u) * kRH;
            raw[u] = stream_load(at.row(p, l < end ? l : end - 1));
        }
        if constexpr (kAhead) __builtin_amdgcn_sched_barrier(0);
    };
    const auto fold = [&](const u32x4 (&raw)[kUnroll]) {
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            float v[kN];
            FIn::unpack(raw[u], v);
#pragma unroll
            for (int i = 0; i < kN; i++) amax[i] = fmaxf(amax[i], fabsf(v[i]));
        }
        if constexpr (kAhead) __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!kAhead) {
        for (uint64_t l0 = begin + ry; l0 < end; l0 += kRH * kUnroll) {
            u32x4 raw[kUnroll];
            load(raw, l0);
            fold(raw);
        }
    } else if (begin + ry < end) {
        u32x4 even[kUnroll], odd[kUnroll];
        uint64_t l0 = begin + ry;
        load(even, l0);
        for (;;) {
            l0 += kRH * kUnroll;
            if (l0 < end) load(odd, l0);
            fold(even);
            if (l0 >= end) break;
            l0 += kRH * kUnroll;
            if (l0 < end) load(even, l0);
            fold(odd);
            if (l0 >= end) break;
        }
    }
    // lanes of a wave that share a column
#pragma unroll
    for (int mask = kCW; mask < kWave; mask <<= 1) {
#pragma unroll
        for (int i = 0; i < kN; i++) amax[i] = fmaxf(amax[i], __shfl_xor(amax[i], mask, kWave));
    }
    __shared__ float lds[kWaves][kCW][kN];
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (lane < kCW) {
#pragma unroll
        for (int i = 0; i < kN; i++) lds[wave][lane][i] = amax[i];
    }
    __syncthreads();
    if (threadIdx.x >= kCW || j >= inner_chunks) return;
#pragma unroll
    for (int w = 1; w < kWaves; w++) {
#pragma unroll
        for (int i = 0; i < kN; i++) amax[i] = fmaxf(amax[i], lds[w][cx][i]);
    }
    const uint64_t first = o * inner + at.at / FIn::kBytes;  // output element of amax[0]
    if constexpr (kMode == kTilePartial) {
        float* dst = static_cast<float*>(out) + static_cast<uint64_t>(slice) * pitch + first;
#pragma unroll
        for (int i = 0; i < kN; i++) dst[i] = amax[i];
    } else if constexpr (kMode == kTileFinalPacked) {
        at.store(static_cast<char*>(out) + o * inner * FOut::kBytes, FOut::pack(amax));
    } else {
#pragma unroll
        for (int i = 0; i < kN; i++)
            if (first + i < count) FOut::store(out, first + i, amax[i]);
    }
}

// ---- strided inputs with a contiguous last dimension ------------------------------------
// The dimensions that are not reduced, innermost first (`count` entries each, multiply-and-shift
// divisions), with their input strides in 32-bit words (rows start on multiples of 4 bytes; the 16-byte
// loads then sit off their natural alignment, which the hardware takes); the outputs are contiguous.
struct ReduceLevels {
    uint32_t levels;
    uint32_t count[CQ_MAX_RANK], magic[CQ_MAX_RANK], shift[CQ_MAX_RANK];
    uint64_t in[CQ_MAX_RANK];
};
__device__ __forceinline__ uint64_t level_offset(const ReduceLevels& r, uint32_t n) {
    uint64_t off = 0;
#pragma unroll
    for (int l = 0; l < CQ_MAX_RANK; l++) {
        if (l < static_cast<int>(r.levels)) {
            uint32_t index = n;
            if (l + 1 < static_cast<int>(r.levels)) {
                const uint32_t q = magic_div(n, r.magic[l], r.shift[l]);
                index = n - q * r.count[l];
                n = q;
            }
            off += index * r.in[l];
        }
    }
    return off;
}

__device__ __forceinline__ const u32x4* words_at(const u32x4* base, uint64_t words) {
    return reinterpret_cast<const u32x4*>(reinterpret_cast<const uint32_t*>(base) + words);
}

// reduce_rows_grouped_kernel with the rows (all dimensions but the last) found through `r`
template <class F, int kGroup, int kUnroll>
__global__ __launch_bounds__(kThreads) void reduce_rows_grouped_strided_kernel(const u32x4* __restrict__ in,
                                                                               void* __restrict__ out, ReduceLevels r,
                                                                               uint64_t num_chunks) {
    const uint64_t first = static_cast<uint64_t>(blockIdx.x) * (kThreads * kUnroll) + threadIdx.x;
    u32x4 raw[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
        uint64_t c = first + static_cast<uint64_t>(u) * kThreads;
        c = c < num_chunks ? c : num_chunks - 1;
        raw[u] = stream_load(words_at(in, level_offset(r, static_cast<uint32_t>(c / kGroup))) + c % kGroup);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
        const uint64_t c = first + static_cast<uint64_t>(u) * kThreads;
        float amax = group_max<kGroup>(chunk_absmax<F>(raw[u], 0.0f));
        if (c < num_chunks && (c % kGroup) == 0) F::store(out, c / kGroup, amax);
    }
}

// reduce_rows_wave_kernel with the rows found through `r`
template <class F, bool kPartial>
__global__ __launch_bounds__(kThreads) void reduce_rows_wave_strided_kernel(const u32x4* __restrict__ in,
                                                                            void* __restrict__ out, ReduceLevels r,
                                                                            uint64_t rows, uint64_t chunks_per_row,
                                                                            uint32_t slices, uint64_t pitch) {
    constexpr int kUnroll = 4;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t job = static_cast<uint64_t>(blockIdx.x) * (kThreads / kWave) + threadIdx.x / kWave;
    if (job >= rows * slices) return;  // whole waves leave together
    const uint64_t row = job / slices;
    const uint32_t slice = static_cast<uint32_t>(job % slices);
    const uint64_t per_slice = (chunks_per_row + slices - 1) / slices;
    const uint64_t begin = slice * per_slice;
    const uint64_t end = begin + per_slice < chunks_per_row ? begin + per_slice : chunks_per_row;
    const u32x4* p = words_at(in, level_offset(r, static_cast<uint32_t>(row)));
    float amax = 0.0f;
    for (uint64_t c0 = begin + lane; c0 < end; c0 += kWave * kUnroll) {
        u32x4 raw[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint64_t c = c0 + static_cast<uint64_t>(u) * kWave;
            raw[u] = stream_load(p + (c < end ? c : end - 1));
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) amax = chunk_absmax<F>(raw[u], amax);
    }
    amax = group_max<64>(amax);
    if (lane == 0) {
        if constexpr (kPartial)
            static_cast<float*>(out)[static_cast<uint64_t>(slice) * pitch + row] = amax;
        else
            F::store(out, row, amax);
    }
}

// reduce_cols_kernel with the output chunks (the last dimension in chunks, then the other kept
// dimensions) found through `r`; the reduced axis steps `len_stride` words
template <class F, bool kPartial>
__global__ __launch_bounds__(kThreads) void reduce_cols_strided_kernel(const u32x4* __restrict__ in, void* __restrict__ out,
                                                                       ReduceLevels r, uint64_t cols, uint64_t len,
                                                                       uint64_t len_stride, uint32_t slices) {
    constexpr int kN = F::kPerChunk;
    constexpr int kUnroll = 4;
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= cols * slices) return;
    const uint32_t slice = static_cast<uint32_t>(t / cols);
    const uint64_t col = t % cols;
    const uint64_t per_slice = (len + slices - 1) / slices;
    const uint64_t begin = slice * per_slice;
    const uint64_t end = begin + per_slice < len ? begin + per_slice : len;
    const u32x4* p = words_at(in, level_offset(r, static_cast<uint32_t>(col)));
    float amax[kN];
#pragma unroll
    for (int i = 0; i < kN; i++) amax[i] = 0.0f;
    for (uint64_t l0 = begin; l0 < end; l0 += kUnroll) {
        u32x4 raw[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const uint64_t l = l0 + u < end ? l0 + u : end - 1;
            raw[u] = stream_load(words_at(p, l * len_stride));
        }
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            float v[kN];
            F::unpack(raw[u], v);
#pragma unroll
            for (int i = 0; i < kN; i++) amax[i] = fmaxf(amax[i], fabsf(v[i]));
        }
    }
    if constexpr (kPartial) {
        float* dst = static_cast<float*>(out) + (static_cast<uint64_t>(slice) * cols + col) * kN;
#pragma unroll
        for (int i = 0; i < kN; i++) dst[i] = amax[i];
    } else {
        static_cast<u32x4*>(out)[col] = F::pack(amax);
    }
}

// ---- fallbacks: any strides -----------------------------------------------------------
struct StridedReduce {
    uint32_t rank, axis;
    uint32_t shape[CQ_MAX_RANK];
    uint64_t in_strides[CQ_MAX_RANK];
    uint64_t out_strides[CQ_MAX_RANK];
};

// kLanes lanes per output element (1 or a whole wave), elements [first, num_out)
template <class F, int kLanes>
__global__ __launch_bounds__(kThreads) void reduce_strided_kernel(const void* __restrict__ in,
                                                                  void* __restrict__ out, StridedReduce r,
                                                                  uint64_t first, uint64_t num_out) {
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const uint64_t i = first + t / kLanes;
    const uint32_t lane = static_cast<uint32_t>(t % kLanes);
    if (i >= num_out) return;  // kLanes divides the wave: whole groups leave together
    uint64_t rem = i, in_off = 0, out_off = 0;
    for (int d = static_cast<int>(r.rank) - 1; d >= 0; d--) {
        if (static_cast<uint32_t>(d) == r.axis) continue;
        const uint64_t c = rem % r.shape[d];
        rem /= r.shape[d];
        in_off += c * r.in_strides[d];
        out_off += c * r.out_strides[d];
    }
    float m = 0.0f;
    for (uint32_t k = lane; k < r.shape[r.axis]; k += kLanes)
        m = fmaxf(m, fabsf(F::load(in, in_off + static_cast<uint64_t>(k) * r.in_strides[r.axis])));
    m = group_max<kLanes>(m);
    if (lane == 0) F::store(out, out_off, m);
}

// Output element i, first <= i < num_out, of a contiguous result -> its place in a strided output tensor.
template <class F>
__global__ __launch_bounds__(kThreads) void scatter_outputs_kernel(const void* __restrict__ packed, void* __restrict__ out,
                                                                   StridedReduce r, uint64_t first, uint64_t num_out) {
    const uint64_t i = first + static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= num_out) return;
    uint64_t rem = i, out_off = 0;
    for (int d = static_cast<int>(r.rank) - 1; d >= 0; d--) {
        if (static_cast<uint32_t>(d) == r.axis) continue;
        const uint64_t c = rem % r.shape[d];
        rem /= r.shape[d];
        out_off += c * r.out_strides[d];
    }
    if constexpr (F::kBytes == 4)
        static_cast<uint32_t*>(out)[out_off] = static_cast<const uint32_t*>(packed)[i];
    else
        static_cast<uint16_t*>(out)[out_off] = static_cast<const uint16_t*>(packed)[i];
}

// bytes of the workspace that hold the contiguous result of a launch whose output tensor is strided
inline uint64_t packed_outputs_bytes(uint64_t num_out, uint64_t elem_bytes) { return (num_out * elem_bytes + 255) / 256 * 256; }

inline dim3 blocks(uint64_t n, uint64_t per_block) { return dim3(static_cast<uint32_t>((n + per_block - 1) / per_block)); }
inline uint64_t round_up(uint64_t v, uint64_t m) { return (v + m - 1) / m * m; }

// enough workgroups / lanes to keep 256 CUs busy
constexpr uint64_t kTargetGroups = 2048;
constexpr uint64_t kTargetLanes = kTargetGroups * kThreads / 2;

// Rows per lane of reduce_cols_kernel with at most `most` slices over `cols` columns of chunks.  Its few workgroups all run
// at once, so a launch lasts as long as the compute unit with the most of them: of two to four workgroups per compute unit
// the split with the least work there, rows in whole loops of kColsUnroll (a last loop of one row loads eight) and eight rows'
// worth for a slice's start and end.  The workgroups do not spread evenly, so a round counts 238 of the 256 units: bf16
// [30000, 3000], workgroups per unit 1.65 34.3, 1.79 33.7, 1.95 39.7, 2.15 38.9, 2.68 35.4 us; [3000, 20008] 1.79 22.6, 2.06
// 26.8, 2.86 23.5 us.  Against slices of even rows, capped by the partials' bytes alone: bf16 [4093, 11008] 19.1 -> 17.1 us,
// f16 [1686, 18520] 16.4 -> 14.5 us, bf16 [30000, 3000] 36.6 -> 33.7 us.
inline uint64_t rows_per_slice(uint64_t len, uint64_t cols, uint64_t most) {
    constexpr uint64_t kRound = 238 * kThreads, kSliceCost = 8;
    uint64_t best = len, best_cost = (cols + kRound - 1) / kRound * (len + kSliceCost);
    for (uint64_t rounds = 2; rounds <= 4; rounds++) {
        uint64_t n = rounds * kRound / cols;
        if (n > (len + 15) / 16) n = (len + 15) / 16;
        if (n > most) n = most;
        if (n < 2) continue;
        const uint64_t rows = round_up((len + n - 1) / n, kColsUnroll), slices = (len + rows - 1) / rows;
        const uint64_t cost = (slices * cols + kRound - 1) / kRound * (rows + kSliceCost);
        if (cost < best_cost) best = rows, best_cost = cost;
    }
    return best;
}

// Rows so few that they would be sliced, with a workgroup to each instead: one launch, no fold (sliced -> one launch, us):
// f16 [6, 25952] 5.7 -> 3.2, f32 [237, 29888] 10.1 -> 6.6, [1500, 32768] 39.5 -> 32.4, bf16 [439, 5504] 6.9 -> 4.0, [500,
// 131072] 26.8 -> 22.9.  Not where one workgroup would read for longer than the fold takes: bf16 [32, 131072] 6.1 -> 7.1,
// [64, 2^20] 26.8 -> 45.0.  256 lanes up to 2048 chunks: of 1024 lanes with four loads each most would read a chunk again.
inline bool block_per_row(uint64_t rows, uint64_t chunks) { return chunks <= 8192 || (chunks <= 16384 && rows >= 256); }
constexpr uint64_t kNarrowBlockRowChunks = 2048;

// How a contiguous [outer, len, inner] view is cut up; shared by the launcher and
// by the workspace size query so that the two always agree.
struct ReducePlan {
    enum Kind { kFallback, kRowsGrouped, kRowsWave, kCols, kTile } kind = kFallback;
    bool ragged = false;  // rows, or rows of columns, that are not whole chunks
    uint64_t chunks_per_row = 0, inner_chunks = 0;  // ragged: whole chunks of a row; chunks that cover the columns
    uint32_t cw = 1, col_tiles = 1;
    uint64_t slices = 1;  // wanted; the launcher lowers it to what the workspace holds
    bool long_axis = false;  // columns: more slices than one, if the partials' bytes allow them
    uint64_t lane_slices = 1;  // kTile on a strided input (one lane per output chunk and slice instead): wanted there
    uint64_t pitch = 0;   // partials per slice
};

ReducePlan plan_reduce(uint64_t outer, uint64_t len, uint64_t inner, uint64_t kN) {
    ReducePlan p;
    // f32 partials of all slices stay below 1/32 of the bytes read; the workspace is sized for these (partials typed like
    // a 16-bit tensor are twice as many in the same bytes)
    const uint64_t traffic_cap = len * (16 / kN) / 128 > 0 ? len * (16 / kN) / 128 : 1;
    if (len == 0 || outer == 0 || inner == 0) return p;
    p.ragged = (inner == 1 ? len : inner) % kN != 0;
    if (inner == 1) {
        if (len < 2 * kN && p.ragged) return p;
        p.chunks_per_row = len / kN;
        if (!p.ragged && p.chunks_per_row <= 64 && (p.chunks_per_row & (p.chunks_per_row - 1)) == 0) {
            p.kind = ReducePlan::kRowsGrouped;
            return p;
        }
        p.kind = ReducePlan::kRowsWave;
        p.pitch = round_up(outer, 4);
        if (outer * kWave < kTargetLanes) {
            p.slices = kTargetLanes / (outer * kWave);
            const uint64_t max_slices = (p.chunks_per_row + 8 * kWave - 1) / (8 * kWave);  // >= 8 KiB per wave and slice
            if (p.slices > max_slices) p.slices = max_slices;
            if (p.slices > traffic_cap) p.slices = traffic_cap;
        }
        return p;
    }
    if (inner < kN) return p;
    p.inner_chunks = (inner + kN - 1) / kN;
    const uint64_t cols = outer * p.inner_chunks;
    if (cols >= kTargetLanes || p.inner_chunks >= kThreads) {
        p.kind = ReducePlan::kCols;
        p.pitch = round_up(outer * inner, kN);
        if (cols < kTargetLanes) {
            p.slices = kTargetLanes / cols;
            const uint64_t max_slices = (len + 15) / 16;  // at least 16 rows per slice
            if (p.slices > max_slices) p.slices = max_slices;
            p.long_axis = p.slices > 1;
            if (p.slices > traffic_cap) p.slices = traffic_cap;
        }
        return p;
    }
    p.kind = ReducePlan::kTile;
    p.lane_slices = kTargetLanes / cols;
    if (p.lane_slices > (len + 15) / 16) p.lane_slices = (len + 15) / 16;
    if (p.lane_slices > traffic_cap) p.lane_slices = traffic_cap;
    if (p.lane_slices < 1) p.lane_slices = 1;
    p.cw = pow2_at_least(p.inner_chunks, kWave);
    p.col_tiles = static_cast<uint32_t>((p.inner_chunks + p.cw - 1) / p.cw);
    p.pitch = round_up(outer * inner, kN);  // whole chunks of partials
    const uint64_t base = outer * p.col_tiles;
    if (base < kTargetGroups) {
        p.slices = kTargetGroups / base;
        const uint64_t rows_per_step = kThreads / p.cw * 4;  // rows one workgroup reads per loop trip
        const uint64_t max_slices = (len + 2 * rows_per_step - 1) / (2 * rows_per_step);
        if (p.slices > max_slices) p.slices = max_slices;
        p.long_axis = p.slices > 1;
        if (p.slices > traffic_cap) p.slices = traffic_cap;
    }
    return p;
}

// kWidest, kNarrowest: of the tiles that the caller asks for
template <class FIn, class FOut, int kT, int kMode, int kWidest = kWave, bool kAhead = false, int kNarrowest = 1>
void launch_tile(hipStream_t s, bool ragged, uint32_t cw, uint64_t jobs, const void* in, void* out, uint64_t len,
                 uint64_t inner, uint32_t col_tiles, uint32_t slices, uint64_t pitch, uint64_t count) {
    auto src = static_cast<const u32x4*>(in);
    dim3 grid(static_cast<uint32_t>(jobs));
    switch (cw * 2 + (ragged ? 1 : 0)) {
#define CQ_TILE(W, R) hipLaunchKernelGGL((reduce_tile_kernel<FIn, FOut, W, kT, kMode, R, kAhead>), grid, dim3(kT), 0, s, src, out, len, inner, col_tiles, slices, pitch, count)
#define CQ_CASE(W) case W * 2: if constexpr (W >= kNarrowest && W <= kWidest) CQ_TILE(W, false); break; case W * 2 + 1: if constexpr (W >= kNarrowest && W <= kWidest && kMode != kTileFinalChecked && !kAhead) CQ_TILE(W, true); break;
        CQ_CASE(1) CQ_CASE(2) CQ_CASE(4) CQ_CASE(8) CQ_CASE(16) CQ_CASE(32) CQ_CASE(64)
#undef CQ_CASE
#undef CQ_TILE
    }
}

// out[i] = max_s partials[s][i], i < count; partials are typed P (f32 or the output's type) with row pitch `pitch`
template <class F, class P = F32>
void launch_fold(hipStream_t s, const void* partials, void* out, uint64_t slices, uint64_t pitch, uint64_t count) {
    constexpr int kFoldThreads = 1024;
    const uint64_t chunks = pitch / P::kPerChunk;
    uint32_t cw = pow2_at_least(chunks, kWave);
    while (cw > 4 && chunks / cw < 128) cw /= 2;  // narrower tiles, more workgroups: the partials sit in L2
    const uint32_t tiles = static_cast<uint32_t>((chunks + cw - 1) / cw);
    launch_tile<P, F, kFoldThreads, kTileFinalChecked>(s, false, cw, tiles, partials, out, slices, pitch, tiles, 1u, 0, count);
}

// The levels of a strided input with a contiguous last dimension of whole chunks, strides of whole words and
// fewer than 2^31 rows and output chunks; false: not such a tensor.
template <class F>
bool strided_levels(const ReduceArgs& a, ReduceLevels* r, uint64_t* len_stride) {
    constexpr uint64_t kN = F::kPerChunk;
    constexpr uint64_t kWordElems = F::kBytes == 4 ? 1 : 2;  // elements per 32-bit word
    if (a.rank < 2 || (reinterpret_cast<uintptr_t>(a.input) & 3u) != 0) return false;
    const uint32_t last = a.rank - 1;
    if (a.in_strides[last] != 1 || a.shape[last] % kN != 0) return false;
    *r = ReduceLevels{};
    *len_stride = 0;
    uint64_t total = 1;
    const auto push = [&](uint64_t count, uint64_t stride) {
        const uint32_t k = r->levels;
        if (k > 0 && stride == r->in[k - 1] * r->count[k - 1] && r->count[k - 1] * count < (1ull << 31)) {
            r->count[k - 1] *= static_cast<uint32_t>(count);  // steps on uniformly from the level inside it
        } else {
            r->count[k] = static_cast<uint32_t>(count);
            r->in[k] = stride;
            r->levels = k + 1;
        }
        total *= count;
    };
    if (a.axis != last) push(a.shape[last] / kN, 4);  // a chunk is four words
    for (int d = static_cast<int>(last) - 1; d >= 0; d--) {
        if (a.in_strides[d] % kWordElems != 0 && a.shape[d] > 1) return false;
        if (static_cast<uint32_t>(d) == a.axis) {
            *len_stride = a.in_strides[d] / kWordElems;
            continue;
        }
        if (a.shape[d] == 1) continue;
        push(a.shape[d], a.in_strides[d] / kWordElems);
    }
    if (r->levels == 0) push(1, 0);
    if (total >= (1ull << 31)) return false;
    for (uint32_t l = 0; l < r->levels; l++) magic_of(r->count[l], &r->magic[l], &r->shift[l]);
    return true;
}

template <class F>
hipError_t reduce_dispatch(hipStream_t s, const ReduceArgs& a) {
    constexpr uint64_t kN = F::kPerChunk;
    // A strided output (one column of a matrix, every other element): the kernels below write a contiguous result
    // into the front of the workspace, and one more small launch puts every element in its place.  Without that much
    // workspace the launch runs one wave (or lane) per output.
    if (!a.out_contiguous) {
        const uint64_t num_out = a.outer * a.inner, front = packed_outputs_bytes(num_out, F::kBytes);
        if (a.workspace != nullptr && a.workspace_bytes >= front && num_out != 0) {
            ReduceArgs b = a;
            b.output = a.workspace;
            b.out_contiguous = true;
            b.contiguous = a.in_contiguous;
            uint64_t acc = 1;
            for (int d = static_cast<int>(a.rank) - 1; d >= 0; d--) {
                b.out_strides[d] = acc;
                if (static_cast<uint32_t>(d) != a.axis) acc *= a.shape[d];
            }
            b.workspace = static_cast<char*>(a.workspace) + front;
            b.workspace_bytes = a.workspace_bytes - front;
            if (b.workspace_bytes == 0) b.workspace = nullptr;
            const hipError_t e = reduce_dispatch<F>(s, b);
            if (e != hipSuccess) return e;
            StridedReduce r{};
            r.rank = a.rank;
            r.axis = a.axis;
            for (uint32_t d = 0; d < a.rank; d++) {
                r.shape[d] = static_cast<uint32_t>(a.shape[d]);
                r.out_strides[d] = a.out_strides[d];
            }
            in_pieces(0, num_out, 1, [&](uint64_t first, uint64_t last) {
                hipLaunchKernelGGL((scatter_outputs_kernel<F>), blocks(last - first, kThreads), dim3(kThreads), 0, s, a.workspace, a.output, r, first, last);
            });
            return hipGetLastError();
        }
    }
    ReducePlan p;
    if (a.contiguous && (reinterpret_cast<uintptr_t>(a.input) & (F::kBytes - 1)) == 0) {
        p = plan_reduce(a.outer, a.len, a.inner, kN);
        if ((reinterpret_cast<uintptr_t>(a.input) & 15u) != 0) {  // whole chunks, none of them aligned
            p.ragged = true;
            if (p.kind == ReducePlan::kRowsGrouped) p.kind = a.len < 2 * kN ? ReducePlan::kFallback : ReducePlan::kRowsWave;
        }
    }
    ReduceLevels levels;
    uint64_t len_stride = 0;
    if (!a.contiguous && a.out_contiguous && strided_levels<F>(a, &levels, &len_stride)) {
        // the plan of the contiguous tensor of this shape, with kernels that look up where rows and columns lie
        p = plan_reduce(a.outer, a.len, a.inner, kN);
        if (p.ragged) p.kind = ReducePlan::kFallback;
        const bool rows = p.kind == ReducePlan::kRowsGrouped || p.kind == ReducePlan::kRowsWave;
        const bool cols = p.kind == ReducePlan::kCols || p.kind == ReducePlan::kTile;
        if ((rows && a.axis != a.rank - 1) || (cols && (a.axis == a.rank - 1 || (reinterpret_cast<uintptr_t>(a.output) & 15u) != 0)))
            p.kind = ReducePlan::kFallback;
        uint64_t slices = p.kind == ReducePlan::kTile ? p.lane_slices : p.slices;
        if (slices > 1) {
            const uint64_t fit = a.workspace == nullptr ? 0 : a.workspace_bytes / (p.pitch * sizeof(float));
            if (slices > fit) slices = fit > 1 ? fit : 1;
        }
        auto in = static_cast<const u32x4*>(a.input);
        if (p.kind == ReducePlan::kRowsGrouped) {
            const uint64_t num_chunks = a.outer * p.chunks_per_row;
            constexpr int kU = 4;
            dim3 grid = blocks(num_chunks, kThreads * kU);
            switch (p.chunks_per_row) {
#define CQ_CASE(G) case G: hipLaunchKernelGGL((reduce_rows_grouped_strided_kernel<F, G, kU>), grid, dim3(kThreads), 0, s, in, a.output, levels, num_chunks); break;
                CQ_CASE(1) CQ_CASE(2) CQ_CASE(4) CQ_CASE(8) CQ_CASE(16) CQ_CASE(32) CQ_CASE(64)
#undef CQ_CASE
            }
            return hipGetLastError();
        }
        if (p.kind == ReducePlan::kRowsWave) {
            dim3 grid = blocks(a.outer * slices, kThreads / kWave);
            if (slices > 1) {
                hipLaunchKernelGGL((reduce_rows_wave_strided_kernel<F, true>), grid, dim3(kThreads), 0, s, in, a.workspace,
                                   levels, a.outer, p.chunks_per_row, static_cast<uint32_t>(slices), p.pitch);
                launch_fold<F>(s, a.workspace, a.output, slices, p.pitch, a.outer);
            } else {
                hipLaunchKernelGGL((reduce_rows_wave_strided_kernel<F, false>), grid, dim3(kThreads), 0, s, in, a.output,
                                   levels, a.outer, p.chunks_per_row, 1u, 0);
            }
            return hipGetLastError();
        }
        if (cols && p.kind != ReducePlan::kFallback) {
            const uint64_t out_chunks = a.outer * p.inner_chunks;
            dim3 grid = blocks(out_chunks * slices, kThreads);
            if (slices > 1) {
                hipLaunchKernelGGL((reduce_cols_strided_kernel<F, true>), grid, dim3(kThreads), 0, s, in, a.workspace, levels,
                                   out_chunks, a.len, len_stride, static_cast<uint32_t>(slices));
                launch_fold<F>(s, a.workspace, a.output, slices, p.pitch, p.pitch);  // whole chunks: no padding
            } else {
                hipLaunchKernelGGL((reduce_cols_strided_kernel<F, false>), grid, dim3(kThreads), 0, s, in, a.output, levels,
                                   out_chunks, a.len, len_stride, 1u);
            }
            return hipGetLastError();
        }
        p = ReducePlan{};
    }
    if ((p.kind == ReducePlan::kCols || p.kind == ReducePlan::kTile) && (reinterpret_cast<uintptr_t>(a.output) & 15u) != 0) {
        p.ragged = true;  // the kernels whose stores need not be aligned either
        if ((reinterpret_cast<uintptr_t>(a.output) & (F::kBytes - 1)) != 0) p.kind = ReducePlan::kFallback;
    }
    uint64_t slices = p.slices;
    if (slices > 1) {
        const uint64_t fit = a.workspace == nullptr ? 0 : a.workspace_bytes / (p.pitch * sizeof(float));
        if (slices > fit) slices = fit > 1 ? fit : 1;
    }
    if (p.kind == ReducePlan::kCols || p.kind == ReducePlan::kTile) {
        ReduceColumns c{};
        c.outer = a.outer, c.len = a.len, c.inner = a.inner, c.per_chunk = kN;
        c.ragged = p.ragged, c.tiles = p.kind == ReducePlan::kTile ? a.outer * p.col_tiles : 0;
        c.long_axis = p.long_axis, c.wanted = p.slices, c.slices = slices;
        const ReduceTile tile = reduce_tile(c);
        switch (reduce_way(c)) {
            case ReduceWay::kOneLaunch: {
                // 512 lanes were the best or within 5 % of it throughout; up to 128 rows 256 of them start and end sooner (f32
                // [37, 15360] 3.2 -> 3.0 us)
                const uint32_t col_tiles = static_cast<uint32_t>(tile.col_tiles);
                if (a.len <= 128)
                    launch_tile<F, F, 256, kTileFinalPacked>(s, p.ragged, tile.cw, a.outer * tile.col_tiles, a.input, a.output, a.len, a.inner, col_tiles, 1u, 0, 0);
                else if (reduce_loads_ahead(c, tile))
                    launch_tile<F, F, 512, kTileFinalPacked, kWidestReduceTile, true, 8>(s, p.ragged, tile.cw, a.outer * tile.col_tiles, a.input, a.output, a.len, a.inner, col_tiles, 1u, 0, 0);
                else
                    launch_tile<F, F, 512, kTileFinalPacked, kWidestReduceTile>(s, p.ragged, tile.cw, a.outer * tile.col_tiles, a.input, a.output, a.len, a.inner, col_tiles, 1u, 0, 0);
                return hipGetLastError();
            }
            case ReduceWay::kPerOutput: p.kind = ReducePlan::kFallback; break;
            case ReduceWay::kPlan: break;
        }
    }
    if (p.kind == ReducePlan::kRowsWave && p.chunks_per_row <= kWave * kRowLoads &&
        a.outer * (p.ragged ? ragged_row_lanes(p.chunks_per_row) : row_lanes(p.chunks_per_row)) > kMostLanes)
        p.kind = ReducePlan::kFallback;  // one lane for each of so many short rows
    auto in = static_cast<const u32x4*>(a.input);
    switch (p.kind) {
        case ReducePlan::kRowsGrouped: {
            const uint64_t num_chunks = a.outer * p.chunks_per_row;
            constexpr int kU = 4;
            dim3 grid = blocks(num_chunks, kThreads * kU);
            switch (p.chunks_per_row) {
#define CQ_CASE(G) case G: hipLaunchKernelGGL((reduce_rows_grouped_kernel<F, G, kU>), grid, dim3(kThreads), 0, s, in, a.output, num_chunks); break;
                CQ_CASE(1) CQ_CASE(2) CQ_CASE(4) CQ_CASE(8) CQ_CASE(16) CQ_CASE(32) CQ_CASE(64)
#undef CQ_CASE
            }
            return hipGetLastError();
        }
        case ReducePlan::kRowsWave: {
            dim3 grid = blocks(a.outer * slices, kThreads / kWave);
            const uint32_t len = static_cast<uint32_t>(a.len);
            if (p.slices > 1 && block_per_row(a.outer, p.chunks_per_row)) {
                const dim3 rows(static_cast<uint32_t>(a.outer));
                if (p.chunks_per_row <= kNarrowBlockRowChunks)
                    hipLaunchKernelGGL((reduce_rows_span_kernel<F, 256, false>), rows, dim3(256), 0, s, a.input, a.output, a.outer, len, 1u, 0);
                else
                    hipLaunchKernelGGL((reduce_rows_span_kernel<F, 1024, false>), rows, dim3(1024), 0, s, a.input, a.output, a.outer, len, 1u, 0);
                return hipGetLastError();
            }
            if (p.ragged) {
                if (slices > 1) {
                    hipLaunchKernelGGL((reduce_rows_span_kernel<F, kWave, true>), grid, dim3(kThreads), 0, s, a.input, a.workspace, a.outer,
                                       len, static_cast<uint32_t>(slices), p.pitch);
                    launch_fold<F>(s, a.workspace, a.output, slices, p.pitch, a.outer);
                } else if (p.chunks_per_row <= kWave * kRowLoads) {
                    const uint32_t lanes = ragged_row_lanes(p.chunks_per_row);
                    const uint32_t loads = static_cast<uint32_t>((p.chunks_per_row + lanes - 1) / lanes);
                    switch (lanes) {
#define CQ_CASE(G) case G: hipLaunchKernelGGL((reduce_ragged_rows_lanes_kernel<F, G>), blocks(a.outer * G, kThreads), dim3(kThreads), 0, s, a.input, a.output, a.outer, len, loads); break;
                        CQ_CASE(8) CQ_CASE(16) CQ_CASE(32) CQ_CASE(64)
#undef CQ_CASE
                    }
                } else {
                    hipLaunchKernelGGL((reduce_rows_span_kernel<F, kWave, false>), grid, dim3(kThreads), 0, s, a.input, a.output, a.outer, len,
                                       1u, 0);
                }
                return hipGetLastError();
            }
            if (slices <= 1 && p.chunks_per_row <= kWave * kRowLoads) {
                const uint32_t lanes = row_lanes(p.chunks_per_row), loads = static_cast<uint32_t>((p.chunks_per_row + lanes - 1) / lanes);
                switch (lanes) {
#define CQ_CASE(G) case G: hipLaunchKernelGGL((reduce_rows_lanes_kernel<F, G>), blocks(a.outer * G, kThreads), dim3(kThreads), 0, s, in, a.output, a.outer, static_cast<uint32_t>(p.chunks_per_row), loads); break;
                    CQ_CASE(1) CQ_CASE(2) CQ_CASE(4) CQ_CASE(8) CQ_CASE(16) CQ_CASE(32) CQ_CASE(64)
#undef CQ_CASE
                }
                return hipGetLastError();
            }
            if (slices > 1) {
                hipLaunchKernelGGL((reduce_rows_wave_kernel<F, true>), grid, dim3(kThreads), 0, s, in, a.workspace, a.outer,
                                   p.chunks_per_row, static_cast<uint32_t>(slices), p.pitch);
                launch_fold<F>(s, a.workspace, a.output, slices, p.pitch, a.outer);
            } else {
                hipLaunchKernelGGL((reduce_rows_wave_kernel<F, false>), grid, dim3(kThreads), 0, s, in, a.output, a.outer,
                                   p.chunks_per_row, 1u, 0);
            }
            return hipGetLastError();
        }
        case ReducePlan::kCols: {
            uint64_t per_slice = a.len;
            if (slices > 1) {
                // the workspace of p.slices in f32 holds twice as many typed in 16 bits
                const uint64_t fit = a.workspace_bytes / (p.pitch * F::kBytes), most = p.slices * (4 / F::kBytes);
                per_slice = rows_per_slice(a.len, a.outer * p.inner_chunks, fit < most ? fit : most);
                slices = (a.len + per_slice - 1) / per_slice;
            }
            const dim3 grid = blocks(a.outer * p.inner_chunks * slices, kThreads);
            void* const dst = slices > 1 ? a.workspace : a.output;
            if (p.ragged)
                hipLaunchKernelGGL((reduce_cols_kernel<F, true>), grid, dim3(kThreads), 0, s, in, dst, a.outer, a.len, a.inner,
                                   static_cast<uint32_t>(slices), per_slice, p.pitch);
            else
                hipLaunchKernelGGL((reduce_cols_kernel<F, false>), grid, dim3(kThreads), 0, s, in, dst, a.outer, a.len, a.inner,
                                   static_cast<uint32_t>(slices), per_slice, p.pitch);
            if (slices > 1) launch_fold<F, F>(s, a.workspace, a.output, slices, p.pitch, a.outer * a.inner);
            return hipGetLastError();
        }
        case ReducePlan::kTile: {
            const uint64_t jobs = a.outer * p.col_tiles * slices;
            const uint32_t n = static_cast<uint32_t>(slices);
            if (slices > 1) {
                launch_tile<F, F, kThreads, kTilePartial>(s, p.ragged, p.cw, jobs, a.input, a.workspace, a.len, a.inner, p.col_tiles, n, p.pitch, 0);
                launch_fold<F>(s, a.workspace, a.output, slices, p.pitch, a.outer * a.inner);
            } else {
                launch_tile<F, F, kThreads, kTileFinalPacked>(s, p.ragged, p.cw, jobs, a.input, a.output, a.len, a.inner, p.col_tiles, 1u, 0, 0);
            }
            return hipGetLastError();
        }
        case ReducePlan::kFallback: break;
    }
    StridedReduce r{};
    r.rank = a.rank;
    r.axis = a.axis;
    uint64_t num_out = 1;
    for (uint32_t d = 0; d < a.rank; d++) {
        r.shape[d] = static_cast<uint32_t>(a.shape[d]);
        r.in_strides[d] = a.in_strides[d];
        r.out_strides[d] = a.out_strides[d];
        if (d != a.axis) num_out *= a.shape[d];
    }
    if (num_out == 0) return hipSuccess;
    const uint64_t lanes = a.shape[a.axis] >= 256 ? kWave : 1;
    in_pieces(0, num_out, lanes, [&](uint64_t first, uint64_t last) {
        const auto kernel = lanes == kWave ? reduce_strided_kernel<F, kWave> : reduce_strided_kernel<F, 1>;
        hipLaunchKernelGGL(kernel, blocks((last - first) * lanes, kThreads), dim3(kThreads), 0, s, a.input, a.output, r, first, last);
    });
    return hipGetLastError();
}

}  // namespace

uint64_t reduce_workspace_bytes(uint64_t outer, uint64_t len, uint64_t inner, int dtype) {
    const ReducePlan p = plan_reduce(outer, len, inner, dtype == CQ_F32 ? 4 : 8);
    const uint64_t slices = p.slices > p.lane_slices ? p.slices : p.lane_slices;  // either kernel set may run
    // ... and room for the contiguous result of a launch whose output tensor turns out to be strided
    return (slices > 1 ? slices * p.pitch * sizeof(float) : 0) + packed_outputs_bytes(outer * inner, dtype == CQ_F32 ? 4 : 2);
}

hipError_t launch_reduce_max_abs(hipStream_t s, int dtype, const ReduceArgs& a) {
    switch (dtype) {
        case CQ_F32: return reduce_dispatch<F32>(s, a);
        case CQ_BF16: return reduce_dispatch<BF16>(s, a);
        case CQ_F16: return reduce_dispatch<F16>(s, a);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cq
