// One scale for a whole contiguous tensor, quantized in one read of it: every workgroup keeps its share of the tensor in
// registers and LDS while the abs-max of the others arrives.
//
// The two-pass quantize (absmax_partials_kernel, then quantize_flat_kernel) reads the tensor twice, and from 64 MB on the
// second read comes from memory again.  The register files and the LDS of the 256 compute units hold 168 MiB.  A workgroup of 512
// lanes with all 256 registers each fills one compute unit; it takes every 256th step of 512 chunks, loads up to 64 of
// them at once (48 stay in registers, 16 in LDS: 128 MiB), publishes the abs-max of what it read, waits for the other
// workgroups', and quantizes what it holds.  What a tensor has beyond that (its first steps) is read twice as before, in
// loops in front of and behind the resident part.
//
// Waiting.  A slot per workgroup holds its abs-max, or kUnset as the launch before this one leaves it.  No workgroup depends
// on another one running: one that has waited for kPatience polls works out the missing shares itself, one by one, from
// memory, and publishes them (the same bits, whoever does), so that it goes on after at most 256 of them whatever else
// occupies the GPU, and workgroups that start late find everything there.
//
// Bound by its phases one after the other.  bf16 128 MiB to 8 bits, 41 us: 4 of the two launches, the read 19.5 (6.9 TB/s), 4
// from the first published maximum to the last one seen, the arithmetic 11.5, which the stores overlap with (39.1 without
// them).  Two passes -> one, us: bf16 8 bits 64 MiB 30.9 -> 27.0, 112 MiB 52.9 -> 37.2, 128 MiB 60.3 -> 41.2, 256 MiB 116 -> 98;
// f32 8 bits 64 MiB 26.1 -> 24.6, 128 MiB 50.6 -> 37.4, 512 MiB 199 -> 181; f16 to e4m3 128 MiB 64.8 -> 50.3.
#include "cq_internal.hpp"
#include "cq_kernels_flat.hpp"
#include "cq_launch_rules.hpp"

namespace cq {
namespace {

constexpr int kThreads = 512;
constexpr uint32_t kGroups = 256;  // workgroups = slots
static_assert(kGroups <= kMaxPartials, "the slots are the caller's workspace");
constexpr uint32_t kUnset = 0xffffffffu;  // no abs-max: NaN elements are ignored
constexpr uint32_t kPatience = 64;        // polls, about a microsecond each
typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));
constexpr uint32_t kPerVector = 8;  // chunks
constexpr uint32_t kInRegisters = 48, kInLds = 16, kResident = kInRegisters + kInLds;  // chunks per lane

__global__ __launch_bounds__(kGroups) void unset_slots_kernel(uint32_t* __restrict__ slots) { slots[threadIdx.x] = kUnset; }

struct ResidentArgs {
    const void* in;
    void* out;
    uint32_t* slots;
    void* scale_out;
    uint64_t chunks;     // whole chunks that the launch quantizes
    uint64_t num_elems;  // elements of the tensor: the abs-max covers those behind the chunks too
    uint32_t rounds;     // steps of the busiest workgroup
    uint32_t streamed;   // the first of them, read twice
    int param_dtype;
    QuantParams qp;
};

typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int kAuxStream = 2, kAuxKeep = 17;  // nt; sc0 sc1 (output_store)

template <class F, int kBits, int kEnc>
struct Resident {
    static constexpr int kN = F::kPerChunk;
    static constexpr int kChunkBits = kN * kBits;
    const ResidentArgs& a;

    // `rounds` rounds of steps from round `first` on as buffers that end with the tensor: lanes past its end read zeros and
    // store nothing.  The byte offset of a lane's chunk is all that differs from step to step.
    struct Window {
        Rsrc in, out;
        __device__ __forceinline__ Window(const ResidentArgs& a, uint32_t first, uint32_t rounds) {
            const uint64_t skip = static_cast<uint64_t>(first) * kRoundChunks, left = a.chunks > skip ? a.chunks - skip : 0;
            const uint32_t most = rounds * kRoundChunks, n = left < most ? static_cast<uint32_t>(left) : most;
            in = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(a.in)) + skip * 16, 0, static_cast<int>(n * 16), 0x00027000);
            out = __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(a.out) + skip * kChunkBits / 8, 0, static_cast<int>(n * kChunkBits / 8), 0x00027000);
        }
        __device__ __forceinline__ u32x4 load(uint32_t chunk) const {
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(in, static_cast<int>(chunk * 16), 0, kAuxStream));
        }
    };
    static constexpr uint32_t kRoundChunks = kGroups * kThreads;
    __device__ __forceinline__ static uint32_t chunk_of(uint32_t group, uint32_t round) { return round * kRoundChunks + group * kThreads + threadIdx.x; }
    // the chunks of rounds [first, first + kUnroll) before `end`, under way
    template <uint32_t kUnroll>
    struct Batch {
        Window window;
        u32x4 raw[kUnroll];
        __device__ __forceinline__ Batch(const Resident& r, uint32_t group, uint32_t first, uint32_t end)
            : window(r.a, first, first < end ? (end - first < kUnroll ? end - first : kUnroll) : 0) {
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; u++) raw[u] = window.load(chunk_of(group, u));
        }
    };
    __device__ __forceinline__ static float absmax(u32x4 raw, float acc) {
        float v[kN];
        F::unpack(raw, v);
#pragma unroll
        for (int i = 0; i < kN; i++) acc = fmaxf(acc, fabsf(v[i]));
        return acc;
    }
    // rounds [0, end) of a share, and the elements behind the last chunk (share 0)
    __device__ __forceinline__ float streamed_absmax(uint32_t group, uint32_t end, float acc) const {
        constexpr uint32_t kUnroll = 8;
        Batch<kUnroll> now(*this, group, 0, end);
        for (uint32_t k0 = 0; k0 < end; k0 += kUnroll) {
            const Batch<kUnroll> next(*this, group, k0 + kUnroll, end);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; u++) acc = absmax(now.raw[u], acc);
            now = next;
        }
        return acc;
    }
    // the elements behind the last chunk: share 0 has them
    __device__ __forceinline__ float tail_absmax(uint32_t group, float acc) const {
        const uint64_t e = a.chunks * kN + threadIdx.x;
        if (group == 0 && e < a.num_elems) acc = fmaxf(acc, fabsf(F::load(a.in, e)));
        return acc;
    }
    // another workgroup's share
    __device__ __forceinline__ float share_absmax(uint32_t group) const {
        float acc = 0.0f;
#pragma unroll 1
        for (uint32_t k = 0; k < a.rounds; k++) acc = absmax(Window(a, k, 1).load(chunk_of(group, 0)), acc);
        return tail_absmax(group, acc);
    }
    // the abs-max of the workgroup's lanes, in lane 0 of the workgroup
    __device__ __forceinline__ static float group_absmax(float acc) {
        __shared__ float wave_max[kThreads / kWave];
        acc = group_max<64>(acc);
        __syncthreads();
        if (threadIdx.x % kWave == 0) wave_max[threadIdx.x / kWave] = acc;
        __syncthreads();
        return group_max<kThreads / kWave>(wave_max[threadIdx.x % (kThreads / kWave)]);
    }
    __device__ __forceinline__ void publish(uint32_t group, float amax) const {
        if (threadIdx.x == 0) __hip_atomic_store(a.slots + group, f32_bits(amax), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // the abs-max of all shares
    __device__ __forceinline__ float collect() const {
        __shared__ uint32_t missing;
        uint32_t mine = 0;
        for (uint32_t polls = 0;; polls++) {
            if (threadIdx.x < kGroups) mine = __hip_atomic_load(a.slots + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (!__syncthreads_or(mine == kUnset)) break;
            if (polls < kPatience) {
                __builtin_amdgcn_s_sleep(2);
                continue;
            }
            // the first share missing from this workgroup's place on, so that those who help start at different ones
            if (threadIdx.x == 0) missing = kGroups;
            __syncthreads();
            const uint32_t place = (threadIdx.x - blockIdx.x * 2) % kGroups;
            if (mine == kUnset) atomicMin(&missing, place);
            __syncthreads();
            const uint32_t share = (missing + blockIdx.x * 2) % kGroups;
            publish(share, group_absmax(share_absmax(share)));
            __syncthreads();
        }
        return group_absmax(threadIdx.x < kGroups ? bits_f32(mine) : 0.0f);
    }
    template <bool kTame>
    __device__ __forceinline__ void quantize(u32x4 raw, const Window& to, uint32_t chunk, float d) const {
        float v[kN];
        F::unpack(raw, v);
        uint32_t w[2];
        if constexpr (F::kDtype == CQ_F16 && kEnc == kEncInt && kTame) {
            quantize_pack_f16_tame<kBits>(v, d, a.qp.lo, a.qp.hi, w);
        } else if constexpr (F::kDtype == CQ_BF16 && kEnc == kEncInt && kTame) {
            quantize_pack_bf16_tame<kBits>(v, d, a.qp.lo, a.qp.hi, w);
        } else {
            float qn[kN];
            quantize_codes<F, kN, kEnc>(v, d, kTame, a.qp.lo, a.qp.hi, a.qp.unrounded != 0, qn);
            if constexpr (kEnc == kEncInt)
                pack_chunk_neg<kBits, kN, false>(qn, w);
            else
                encode_chunk<kEnc, kN>(qn, w);
        }
        if constexpr (kChunkBits == 64) {
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{w[0], w[1]}, to.out, static_cast<int>(chunk * 8), 0, kAuxKeep);
        } else {
            constexpr uint32_t kLanesPerWord = kChunkBits >= 32 ? 1 : 32 / kChunkBits;
            const uint32_t sub = threadIdx.x % kLanesPerWord;
            const uint32_t word = kLanesPerWord == 1 ? w[0] : group_or<kLanesPerWord>(w[0] << (sub * kChunkBits % 32));
            const int at = static_cast<int>(chunk / kLanesPerWord * 4);
            if (sub == 0) __builtin_amdgcn_raw_buffer_store_b32(word, to.out, at, 0, kAuxKeep);
        }
    }
    // rounds [0, end), read again
    __device__ __forceinline__ void quantize_streamed(uint32_t end, float d) const {
        constexpr uint32_t kUnroll = 8;
        Batch<kUnroll> now(*this, blockIdx.x, 0, end);
        for (uint32_t k0 = 0; k0 < end; k0 += kUnroll) {
            const Batch<kUnroll> next(*this, blockIdx.x, k0 + kUnroll, end);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; u++) quantize<true>(now.raw[u], now.window, chunk_of(blockIdx.x, u), d);
            now = next;
        }
    }
    __device__ __forceinline__ void run() const {
        __shared__ u32x4 lds[kInLds][kThreads];
        float amax = streamed_absmax(blockIdx.x, a.streamed, 0.0f);
        amax = tail_absmax(blockIdx.x, amax);
        const Window w(a, a.streamed, kResident);
        const uint32_t held = a.rounds - a.streamed;  // of the kResident chunks: the others read as zeros, and are skipped
        const auto load = [&](uint32_t u) { return w.load(chunk_of(blockIdx.x, u)); };
        const auto keep = [&](u32x4 raw, uint32_t u) {
            amax = absmax(raw, amax);
            lds[u][threadIdx.x] = raw;
        };
        u32x32 kept[kInRegisters / kPerVector];
        const auto hold = [&](uint32_t u, u32x4 raw) {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) kept[u / kPerVector][u % kPerVector * 4 + i] = raw[i];
        };
        const auto held_chunk = [&](uint32_t v, uint32_t u) { return u32x4{kept[v][u * 4], kept[v][u * 4 + 1], kept[v][u * 4 + 2], kept[v][u * 4 + 3]}; };
        // the chunks for LDS come first, and the last registers are loaded in their place
        {
            u32x4 raw[kInLds];
#pragma unroll
            for (uint32_t u = 0; u < kInLds; u++) raw[u] = load(kInRegisters + u);
#pragma unroll
            for (uint32_t u = 0; u < kInRegisters - kInLds; u++) hold(u, load(u));
            __builtin_amdgcn_sched_barrier(0);  // every load ahead of the arithmetic
#pragma unroll
            for (uint32_t u = 0; u < kInLds; u++) {
                keep(raw[u], u);
                hold(kInRegisters - kInLds + u, load(kInRegisters - kInLds + u));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kInRegisters; u += 4) {
            if (u < held) {
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) amax = absmax(held_chunk((u + j) / kPerVector, (u + j) % kPerVector), amax);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        publish(blockIdx.x, group_absmax(amax));
        amax = collect();
        // the scale as quantize_flat_body derives it
        const float s_f = F::round(scale_from_absmax(amax, a.qp.width));
        const bool fs_rounds = a.param_dtype != CQ_F32 && a.param_dtype != F::kDtype;
        const float s_fs = fs_rounds ? round_to_dtype(a.param_dtype, s_f) : s_f;
        if (blockIdx.x == 0 && threadIdx.x == 0) store_dtype(a.param_dtype, a.scale_out, 0, s_fs);
        const float d = fs_rounds ? F::round(s_fs) : s_f;
        if (!__builtin_amdgcn_readfirstlane(divisor_is_tame(d))) {  // divisions: all of it from memory again
#pragma unroll 1
            for (uint32_t k = 0; k < a.rounds; k++) {
                const Window again(a, k, 1);
                quantize<false>(again.load(chunk_of(blockIdx.x, 0)), again, chunk_of(blockIdx.x, 0), d);
            }
            return;
        }
        // a loop over the chunks of a vector, each picked by the vector index register: 48 copies of the code for one chunk
        // would take as long (bf16 128 MiB 41.2 and 42.4 us), in five times the bytes
#pragma unroll
        for (uint32_t v = 0; v < kInRegisters / kPerVector; v++) {
            const uint32_t first = v * kPerVector;
#pragma unroll 1
            for (uint32_t u = 0; u < kPerVector && first + u < held; u++) quantize<true>(held_chunk(v, u), w, chunk_of(blockIdx.x, first + u), d);
        }
#pragma unroll 1
        for (uint32_t u = 0; kInRegisters + u < held; u++) quantize<true>(lds[u][threadIdx.x], w, chunk_of(blockIdx.x, kInRegisters + u), d);
        quantize_streamed(a.streamed, d);
    }
};

template <class F, int kBits, int kEnc>
__global__ __launch_bounds__(kThreads, 2) void quantize_resident_kernel(ResidentArgs a) {
    const Resident<F, kBits, kEnc> r{a};
    r.run();
}

template <class F, int kBits, int kEnc>
hipError_t launch(hipStream_t s, ResidentArgs a) {
    const uint64_t steps = (a.chunks + kThreads - 1) / kThreads;
    a.rounds = static_cast<uint32_t>((steps + kGroups - 1) / kGroups);
    a.streamed = a.rounds > kResident ? a.rounds - kResident : 0;
    hipLaunchKernelGGL(unset_slots_kernel, dim3(1), dim3(kGroups), 0, s, a.slots);
    hipLaunchKernelGGL((quantize_resident_kernel<F, kBits, kEnc>), dim3(kGroups), dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

template <class F>
hipError_t launch_encoding(hipStream_t s, int bits, int encoding, const ResidentArgs& a) {
    switch (encoding) {
        case kEncInt:
            switch (bits) {
                case 2: return launch<F, 2, kEncInt>(s, a);
                case 4: return launch<F, 4, kEncInt>(s, a);
                case 8: return launch<F, 8, kEncInt>(s, a);
            }
            break;
        case kEncE4M3: return launch<F, 8, kEncE4M3>(s, a);
        case kEncE5M2: return launch<F, 8, kEncE5M2>(s, a);
        case kEncE2M1: return launch<F, 4, kEncE2M1>(s, a);
    }
    return hipErrorInvalidValue;
}

}  // namespace

bool quantize_resident(int bits, const FlatArgs& f) {
    if (!quantize_stays_resident(f.num_chunks, bits)) return false;
    int device = 0, units = 0;  // a partition of the GPU with fewer compute units would run the workgroups in turns
    return hipGetDevice(&device) == hipSuccess && hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
           units >= static_cast<int>(kGroups);
}

hipError_t launch_quantize_resident(hipStream_t s, int dtype, int bits, const FlatArgs& f, uint64_t num_elems, void* slots) {
    ResidentArgs a{};
    a.in = f.input;
    a.out = f.output;
    a.slots = static_cast<uint32_t*>(slots);
    a.scale_out = f.scale_out;
    a.chunks = f.num_chunks;
    a.num_elems = num_elems;
    a.param_dtype = f.param_dtype;
    a.qp = quant_params(f.range);
    switch (dtype) {
        case CQ_F32: return launch_encoding<F32>(s, bits, f.encoding, a);
        case CQ_BF16: return launch_encoding<BF16>(s, bits, f.encoding, a);
        case CQ_F16: return launch_encoding<F16>(s, bits, f.encoding, a);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cq
