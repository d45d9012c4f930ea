// One scale for a whole contiguous tensor, quantized in one read of it: every workgroup keeps its share of the tensor in
// registers and LDS while the abs-max of the others arrives.
//
// The two-pass quantize (absmax_partials_kernel, then quantize_flat_kernel) reads the tensor twice, from 64 MB on both times from
// memory, and is two launches, which for small tensors is all of its time.  The register files and the LDS of the 256 compute
// units hold 168 MiB.  A workgroup of 512 lanes with all 256 registers each fills one compute unit; it takes every 256th step of
// 512 chunks, loads up to 64 of them at once (48 stay in registers, 16 in LDS: 128 MiB), publishes the abs-max of what it read,
// waits for the other workgroups', and quantizes what it holds.  What a tensor has beyond that (its first steps) is read twice
// as before, in loops in front of and behind the resident part.  Up to 2 or 8 chunks per lane go through kernels of their own,
// without loops, and up to 8 steps through one workgroup.
//
// Waiting.  A slot per workgroup holds the launch's number and kStarted (in the large kernel), then the workgroup's abs-max; launches of
// several workgroups take turns at kRegions regions of slots.  Numbers differ until 2^32 such launches have gone by on a device, and each of
// them writes all slots of its region, so what a slot held before is never taken for this launch's.  A replay of a captured
// launch would bring the same number again: captured launches have their slots in the caller's workspace, where a launch before
// them leaves kUnset.
// No workgroup depends on another one running.  Where other launches have taken compute units, or the stream has few, some
// workgroups start only when others end: after kGrace polls those that wait work out such a share from memory, each another one
// (it marks the slot as started), and publish it for all, itself included if the slots go to a later launch meanwhile.  One that has
// started runs and will publish; all the same a workgroup waits for kPatience polls at most, and then works out
// whatever is missing, so that it goes on after at most 256 shares.
//
// Bound by its phases one after the other.  bf16 128 MiB to 8 bits, 38 us: 2 of the launch, the read 19.5 (6.9 TB/s), 4
// from the first published maximum to the last one seen, the arithmetic 11.5, which the stores overlap with.  Two passes -> one,
// us, calls on rotated buffers: bf16 8 bits 1 MiB 6.0 -> 4.6, 4 MiB 6.0 -> 5.2, 16 MiB 8.6 -> 7.8, 48 MiB 22.8 -> 17.8, 64 MiB 30.1 -> 22.2,
// 128 MiB 58.8 -> 38.2, 192 MiB 86.1 -> 65.5; f32 8 bits 64 MiB 22.3 -> 19.5, 128 MiB 49.8 -> 34.8; f16 to e4m3 128 MiB 60.1 -> 45.2.
#pragma once

#include <atomic>

#include "cq_internal.hpp"
#include "cq_kernels_flat.hpp"
#include "cq_launch_rules.hpp"

namespace cq {
namespace resident {

constexpr int kThreads = 512;
constexpr uint32_t kGroups = 256;  // most workgroups = slots
static_assert(kGroups <= kMaxPartials, "a captured launch's slots are the caller's workspace");
constexpr uint32_t kUnset = 0xffffffffu, kStarted = 0xfffffffeu;  // no abs-maxima: NaN elements are ignored
constexpr uint32_t kGrace = 8, kGraceOfSmall = 32, kPatience = 1024, kBySize = 0xffffu;  // polls
typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));
constexpr uint32_t kPerVector = 8;  // chunks

// Slots of launches outside a graph: regions of kGroups, taken in turn, so that up to kRegions launches at once have one
// each.  A slot holds a launch's number beside an abs-max.
constexpr uint32_t kRegions = 64;
static __device__ uint64_t g_slots[kRegions * kGroups];

__global__ __launch_bounds__(kGroups) void unset_slots_kernel(uint32_t* __restrict__ slots) { slots[threadIdx.x] = kUnset; }

struct ResidentArgs {  // the first 16 words come in registers: what is read while others wait
    const void* in;
    void* out;
    uint32_t* slots;     // of a captured launch
    void* scale_out;
    uint64_t chunks;     // whole chunks that the launch quantizes
    uint32_t tail;       // elements behind them, which the abs-max covers too
    uint32_t groups;     // workgroups, a power of two
    uint32_t rounds;     // steps of the busiest one
    uint32_t streamed;   // the first of them, read twice
    uint32_t number;     // of the launch; 0: a captured one, with slots in the workspace
    uint16_t grace, patience;
    int param_dtype;
    QuantParams qp;
};

typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int kAuxStream = 2, kAuxKeep = 17;  // nt; sc0 sc1 (output_store)

// kInRegisters, kInLds: chunks that a lane keeps
template <class F, int kBits, int kEnc, uint32_t kInRegisters, uint32_t kInLds>
struct Resident {
    static constexpr uint32_t kResident = kInRegisters + kInLds;
    static constexpr int kN = F::kPerChunk;
    static constexpr int kChunkBits = kN * kBits;
    const ResidentArgs& a;

    // `rounds` rounds of steps from round `first` on as buffers that end with the tensor: lanes past its end read zeros and
    // store nothing.  The byte offset of a lane's chunk is all that differs from step to step.
    struct Window {
        Rsrc in, out;
        __device__ __forceinline__ Window(const ResidentArgs& a, uint32_t first, uint32_t rounds) {
            const uint64_t skip = static_cast<uint64_t>(first) * (a.groups * kThreads), left = a.chunks > skip ? a.chunks - skip : 0;
            const uint32_t most = rounds * (a.groups * kThreads), n = left < most ? static_cast<uint32_t>(left) : most;
            in = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(a.in)) + skip * 16, 0, static_cast<int>(n * 16), 0x00027000);
            out = __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(a.out) + skip * kChunkBits / 8, 0, static_cast<int>(n * kChunkBits / 8), 0x00027000);
        }
        __device__ __forceinline__ u32x4 load(uint32_t chunk) const {
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(in, static_cast<int>(chunk * 16), 0, kAuxStream));
        }
    };
    __device__ __forceinline__ uint32_t chunk_of(uint32_t group, uint32_t round) const { return (round * a.groups + group) * kThreads + threadIdx.x; }
    // the chunks of rounds [first, first + kUnroll) before `end`, under way
    template <uint32_t kUnroll>
    struct Batch {
        Window window;
        u32x4 raw[kUnroll];
        __device__ __forceinline__ Batch(const Resident& r, uint32_t group, uint32_t first, uint32_t end)
            : window(r.a, first, first < end ? (end - first < kUnroll ? end - first : kUnroll) : 0) {
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; u++) raw[u] = window.load(r.chunk_of(group, u));
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
        if (group == 0 && threadIdx.x < a.tail) acc = fmaxf(acc, fabsf(F::load(a.in, a.chunks * kN + threadIdx.x)));
        return acc;
    }
    // another workgroup's share, a few loads at a time: the registers are full
    __device__ __forceinline__ float share_absmax(uint32_t group) const {
        constexpr uint32_t kUnroll = kInRegisters < 4 ? kInRegisters : 4;
        float acc = 0.0f;
#pragma unroll 1
        for (uint32_t k0 = 0; k0 < a.rounds; k0 += kUnroll) {
            const Batch<kUnroll> now(*this, group, k0, a.rounds);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t u = 0; u < kUnroll; u++) acc = absmax(now.raw[u], acc);
        }
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
    // Slots behind those of the launch's workgroups are written too, so that no slot keeps a number until the count of
    // launches comes round to it.
    __device__ __forceinline__ void publish(uint32_t group, uint32_t what) const {
        if (a.number == 0) {
            if (threadIdx.x == 0) __hip_atomic_store(a.slots + group, what, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (threadIdx.x < kGroups && threadIdx.x % a.groups == group) {
            __hip_atomic_store(region() + threadIdx.x, tagged(what), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __device__ __forceinline__ uint64_t* region() const { return g_slots + a.number % kRegions * kGroups; }
    __device__ __forceinline__ uint64_t tagged(uint32_t what) const { return static_cast<uint64_t>(a.number) << 32 | what; }
    __device__ __forceinline__ uint32_t poll(uint32_t group) const {
        if (a.number == 0) return __hip_atomic_load(a.slots + group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t slot = __hip_atomic_load(region() + group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return slot >> 32 == a.number ? static_cast<uint32_t>(slot) : kUnset;
    }
    // Marks a share that has not started; false: it has meanwhile.
    __device__ __forceinline__ bool claim(uint32_t group) const {
        if (a.number == 0) {
            uint32_t seen = kUnset;
            return __hip_atomic_compare_exchange_strong(a.slots + group, &seen, kStarted, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        uint64_t seen = __hip_atomic_load(region() + group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return seen >> 32 != a.number &&
               __hip_atomic_compare_exchange_strong(region() + group, &seen, tagged(kStarted), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // the abs-max of all shares
    __device__ __forceinline__ float collect() const {
        __shared__ uint32_t missing, claimed;
        __shared__ float found;
        uint32_t mine = threadIdx.x < a.groups ? kUnset : 0;
        for (uint32_t polls = 0;; polls++) {
            if (mine >= kStarted) mine = poll(threadIdx.x);
            if (!__syncthreads_or(mine >= kStarted)) break;
            const bool impatient = polls >= a.patience, help = impatient ? mine >= kStarted : mine == kUnset;
            if (!(impatient || (polls >= a.grace && __syncthreads_or(help)))) {
                __builtin_amdgcn_s_sleep(2);
                continue;
            }
            // the first one from this workgroup's place on, so that those who help start at different ones
            if (threadIdx.x == 0) missing = kGroups;
            __syncthreads();
            const uint32_t place = (threadIdx.x - blockIdx.x * 2) % kGroups;
            if (help) atomicMin(&missing, place);
            __syncthreads();
            const uint32_t share = (missing + blockIdx.x * 2) % kGroups;
            if (threadIdx.x == share) claimed = impatient || claim(share);
            __syncthreads();
            if (!claimed) continue;
            const float amax = group_absmax(share_absmax(share));
            publish(share, f32_bits(amax));
            // kept here as well: a launch kRegions later may have taken the slot
            if (threadIdx.x == 0) found = amax;
            __syncthreads();
            if (threadIdx.x == share) mine = f32_bits(found);
        }
        return group_absmax(bits_f32(mine));
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
    // the divisor, from the abs-max of what the workgroup read; block 0 stores the scale
    __device__ __forceinline__ float divisor(float amax) const {
        amax = group_absmax(amax);
        if (a.groups > 1) {
            publish(blockIdx.x, f32_bits(amax));
            amax = collect();
        }
        // the scale as quantize_flat_body derives it
        const float s_f = F::round(scale_from_absmax(amax, a.qp.width));
        const bool fs_rounds = a.param_dtype != CQ_F32 && a.param_dtype != F::kDtype;
        const float s_fs = fs_rounds ? round_to_dtype(a.param_dtype, s_f) : s_f;
        if (blockIdx.x == 0 && threadIdx.x == 0) store_dtype(a.param_dtype, a.scale_out, 0, s_fs);
        return fs_rounds ? F::round(s_fs) : s_f;
    }
    // divisions, for the divisors that need them: all of the share from memory again
    __device__ __forceinline__ void quantize_exact(float d) const {
#pragma unroll 1
        for (uint32_t k = 0; k < a.rounds; k++) {
            const Window again(a, k, 1);
            quantize<false>(again.load(chunk_of(blockIdx.x, 0)), again, chunk_of(blockIdx.x, 0), d);
        }
    }
    // few chunks
    __device__ __forceinline__ void run_small() const {
        const Window w(a, 0, kResident);
        u32x4 raw[kInRegisters];
#pragma unroll
        for (uint32_t u = 0; u < kInRegisters; u++) raw[u] = w.load(chunk_of(blockIdx.x, u));
        float amax = tail_absmax(blockIdx.x, 0.0f);
#pragma unroll
        for (uint32_t u = 0; u < kInRegisters; u++) amax = absmax(raw[u], amax);
        const float d = divisor(amax);
        if (!__builtin_amdgcn_readfirstlane(divisor_is_tame(d))) return quantize_exact(d);
#pragma unroll
        for (uint32_t u = 0; u < kInRegisters; u++) {
            if (u >= a.rounds) break;
            quantize<true>(raw[u], w, chunk_of(blockIdx.x, u), d);
        }
    }
    __device__ __forceinline__ void run() const {
        __shared__ u32x4 lds[kInLds][kThreads];
        float amax = 0.0f;
        if (a.streamed) {
            publish(blockIdx.x, kStarted);
            amax = streamed_absmax(blockIdx.x, a.streamed, amax);
        }
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
        // vectors that the share does not reach are not loaded; the chunks for LDS come first, and the last registers are loaded
        // in their place
        if (held > kInRegisters) {
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
        } else {
#pragma unroll
            for (uint32_t v = 0; v < kInRegisters; v += kPerVector) {
                if (v < held) {
#pragma unroll
                    for (uint32_t u = 0; u < kPerVector; u++) hold(v + u, load(v + u));
                }
            }
        }
        if (!a.streamed) publish(blockIdx.x, kStarted);  // behind the loads, so that none of them waits for it
#pragma unroll
        for (uint32_t u = 0; u < kInRegisters; u += 4) {
            if (u < held) {
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) amax = absmax(held_chunk((u + j) / kPerVector, (u + j) % kPerVector), amax);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const float d = divisor(amax);
        if (!__builtin_amdgcn_readfirstlane(divisor_is_tame(d))) return quantize_exact(d);
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
        if (a.streamed) quantize_streamed(a.streamed, d);
    }
};

constexpr uint32_t kFew = 2, kSome = 8, kMostRegisters = 48, kMostLds = 16;  // chunks per lane

template <class F, int kBits, int kEnc, uint32_t kInRegisters, uint32_t kInLds>
__global__ __launch_bounds__(kThreads, 2) void quantize_resident_kernel(ResidentArgs a) {
    const Resident<F, kBits, kEnc, kInRegisters, kInLds> r{a};
    if constexpr (kInLds == 0)
        r.run_small();
    else
        r.run();
}

// Whether `stream` is one of the last two that asked on this device.  Launches on two streams mostly take turns, but three or more at
// once each get a part of the compute units, and a workgroup here holds one while it waits: bf16 to 8 bits on 2, 3, 4
// streams, two passes and one, us a launch: 64 MiB 24.2 and 21.0, 25.2 and 37.6, 27.7 and 72; 128 MiB 53 and 38, 58 and 61, 58 and
// 77; 256 MiB 115 and 90, 118 and 142, 120 and 172; 16 MiB on four 7.3 and 13.4.
inline bool streams_are_few(int device, hipStream_t stream) {
    struct Recent {
        std::atomic<uintptr_t> streams[2]{~uintptr_t{0}, ~uintptr_t{0}};  // none yet
    };
    static Recent recent[16];
    auto& [first, second] = recent[device % 16].streams;
    const uintptr_t s = reinterpret_cast<uintptr_t>(stream);
    const uintptr_t last = first.load(std::memory_order_relaxed), one_before = second.load(std::memory_order_relaxed);
    if (s == last || s == one_before) return true;
    first.store(s, std::memory_order_relaxed);
    second.store(last, std::memory_order_relaxed);
    return one_before == ~uintptr_t{0};
}

// Whether `stream` may use a compute unit for each workgroup.  With a mask of 128 or 200 of them, two passes and one, us: 64 MiB 33 and
// 61, 28 and 61; 256 MiB 136 and 190, 128 and 187.
inline bool has_every_unit(hipStream_t stream) {
    uint32_t mask[kGroups / 32] = {};
    if (hipExtStreamGetCUMask(stream, kGroups / 32, mask) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    uint32_t units = 0;
    for (uint32_t m : mask) units += static_cast<uint32_t>(__builtin_popcount(m));
    return units == 0 || units >= kGroups;  // no bit: no mask
}

// The number of a launch of several workgroups; not 0.
inline uint32_t next_number(int device) {
    static std::atomic<uint32_t> counts[16];
    uint32_t n;
    do n = counts[device % 16].fetch_add(1, std::memory_order_relaxed) + 1;
    while (n == 0);
    return n;
}

template <class F, int kBits, int kEnc>
hipError_t launch(hipStream_t s, ResidentWay way, ResidentArgs a, uint64_t num_elems) {
    a.tail = static_cast<uint32_t>(num_elems - a.chunks * F::kPerChunk);
    const uint64_t steps = (a.chunks + kThreads - 1) / kThreads;
    a.groups = 1;
    if (steps > kSome)  // up to there a workgroup alone has nothing to wait for
        while (a.groups < kGroups && a.groups < steps) a.groups *= 2;
    a.rounds = static_cast<uint32_t>((steps + a.groups - 1) / a.groups);
    constexpr uint32_t kMost = kMostRegisters + kMostLds;
    a.streamed = a.rounds > kMost ? a.rounds - kMost : 0;
    if (a.grace == kBySize) a.grace = a.rounds > kSome ? kGrace : kGraceOfSmall;
    if (a.groups > 1) {
        if (way.captured)
            hipLaunchKernelGGL(unset_slots_kernel, dim3(1), dim3(kGroups), 0, s, a.slots);
        else
            a.number = next_number(way.device);
    }
    const auto kernel = a.rounds <= kFew    ? quantize_resident_kernel<F, kBits, kEnc, kFew, 0>
                        : a.rounds <= kSome ? quantize_resident_kernel<F, kBits, kEnc, kSome, 0>
                                            : quantize_resident_kernel<F, kBits, kEnc, kMostRegisters, kMostLds>;
    hipLaunchKernelGGL(kernel, dim3(a.groups), dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

template <class F>
hipError_t launch_encoding(hipStream_t s, ResidentWay way, int bits, int encoding, const ResidentArgs& a, uint64_t num_elems) {
    switch (encoding) {
        case kEncInt:
            switch (bits) {
                case 2: return launch<F, 2, kEncInt>(s, way, a, num_elems);
                case 4: return launch<F, 4, kEncInt>(s, way, a, num_elems);
                case 8: return launch<F, 8, kEncInt>(s, way, a, num_elems);
            }
            break;
        case kEncE4M3: return launch<F, 8, kEncE4M3>(s, way, a, num_elems);
        case kEncE5M2: return launch<F, 8, kEncE5M2>(s, way, a, num_elems);
        case kEncE2M1: return launch<F, 4, kEncE2M1>(s, way, a, num_elems);
    }
    return hipErrorInvalidValue;
}

}  // namespace resident

ResidentWay quantize_resident(hipStream_t stream, int bits, int float_bytes, const FlatArgs& f) {
    const bool numbered = quantize_stays_resident(f.num_chunks, bits, float_bytes, false);
    const bool captured = quantize_stays_resident(f.num_chunks, bits, float_bytes, true);
    if (!numbered && !captured) return {};
    int device = 0, units = 0;  // a partition of the GPU with fewer compute units would run the workgroups in turns
    if (hipGetDevice(&device) != hipSuccess || hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        units < static_cast<int>(resident::kGroups))
        return {};
    hipStreamCaptureStatus status = hipStreamCaptureStatusActive;
    if (hipStreamIsCapturing(stream, &status) == hipSuccess && status == hipStreamCaptureStatusNone) {
        const bool large = f.num_chunks > resident::kSome * resident::kThreads * resident::kGroups;
        return {numbered && resident::streams_are_few(device, stream) && !(large && !resident::has_every_unit(stream)), false, device};
    }
    (void)hipGetLastError();  // the default stream during another one's capture: an error, for the launch to report
    return {captured, true, device};  // replays may be on any stream
}

hipError_t launch_quantize_resident(hipStream_t s, ResidentWay way, int dtype, int bits, const FlatArgs& f, uint64_t num_elems, void* slots) {
    resident::ResidentArgs a{};
    a.in = f.input;
    a.out = f.output;
    a.slots = static_cast<uint32_t*>(slots);
    a.scale_out = f.scale_out;
    a.chunks = f.num_chunks;
    a.grace = resident::kBySize;
    a.patience = resident::kPatience;
    a.param_dtype = f.param_dtype;
    a.qp = quant_params(f.range);
    switch (dtype) {
        case CQ_F32: return resident::launch_encoding<F32>(s, way, bits, f.encoding, a, num_elems);
        case CQ_BF16: return resident::launch_encoding<BF16>(s, way, bits, f.encoding, a, num_elems);
        case CQ_F16: return resident::launch_encoding<F16>(s, way, bits, f.encoding, a, num_elems);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cq
