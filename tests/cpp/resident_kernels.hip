// The one-read quantize (cubek_amd/csrc/cq_kernels_resident.hpp) with the waits that a test asks for: with none, workgroups work out one
// another's shares in every launch.  A library of its own, driven by pytest.
#include "../../cubek_amd/csrc/cq_kernels_resident.hpp"

using namespace cq;

// kind: 0 8 bits of bf16, 1 4 bits of f32, 2 f16 to e4m3.  slots: nullptr for a numbered launch.  Returns a hipError_t.
extern "C" int cq_test_resident(int kind, void* stream, const void* in, void* out, void* scale, void* slots, uint64_t chunks, uint64_t num_elems,
                                uint32_t grace, uint32_t patience) {
    resident::ResidentArgs a{};
    a.in = in;
    a.out = out;
    a.slots = static_cast<uint32_t*>(slots);
    a.scale_out = scale;
    a.chunks = chunks;
    a.param_dtype = CQ_F32;
    a.grace = static_cast<uint16_t>(grace);
    a.patience = static_cast<uint16_t>(patience);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const ResidentWay way{true, slots != nullptr, 0};
    Range range{};
    switch (kind) {
        case 0: range.lo = -127.0f, range.hi = 127.0f; break;
        case 1: range.lo = -7.0f, range.hi = 7.0f; break;
        case 2: range.lo = -448.0f, range.hi = 448.0f; break;
        default: return hipErrorInvalidValue;
    }
    a.qp = quant_params(range);
    switch (kind) {
        case 0: return resident::launch<BF16, 8, kEncInt>(s, way, a, num_elems);
        case 1: return resident::launch<F32, 4, kEncInt>(s, way, a, num_elems);
        default: return resident::launch<F16, 8, kEncE4M3>(s, way, a, num_elems);
    }
}
