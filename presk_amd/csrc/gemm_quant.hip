// Contractions with int8 or int4 weights (B) whose scales run along the
// output's columns: sum_k x_k f32(q_k) s = s sum_k x_k q_k.
//
// The integers are read as they are stored and become 16-bit floats on their
// way to LDS (both types hold every int8 exactly), so a weight is one byte, or
// half of one, of memory traffic and the products run on the 16-bit matrix
// cores: exact in f32 for 16-bit activations, three products (the activation's
// three bf16 parts) for f32 ones.  The scale multiplies each finished sum, one
// rounding where the weights' loads f32(q) s round every term.  The path this
// replaces wrote f32 copies of both operands and of the output to memory and
// multiplied on the f32 MFMAs: 512 x 4096 x 11008 in bf16 636 -> 74 us,
// 8 x 4096 x 4096 87 -> 12.4 us, 512 x 4096 x 4096 in f32 215 -> 72 us.
#include "gemm_stage.hpp"

namespace presk {

namespace {

template <int OB, int ST, bool EDGE>
hipError_t half(const GemmArgs& g, hipStream_t stream) {
    return g.bm == 32 ? staged_launch<kOpHalf, OB, ST, 1, 1, 4, 4, 64, EDGE>(g, stream)
                      : staged_launch<kOpHalf, OB, ST, 1, 2, 8, 2, 64, EDGE>(g, stream);
}
template <int OB, bool EDGE>
hipError_t f32(const GemmArgs& g, hipStream_t stream) {
    return g.bm == 32 ? staged_launch<kOpF32, OB, kF32, 1, 1, 4, 4, 32, EDGE>(g, stream)
                      : staged_launch<kOpF32, OB, kF32, 1, 2, 8, 2, 32, EDGE>(g, stream);
}
template <int OB>
hipError_t weights(const GemmArgs& g, hipStream_t stream) {
    // (int4: a vector of eight is four bytes where it starts at an even element)
    bool whole = staged_whole(g, g.storage == kF32 ? 4 : 8, 8);
    if (OB == kOpQ4) {
        whole = whole && g.b_elem % 2 == 0 && (g.b_kcontig ? g.sb_n : g.sb_k) % 2 == 0;
        for (int d = 0; d < g.nbatch; ++d) whole = whole && g.sb_b[d] % 2 == 0;
    }
    switch (g.storage) {
        case kF32: return whole ? f32<OB, false>(g, stream) : f32<OB, true>(g, stream);
        case kBF16: return whole ? half<OB, kBF16, false>(g, stream) : half<OB, kBF16, true>(g, stream);
        case kF16: return whole ? half<OB, kF16, false>(g, stream) : half<OB, kF16, true>(g, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace

bool gemm_quant_fits(const GemmArgs& g) { return g.a_kcontig && staged_strides(g); }

hipError_t gemm_quant_launch(const GemmArgs& g, hipStream_t stream) {
    return g.b_bits == 8 ? weights<kOpQ8>(g, stream) : g.b_bits == 4 ? weights<kOpQ4>(g, stream) : hipErrorInvalidValue;
}

}  // namespace presk
