// 16-bit contractions staged through registers (gemm_stage.hpp), the same
// MFMAs over the same k-steps as the tiles loaded straight into LDS, so the
// same bits.
//
// Operands whose rows or k are no multiple of eight: the straight loads need
// whole aligned vectors, and such operands ran element by element (eight
// two-byte loads a vector).  Here only a vector that crosses the operand's
// end is; the others are 16-byte loads at whatever byte they start.  1999 x
// 1021 x 777: 49 -> 14.3 us.
//
// At most 32 rows (a few tokens against a weight matrix): the weight's bytes
// bound it, read once, so 32-row tiles of 128 columns and a k-split that puts
// two workgroups on every CU; the 128-row tiles with their long splits left
// most CUs idle.  8 x 4096 x 4096: 15.0 -> 12.0 us.
#include "gemm_stage.hpp"

namespace presk {

namespace {

template <int ST>
hipError_t ragged(const GemmArgs& g, hipStream_t stream) {
    if (g.bm == 32)
        return staged_whole(g, 8, 8) ? staged_launch<kOpHalf, kOpHalf, ST, 1, 1, 4, 4, 64, false>(g, stream)
                                     : staged_launch<kOpHalf, kOpHalf, ST, 1, 1, 4, 4, 64, true>(g, stream);
    return g.bn == 64 ? staged_launch<kOpHalf, kOpHalf, ST, 1, 1, 8, 2, 64, true>(g, stream)
                      : staged_launch<kOpHalf, kOpHalf, ST, 1, 2, 8, 2, 64, true>(g, stream);
}

}  // namespace

bool gemm_ragged_fits(const GemmArgs& g) { return g.storage != kF32 && staged_strides(g); }

hipError_t gemm_ragged_launch(const GemmArgs& g, hipStream_t stream) {
    if (g.storage == kBF16) return ragged<kBF16>(g, stream);
    if (g.storage == kF16) return ragged<kF16>(g, stream);
    return hipErrorInvalidValue;
}

}  // namespace presk
