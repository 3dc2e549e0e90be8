// f32 contractions on the bf16 matrix cores: every f32 operand element as the
// sum of three bf16 values.
//
// 2^16 x = h + m + l, each the bf16 nearest what is left (8 + 8 + 8 significant
// bits; exact down to f32's last subnormal thanks to the 2^16, see kSplitUp), and
//   2^32 x w = h h' + (h m' + m h') + (h l' + m m' + l h') + ...
// whose six written terms are exact products in f32; what is dropped is below
// 2^-25 of it.  The largest term is summed in one f32 accumulator and the
// five small ones in another, added once at the end, so that an output takes
// K/16 roundings at its full magnitude where the f32 MFMA (16x16x4) takes K/4:
// the distance from float64 (2-norm) falls from 5.7e-7 to 1.9e-7 at 4096 x
// 1024 x 1024 and from 8.7e-7 to 3.0e-7 at K 16384.  An infinite or NaN
// operand splits into NaNs, so an output that is not finite is summed again
// by f32 MFMAs, and comes out as they give it.  (The 2^16 costs 1.0-1.5 % of a
// product: 4096 x 1024 x 1024 50.9 -> 51.7 us.  Without it operands of 1e-35
// were off by 2.7e-6, of 1e-39 by 2.6e-2.)
//
// Six 32x32x16 bf16 MFMAs take 6/16 of the f32 MFMAs' time for the same
// products.  The operands are split once a workgroup, on the way from the
// load's registers to LDS (6.5 VALU instructions an element, one vector
// between every few MFMAs); splitting after the LDS reads would repeat it in
// every wave that shares the operand.  Each vector is loaded again as soon as
// it has been split, a whole block ahead of its use.  Against the f32 MFMA
// tiles, operands in cache: 16384 x 384 x 1536 160 -> 109 us (177 TFLOP/s), 16384
// x 1536 x 384 178 -> 129 us, the weight gradient [384 x 1536] over K 16384 166
// -> 116 us, 4096 x 1024 x 1024 68 -> 51 us; over rings of operands larger than
// the Infinity Cache 160 -> 130, 174 -> 151, 174 -> 139 us and 16384 x 384 x 384
// 48 -> 41.  The MFMA pipes are busy 55, 44 and 51 % of the cycles of the first
// three, at the 1.85-1.96 GHz that the chip holds under them (2.2 under the f32
// MFMAs); LDS reads are free of conflicts.  The rest is the splitting beside
// them, the waits between blocks, and each tile's prologue and stores, which
// weigh more the shorter K is; their shares were not told apart.
#include "gemm_stage.hpp"

namespace presk {

bool gemm_split_fits(const GemmArgs& g) {
    // At most 64 rows or columns: 32 flops a byte of the long operand or
    // fewer, so the f32 MFMAs keep up with memory (384 products of 256 x 64 x
    // 256 in a training step: 502 us for the attention layer's launches
    // either way).  K below 96 (65 at 128 columns): the tile is its prologue
    // and epilogue (16384 x 65 x 72: 12.6 us on the f32 tiles, 13.8 us here).
    if (g.M <= 64 || g.N <= 64) return false;
    return g.storage == kF32 && g.K >= (g.N >= 128 ? 65 : 96) && staged_strides(g);
}

hipError_t gemm_split_launch(const GemmArgs& g, hipStream_t stream) {
    // vectors that end inside the operand: the same products, 128 or 64 columns
    if (!staged_whole(g, 4, 4))
        return g.bn == 64 ? staged_launch<kOpF32, kOpF32, kF32, 2, 1, 4, 2, 32, true>(g, stream)
                          : staged_launch<kOpF32, kOpF32, kF32, 1, 2, 8, 2, 32, true>(g, stream);
    if (g.bn == 192) return staged_launch<kOpF32, kOpF32, kF32, 1, 3, 8, 2, 32, false>(g, stream);
    if (g.bn == 64) return staged_launch<kOpF32, kOpF32, kF32, 2, 1, 4, 2, 32, false>(g, stream);
    return g.eight ? staged_launch<kOpF32, kOpF32, kF32, 1, 2, 8, 2, 32, false>(g, stream)
                   : staged_launch<kOpF32, kOpF32, kF32, 2, 2, 4, 2, 16, false>(g, stream);
}

}  // namespace presk
