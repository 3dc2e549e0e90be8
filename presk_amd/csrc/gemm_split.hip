// f32 contractions on the bf16 matrix cores: every f32 operand element as the
// sum of three bf16 values.
//
// x = h + m + l, each the bf16 nearest what is left (8 + 8 + 8 significant
// bits, bf16 having f32's exponent range), and
//   x w = h h' + (h m' + m h') + (h l' + m m' + l h') + ...
// whose six written terms are exact products in f32; what is dropped is below
// 2^-25 of |x w|.  The largest term is summed in one f32 accumulator and the
// five small ones in another, added once at the end, so that an output takes
// K/16 roundings at its full magnitude where the f32 MFMA (16x16x4) takes K/4:
// the distance from float64 (2-norm) falls from 5.7e-7 to 1.9e-7 at 4096 x
// 1024 x 1024 and from 8.7e-7 to 3.0e-7 at K 16384.  An infinite or NaN
// operand splits into NaNs, so an output that is not finite is summed again
// by f32 MFMAs, and comes out as they give it.
//
// Six 32x32x16 bf16 MFMAs take 6/16 of the f32 MFMAs' time for the same
// products.  The operands are split once a workgroup, on the way from the
// load's registers to LDS (5.5 VALU instructions an element, one vector
// between every few MFMAs); splitting after the LDS reads would repeat it in
// every wave that shares the operand.  Each vector is loaded again as soon as
// it has been split, a whole block ahead of its use.  Rates against the f32
// MFMA tiles (operands larger than the Infinity Cache): 16384 x 384 x 1536
// 162 -> 109 us, 16384 x 1536 x 384 174 -> 122 us, 16384 x 384 x 384 48 -> 33
// us, 4096 x 1024 x 1024 68 -> 51 us, the weight gradient [384 x 1536] over K
// 16384 161 -> 109 us.  Large products run at 190-200 TFLOP/s, which is 1.2
// PFLOP/s of bf16 MFMAs at the 1.75 GHz that the chip holds under them (MFMA
// pipes 60 % busy by the counters): the power limit.  Short K is bound by
// each tile's prologue and stores.
#include <hip/hip_runtime.h>

#include "gemm.hpp"

#include <type_traits>

namespace presk {

namespace {


typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

__device__ __forceinline__ unsigned pk_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float lo_f32(unsigned w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float hi_f32(unsigned w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// One operand's k-block (ROWS x 32 f32): loaded into registers, split there
// and stored as three bf16 planes.  k-contiguous operands lie in a plane as
// [row][32 k], 16-byte chunk c of row r in slot c ^ ((r >> 2) & 3); m- or
// n-contiguous ones as [k][ROWS], chunk j of k-row r in slot j ^ swz(r) (the
// fragments then come by gfx950's transposing LDS read).  Both swizzles keep
// the fragment reads and the stores free of bank conflicts.
template <bool KC, int ROWS, int NTH, int BK, bool SAFE>
struct SplitLoader {
    static constexpr int PLANE = ROWS * BK * 2;              // bytes
    static constexpr int BYTES = 3 * PLANE;
    static constexpr int NV = ROWS * BK / 4 / NTH;           // float4s a thread
    static constexpr int VPR = KC ? BK / 4 : ROWS / 4;       // float4s a (row or k-row)
    static_assert(ROWS * BK / 4 % NTH == 0, "whole rounds");
    const char* origin;
    unsigned voff[NV];           // this thread's vectors (SAFE: their rows) from the origin, in bytes
    unsigned rstr, kstr;         // bytes between rows and between k
    int last;                    // the tile's last existing row
    long long step;              // bytes a k-block
    f32x4 r[NV];

    __device__ static __forceinline__ int swz(int k) {
        return ROWS % 128 == 0 ? (2 * (k & 3)) ^ (8 * (k & 1)) : 2 * (k & 3);
    }
    __device__ static __forceinline__ int rswz(int row) { return BK == 32 ? (row >> 2) & 3 : (row >> 3) & 1; }
    __device__ __forceinline__ static int k_of(int q) {
        const int slot = q * NTH + threadIdx.x;
        return KC ? (slot % VPR) * 4 : slot / VPR;
    }
    __device__ __forceinline__ static int row_of(int q) {
        const int slot = q * NTH + threadIdx.x;
        return KC ? slot / VPR : (slot % VPR) * 4;
    }
    // rows from row0 (row0 < rows), strides in elements.  Rows past the
    // operand read its last row (or last whole vector): the results of such
    // rows are never stored.
    __device__ __forceinline__ void init(const float* p, int rows, long long rs, long long ks, int row0, int k0) {
        origin = (const char*)(p + (long long)row0 * rs + (long long)k0 * ks);
        step = (long long)BK * ks * 4;
        rstr = 4u * (unsigned)rs;
        kstr = 4u * (unsigned)ks;
        last = rows - 1 - row0;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int row = row_of(q);
            if (SAFE) voff[q] = (unsigned)(row < last ? row : last) * rstr;
            else if (KC) voff[q] = (unsigned)(row < last ? row : last) * rstr + 4u * (unsigned)k_of(q);
            else voff[q] = (unsigned)k_of(q) * kstr + 4u * (unsigned)(row + 3 <= last ? row : last - 3);
        }
    }
    // vector q of the block at the origin, `left` of whose k exist (at least
    // one); k past them reads the row's first k instead and is zeroed by
    // store1, so that the loads need no branch.  SAFE: four elements by
    // general strides, any alignment, row and k ends anywhere.
    __device__ __forceinline__ void load1(int q, int left) {
        const int k = k_of(q);
        if constexpr (SAFE) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int ke = KC ? k + e : k, row = row_of(q);
                const unsigned ro = KC || e == 0 ? voff[q] : (unsigned)(row + e < last ? row + e : last) * rstr;
                r[q][e] = *(const float*)(origin + ro + (ke < left ? (unsigned)ke * kstr : 0u));
            }
        } else {
            const unsigned back = KC ? 4u * (unsigned)k : (unsigned)k * kstr;
            r[q] = *(const f32x4*)(origin + (left >= BK || k < left ? voff[q] : voff[q] - back));
        }
    }
    __device__ __forceinline__ void load(int left) {
#pragma unroll
        for (int q = 0; q < NV; ++q) load1(q, left);
        origin += step;
    }
    // vector q of the thread, split and stored
    __device__ __forceinline__ void store1(char* tile, int q, int left) const {
        const int slot = q * NTH + threadIdx.x;
        int off;
        if (KC) {
            const int row = slot / VPR, c = (slot % VPR) >> 1;
            off = row * BK * 2 + ((c ^ rswz(row)) << 4) + (slot & 1) * 8;
        } else {
            const int k = slot / VPR, v = slot % VPR;
            off = k * ROWS * 2 + (((v >> 1) ^ swz(k)) << 4) + (v & 1) * 8;
        }
        f32x4 x = r[q];
        if (left < BK) {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = (KC ? k_of(q) + e : k_of(q)) < left ? x[e] : 0.f;
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const unsigned a = pk_bf16(x[0], x[1]), b = pk_bf16(x[2], x[3]);
            *(u32x2*)(tile + p * PLANE + off) = u32x2{a, b};
            if (p < 2) {
                x[0] = x[0] - lo_f32(a);
                x[1] = x[1] - hi_f32(a);
                x[2] = x[2] - lo_f32(b);
                x[3] = x[3] - hi_f32(b);
            }
        }
    }
    __device__ __forceinline__ void store(char* tile, int left) const {
#pragma unroll
        for (int q = 0; q < NV; ++q) store1(tile, q, left);
    }
    // plane p's 32x32x16 fragment: lane holds k = kk + 8 (lane >> 5) .. + 8 of
    // row base + (lane & 31)
    __device__ static __forceinline__ bf16x8 frag(const char* tile, int p, int base, int kk, int lane) {
        const char* xs = tile + p * PLANE;
        if constexpr (KC) {
            const int row = base + (lane & 31), c = (kk >> 3) + (lane >> 5);
            return __builtin_bit_cast(bf16x8, *(const u32x4*)(xs + row * BK * 2 + ((c ^ rswz(row)) << 4)));
        } else {
            const int L = lane & 15, g = lane >> 4;
            const int k = kk + 8 * (g >> 1) + (L >> 2), col = base + 16 * (g & 1) + 4 * (L & 3);
            const int off = k * ROWS * 2 + (((col >> 3) ^ swz(k)) << 4) + (col & 7) * 2;
            // k-row k + 4 has k's swizzle
            const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(xs + off));
            const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(xs + off + 4 * ROWS * 2));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

__device__ __forceinline__ f32x16 mm(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// NW waves, WAN of them along the columns, each WM x WN tiles of 32 x 32.
template <bool AK, bool BKC, int WM, int WN, int NW, int WAN, int BK, bool SAFE>
__global__ void __launch_bounds__(64 * NW, 2) split_gemm_kernel(GemmArgs g) {
    constexpr int NTH = 64 * NW, WAM = NW / WAN, BM = WAM * WM * 32, BN = WAN * WN * 32;
    typedef SplitLoader<AK, BM, NTH, BK, SAFE> LA;
    typedef SplitLoader<BKC, BN, NTH, BK, SAFE> LB;
    constexpr int STAGE = LA::BYTES + LB::BYTES;
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];

    // the work order of gemm_kernel: one line of (split, batch, tile) items,
    // each XCD a contiguous run of them, GROUP row-tiles at a time
    const unsigned tiles = (unsigned)g.tiles_m * (unsigned)g.tiles_n;
    const unsigned total = gridDim.x, nb = (unsigned)g.batch;
    const unsigned xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const unsigned q8 = total / 8, r8 = total % 8;
    const unsigned item = xcd * q8 + (xcd < r8 ? xcd : r8) + local;
    const unsigned tb = item / tiles;
    const int split = (int)(tb / nb);
    const unsigned batch = tb - (unsigned)split * nb;
    const unsigned bid = item - tb * tiles;
    constexpr unsigned GROUP = BM == 256 ? 4 : 8;
    const unsigned tiles_m = (unsigned)g.tiles_m;
    const unsigned group_size = GROUP * (unsigned)g.tiles_n;
    const unsigned grp = bid / group_size;
    const unsigned first_m = grp * GROUP;
    const unsigned gm = (tiles_m - first_m) < GROUP ? (tiles_m - first_m) : GROUP;
    const unsigned in_grp = bid - grp * group_size;
    const unsigned tn_idx = in_grp / gm;
    const unsigned tm_idx = first_m + (in_grp - tn_idx * gm);
    const int m0 = (int)(tm_idx * BM), n0 = (int)(tn_idx * BN);

    long long a_off = 0, b_off = 0, c_off = 0;
    {
        unsigned rest = batch;
        for (int d = g.nbatch - 1; d >= 0; --d) {
            const unsigned dim = (unsigned)g.bdim[d], q = rest / dim, i = rest - q * dim;
            rest = q;
            a_off += (long long)i * g.sa_b[d];
            b_off += (long long)i * g.sb_b[d];
            c_off += (long long)i * g.sc_b[d];
        }
    }
    const float* A = (const float*)g.A + a_off;
    const float* B = (const float*)g.B + b_off;
    // split s of S takes the 32-deep blocks [s*nkb/S, (s+1)*nkb/S)
    const unsigned nkb = (unsigned)((g.K + 31) / 32), ns = (unsigned)g.splits;
    const int kbeg = (int)((unsigned)split * nkb / ns * 32);
    int kend = (int)(((unsigned)split + 1) * nkb / ns * 32);
    if (kend > (int)g.K) kend = (int)g.K;
    const int M = (int)g.M, N = (int)g.N;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave / WAN) * (WM * 32), wn = (wave % WAN) * (WN * 32);
    f32x16 big[WM][WN], small[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            big[i][j] = f32x16{};
            small[i][j] = f32x16{};
        }

    const int nk = (kend - kbeg + BK - 1) / BK;
    LA la;
    LB lb;
    la.init(A, M, g.sa_m, g.sa_k, m0, kbeg);
    lb.init(B, N, g.sb_n, g.sb_k, n0, kbeg);
    if (nk > 0) {
        la.load(kend - kbeg);
        lb.load(kend - kbeg);
        la.store(smem, kend - kbeg);
        lb.store(smem + LA::BYTES, kend - kbeg);
    }
    if (nk > 1) {
        la.load(kend - kbeg - BK);
        lb.load(kend - kbeg - BK);
    }
    __syncthreads();
    bf16x8 a0[WM], b0[WN];
    auto read0 = [&](const char* st, int kk) {
#pragma unroll
        for (int i = 0; i < WM; ++i) a0[i] = LA::frag(st, 0, wm + i * 32, kk, lane);
#pragma unroll
        for (int j = 0; j < WN; ++j) b0[j] = LB::frag(st + LA::BYTES, 0, wn + j * 32, kk, lane);
    };
    if (nk > 0) read0(smem, 0);
    // block kt: STORE, the next block (loaded during block kt - 1) split into
    // the other stage, one vector after every few MFMAs; LOAD, the loads of
    // the block after it, `left` of its k existing
    auto block = [&](int kt, auto store, auto load, int sleft, int lleft) {
        constexpr bool STORE = decltype(store)::value, LOAD = decltype(load)::value;
        char* const cur = smem + (kt & 1) * STAGE;
        char* const nx = smem + ((kt & 1) ^ 1) * STAGE;
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            bf16x8 a1[WM], b1[WN], a2[WM], b2[WN];
#pragma unroll
            for (int i = 0; i < WM; ++i) a1[i] = LA::frag(cur, 1, wm + i * 32, kk, lane);
#pragma unroll
            for (int j = 0; j < WN; ++j) b1[j] = LB::frag(cur + LA::BYTES, 1, wn + j * 32, kk, lane);
#pragma unroll
            for (int i = 0; i < WM; ++i) a2[i] = LA::frag(cur, 2, wm + i * 32, kk, lane);
#pragma unroll
            for (int j = 0; j < WN; ++j) b2[j] = LB::frag(cur + LA::BYTES, 2, wn + j * 32, kk, lane);
            // the vectors split beside this step's MFMAs
            constexpr int NVT = LA::NV + LB::NV, STEPS = BK / 16, SPAN = 4 * WM * WN;
            const int v0 = NVT * (kk / 16) / STEPS, v1 = NVT * (kk / 16 + 1) / STEPS;
            int done = v0, mi = 0;
            // roles exchanged (D = B^T A^T): a lane holds runs of four
            // consecutive columns of one output row
            auto mul = [&](f32x16 (&acc)[WM][WN], const bf16x8 (&bb)[WN], const bf16x8 (&aa)[WM]) {
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j) {
                        acc[i][j] = mm(bb[j], aa[i], acc[i][j]);
                        ++mi;
                        if (STORE && done < v1 && (done - v0) * SPAN <= (mi - 1) * (v1 - v0)) {
                            __builtin_amdgcn_sched_barrier(0);
                            if (done < LA::NV) {
                                la.store1(nx, done, sleft);
                                if (LOAD) la.load1(done, lleft);
                            } else {
                                lb.store1(nx + LA::BYTES, done - LA::NV, sleft);
                                if (LOAD) lb.load1(done - LA::NV, lleft);
                            }
                            ++done;
                        }
                    }
            };
            mul(big, b0, a0);
            mul(small, b0, a1);
            mul(small, b1, a0);
            mul(small, b1, a1);
            bf16x8 pa[WM], pb[WN];
#pragma unroll
            for (int i = 0; i < WM; ++i) pa[i] = a0[i];
#pragma unroll
            for (int j = 0; j < WN; ++j) pb[j] = b0[j];
            if (kk + 16 < BK) {
                read0(cur, kk + 16);
            } else if (STORE) {
                __syncthreads();
                read0(nx, 0);
            }
            mul(small, pb, a2);
            mul(small, b2, pa);
        }
        if (LOAD) {
            la.origin += la.step;
            lb.origin += lb.step;
        }
    };
    const std::integral_constant<bool, true> yes;
    const std::integral_constant<bool, false> no;
    int kt = 0;
    // (the block loaded last may be partial)
    for (; kt + 3 < nk; ++kt) block(kt, yes, yes, BK, BK);
    if (kt + 2 < nk) {
        block(kt, yes, yes, BK, kend - kbeg - (kt + 2) * BK);
        ++kt;
    }
    if (kt + 1 < nk) {
        block(kt, yes, no, kend - kbeg - (kt + 1) * BK, 0);
        ++kt;
    }
    if (kt < nk) block(kt, no, no, 0, 0);

    // the sums; an infinite or NaN one (an infinite or NaN operand, whose
    // split is NaN, or a sum past f32's range) is taken again by f32 MFMAs
    // over the same k
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            f32x16 v = big[i][j] + small[i][j];
            bool bad = false;
#pragma unroll
            for (int e = 0; e < 16; ++e) bad |= !__builtin_isfinite(v[e]);
            if (__any(bad)) {
                const int m = m0 + wm + i * 32 + (lane & 31), n = n0 + wn + j * 32 + (lane & 31);
                const float* pa = A + (long long)(m < M ? m : M - 1) * g.sa_m;
                const float* pb = B + (long long)(n < N ? n : N - 1) * g.sb_n;
                f32x16 s = {};
                for (int k = kbeg; k < kend; k += 2) {
                    const int kl = k + (lane >> 5);
                    const bool in = kl < kend;
                    const float x = in ? pa[(long long)kl * g.sa_k] : 0.f, y = in ? pb[(long long)kl * g.sb_k] : 0.f;
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(y, x, s, 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (!__builtin_isfinite(v[e])) v[e] = s[e];
            }
            big[i][j] = v;
        }

    float* const C = (float*)g.C + c_off;
    const bool cvec = g.sc_m % 4 == 0 && (uintptr_t)C % 16 == 0, wvec = N % 4 == 0;
    const bool has_bias = g.bias && g.splits <= 1;
    const float* const bias = (const float*)g.bias;
    const float bscalar = has_bias && g.bias_kind == 3 ? bias[0] : 0.f;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        const int m = m0 + wm + i * 32 + (lane & 31);
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + wn + j * 32 + 8 * q + 4 * (lane >> 5);
                if (n >= N) continue;
                const bool full = n + 4 <= N;
                f32x4 v = {big[i][j][4 * q], big[i][j][4 * q + 1], big[i][j][4 * q + 2], big[i][j][4 * q + 3]};
                if (g.splits > 1) {
                    float* w = g.work + ((long long)split * M + m) * N + n;
                    if (full && wvec) {
                        *(f32x4*)w = v;
                    } else {
                        for (int e = 0; e < 4 && n + e < N; ++e) w[e] = v[e];
                    }
                    continue;
                }
                if (has_bias)
                    for (int e = 0; e < 4 && n + e < N; ++e)
                        v[e] = v[e] + (g.bias_kind == 1 ? bias[n + e] : g.bias_kind == 2 ? bias[(long long)m * N + n + e] : bscalar);
                float* c = C + (long long)m * g.sc_m + n;
                if (full && cvec) {
                    *(f32x4*)c = v;
                } else {
                    for (int e = 0; e < 4 && n + e < N; ++e) c[e] = v[e];
                }
            }
    }
}

template <int WM, int WN, int NW, int WAN, int BK, bool SAFE>
hipError_t launch(const GemmArgs& g, hipStream_t stream) {
    const long long items = (long long)g.tiles_m * g.tiles_n * g.batch * g.splits;
    if (items <= 0) return hipSuccess;
    if (items > 0x7fffffffLL) return hipErrorInvalidValue;
    const unsigned n = (unsigned)items;
    if (g.a_kcontig && g.b_kcontig) split_gemm_kernel<true, true, WM, WN, NW, WAN, BK, SAFE><<<n, 64 * NW, 0, stream>>>(g);
    else if (g.a_kcontig) split_gemm_kernel<true, false, WM, WN, NW, WAN, BK, SAFE><<<n, 64 * NW, 0, stream>>>(g);
    else if (g.b_kcontig) split_gemm_kernel<false, true, WM, WN, NW, WAN, BK, SAFE><<<n, 64 * NW, 0, stream>>>(g);
    else split_gemm_kernel<false, false, WM, WN, NW, WAN, BK, SAFE><<<n, 64 * NW, 0, stream>>>(g);
    return hipGetLastError();
}

}  // namespace

bool gemm_split_fits(const GemmArgs& g) {
    // At most 64 rows or columns: 32 flops a byte of the long operand or
    // fewer, so the f32 MFMAs keep up with memory (384 products of 256 x 64 x
    // 256 in a training step: 502 us for the attention layer's launches
    // either way).  K below 96 (65 at 128 columns): the tile is its prologue
    // and epilogue (16384 x 65 x 72: 12.6 us on the f32 tiles, 13.8 us here).
    if (g.M <= 64 || g.N <= 64) return false;
    // 32-bit byte offsets inside a tile: 192 rows, 32 k
    const long long lim = 1ll << 22;
    return g.storage == kF32 && g.K >= (g.N >= 128 ? 65 : 96) && g.sa_m < lim && g.sa_k < lim && g.sb_k < lim && g.sb_n < lim;
}

hipError_t gemm_split_launch(const GemmArgs& g0, hipStream_t stream) {
    GemmArgs g = g0;
    const bool whole = g.a_vec && g.b_vec && (g.a_kcontig || g.sa_m == 1) && (g.b_kcontig || g.sb_n == 1);
    if (!whole && g.bn == 192) g.bn = 128;
    g.tiles_m = (int)((g.M + 127) / 128);
    g.tiles_n = (int)((g.N + g.bn - 1) / g.bn);
    if (whole) {
        if (g.bn == 192) return launch<1, 3, 8, 2, 32, false>(g, stream);
        if (g.bn == 128 && g.eight) return launch<1, 2, 8, 2, 32, false>(g, stream);
        if (g.bn == 128) return launch<2, 2, 4, 2, 16, false>(g, stream);
        if (g.bn == 64) return launch<2, 1, 4, 2, 32, false>(g, stream);
    } else {
        if (g.bn == 128) return launch<1, 2, 8, 2, 32, true>(g, stream);
        if (g.bn == 64) return launch<2, 1, 4, 2, 32, true>(g, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace presk
