// Contractions whose operands are staged through registers on their way to
// LDS, because something is done to them there: an f32 element split into
// three bf16 parts (gemm_split.hip), an integer weight made the 16-bit float
// it is (gemm_quant.hip), or vectors that start and end anywhere
// (gemm_ragged.hip).
//
// 32x32x16 MFMAs, two LDS stages.  A block's vectors are loaded a whole block
// before they are converted and stored, each loaded again as soon as it has
// been stored, so a load has a block's time to land.  Vectors are read at any
// alignment (gfx950's global loads take any byte address); where EDGE, one
// that runs past its row's end reads what follows there, which no result uses
// (k past the end is zeroed on the way to LDS), and only one that runs past
// the operand's last element is read element by element (read so at every
// row's end, those loads' waits left nothing in flight: 1999 x 1021 x 777 in
// f16 22.3 us against 16.5; the f32 gradient [384 x 65] over K 16384 27.2
// against 23.7).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_store.hpp"

namespace presk {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

// What an operand's elements are: f32 (three bf16 planes), the storage's own
// 16-bit floats, int8 or int4 weights (one plane of the 16-bit type)
enum Operand { kOpF32, kOpHalf, kOpQ8, kOpQ4 };

__device__ __forceinline__ unsigned pk_bf16(float a, float b) {
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
// An f32 element is split times 2^16 (exact): bf16 has f32's exponents but not
// its subnormals' steps (2^-133 against 2^-149), so the parts of an element
// below 2^-110 would be cut, and one below 2^-134 lost.  Times 2^16 every f32,
// subnormal ones too, is the sum of its three parts.  Sums leave times 2^-16
// an operand.  What this pushes past f32's range instead -- an element from
// 2^112, a sum from 2^96 -- is not finite and is summed again by the f32 MFMAs
// as any such sum is.
constexpr float kSplitUp = 65536.f, kSplitDown = 1.f / 65536.f;

template <int ST>
__device__ __forceinline__ unsigned pk_half(float a, float b) {
    if (ST != kF16) return pk_bf16(a, b);
    const f32x2 v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, f16x2));
}
__device__ __forceinline__ float lo_f32(unsigned w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float hi_f32(unsigned w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// element e as f32 (an integer weight without its scale)
template <int OP, int ST>
__device__ __forceinline__ float element(const void* p, long long e) {
    if (OP == kOpF32) return ((const float*)p)[e];
    if (OP == kOpQ8) return (float)((const signed char*)p)[e];
    if (OP == kOpQ4) return (float)pk_nibble((const unsigned char*)p, e);
    return ST == kF16 ? pk_f16_to_f32(((const unsigned short*)p)[e]) : pk_bf16_to_f32(((const unsigned short*)p)[e]);
}

// One operand's k-block (ROWS x BK): loaded into registers in vectors of V
// elements along its contiguous axis, converted there and stored as planes of
// 16-bit floats.  k-contiguous operands lie in a plane as [row][BK], 16-byte
// chunk c of row r in slot c ^ rswz(r); m- or n-contiguous ones as [k][ROWS],
// chunk j of k-row r in slot j ^ swz(r) (the fragments then come by gfx950's
// transposing LDS read).  Both swizzles keep the fragment reads and the
// stores free of bank conflicts (from 64 rows).
template <int OP, int ST, bool KC, int ROWS, int NTH, int BK, bool EDGE>
struct StageLoader {
    static constexpr int PLANES = OP == kOpF32 ? 3 : 1;
    static constexpr int PLANE = ROWS * BK * 2;              // bytes
    static constexpr int BYTES = PLANES * PLANE;
    static constexpr int V = OP == kOpF32 ? 4 : 8;           // elements a vector
    static constexpr int NV = ROWS * BK / V / NTH;           // vectors a thread
    static constexpr int VPR = KC ? BK / V : ROWS / V;       // vectors a (row or k-row)
    static_assert(ROWS * BK / V % NTH == 0, "whole rounds");
    // int4 that may start in the middle of a byte: its first four bytes, and the
    // one after them (a branch for those that do made every vector wait where
    // it was loaded: 554 x 602 x 1792 with int4 weights in bf16 72.5 us, now 24.0)
    static constexpr bool HALVES = OP == kOpQ4 && EDGE;
    typedef typename std::conditional<OP == kOpQ4 && !EDGE, unsigned,
                                      typename std::conditional<OP == kOpQ8 || HALVES, u32x2, u32x4>::type>::type Raw;
    const char* base;
    long long origin;            // the block's first element (uniform)
    unsigned voff[NV];           // this thread's vectors from it, in elements
    unsigned rstr, kstr;         // elements between rows and between k
    int last;                    // the tile's last existing row
    long long step;              // elements a k-block
    long long end;               // one past the operand's last element (EDGE)
    unsigned odd;                // bit q: vector q starts in the middle of a byte (HALVES; a block is whole bytes)
    Raw r[NV];

    __device__ static __forceinline__ int swz(int k) {
        return ROWS % 128 == 0 ? (2 * (k & 3)) ^ (8 * (k & 1)) : ROWS >= 64 ? 2 * (k & 3) : 0;
    }
    __device__ static __forceinline__ int rswz(int row) {
        return BK == 64 ? (row ^ (row >> 3)) & 7 : BK == 32 ? (row >> 2) & 3 : (row >> 3) & 1;
    }
    __device__ __forceinline__ static int k_of(int q) {
        const int slot = q * NTH + threadIdx.x;
        return KC ? (slot % VPR) * V : slot / VPR;
    }
    __device__ __forceinline__ static int row_of(int q) {
        const int slot = q * NTH + threadIdx.x;
        return KC ? slot / VPR : (slot % VPR) * V;
    }
    // element `off` from the operand's first, rows from row0 (row0 < rows),
    // strides in elements, K of the whole operand.  Rows past it read its last
    // row (or last whole vector): the results of such rows are never stored.
    __device__ __forceinline__ void init(const void* p, long long off, int rows, long long rs, long long ks, int row0, int k0,
                                         long long K) {
        base = (const char*)p;
        origin = off + (long long)row0 * rs + (long long)k0 * ks;
        step = (long long)BK * ks;
        rstr = (unsigned)rs;
        kstr = (unsigned)ks;
        last = rows - 1 - row0;
        end = off + (long long)(rows - 1) * rs + (K - 1) * ks + 1;
        odd = 0;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int row = row_of(q);
            if (KC) voff[q] = (unsigned)(row < last ? row : last) * rstr + (unsigned)k_of(q);
            else voff[q] = (unsigned)k_of(q) * kstr + (unsigned)(EDGE ? (row < last ? row : last) : row + V - 1 <= last ? row : last - (V - 1));
            if (HALVES) odd |= (((unsigned)origin + voff[q]) & 1) << q;
        }
    }
    __device__ __forceinline__ Raw vec(unsigned off) const {
        Raw x;
        if constexpr (OP == kOpQ4) {
            const unsigned at = (unsigned)(origin & 1) + off;
            const char* const p = base + (origin >> 1) + (at >> 1);
            unsigned first;
            __builtin_memcpy(&first, p, 4);
            if constexpr (HALVES) x = Raw{first, (unsigned)*(const unsigned char*)(p + 3 + (at & 1))};
            else x = first;
        } else __builtin_memcpy(&x, base + origin * (OP == kOpF32 ? 4 : OP == kOpQ8 ? 1 : 2) + off * (OP == kOpF32 ? 4u : OP == kOpQ8 ? 1u : 2u), sizeof x);
        return x;
    }
    // one element's bits, in its place in a vector
    __device__ __forceinline__ void put(Raw& x, int e, long long at) const {
        if constexpr (OP == kOpF32) x[e] = ((const unsigned*)base)[at];
        else if constexpr (OP == kOpHalf) x[e >> 1] |= (unsigned)((const unsigned short*)base)[at] << (16 * (e & 1));
        else if constexpr (OP == kOpQ8) x[e >> 2] |= (unsigned)((const unsigned char*)base)[at] << (8 * (e & 3));
        else if constexpr (HALVES) {
            // (where vec reads it: an odd vector from the second nibble)
            const unsigned n = (unsigned)pk_nibble((const unsigned char*)base, at) & 15u, d = e + ((unsigned)(at - e) & 1);
            x[d >> 3] |= n << (4 * (d & 7));
        }
    }
    // vector q's eight int4
    __device__ __forceinline__ unsigned nibbles(int q) const {
        if constexpr (HALVES) return odd >> q & 1 ? r[q][0] >> 4 | r[q][1] << 28 : r[q][0];
        else return r[q];
    }
    // vector q of the block at the origin, `left` of whose k exist (at least
    // one); k past them reads the row's first k instead and is zeroed by
    // store1, so that the loads need no branch (EDGE: but for a vector past
    // the operand's last element; SURE: a whole block, and no vector of it is
    // past the operand)
    template <bool SURE = false>
    __device__ __forceinline__ void load1(int q, int left) {
        const int k = k_of(q);
        const unsigned back = KC ? (unsigned)k : (unsigned)k * kstr;
        const unsigned off = left >= BK || k < left ? voff[q] : voff[q] - back;
        if constexpr (EDGE) {
            const long long at = origin + off;
            if (SURE || (KC && left >= BK) || at + V <= end) {
                r[q] = vec(off);
            } else {
                Raw x = {};
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (at + e < end) put(x, e, at + e);
                r[q] = x;
            }
        } else {
            r[q] = vec(off);
        }
    }
    __device__ __forceinline__ void load(int left) {
#pragma unroll
        for (int q = 0; q < NV; ++q) load1(q, left);
        origin += step;
    }
    // vector q of the thread, converted and stored
    __device__ __forceinline__ void store1(char* tile, int q, int left) const {
        const int slot = q * NTH + threadIdx.x;
        int off;
        if (KC) {
            const int row = slot / VPR, c = (slot % VPR) * V / 8;
            off = row * BK * 2 + ((c ^ rswz(row)) << 4);
        } else {
            const int k = slot / VPR, c = (slot % VPR) * V / 8;
            off = k * ROWS * 2 + ((c ^ swz(k)) << 4);
        }
        const bool none = left < BK && k_of(q) >= left;    // a whole vector of k past the end
        // the elements of the vector whose k exists
        const int some = EDGE && KC && left < BK ? left - k_of(q) : V;
        if constexpr (OP == kOpF32) {
            f32x4 x = __builtin_bit_cast(f32x4, r[q]);
#pragma unroll
            for (int e = 0; e < V; ++e) x[e] = none ? 0.f : x[e] * kSplitUp;
            if (EDGE && KC && left < BK) {
#pragma unroll
                for (int e = 1; e < V; ++e) x[e] = e < some ? x[e] : 0.f;
            }
            off += (slot & 1) * 8;
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
        } else if constexpr (OP == kOpHalf) {
            u32x4 w = none ? u32x4{} : r[q];
            if (EDGE && KC && left < BK) {
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] &= some >= 2 * i + 2 ? ~0u : some == 2 * i + 1 ? 0xffffu : 0u;
            }
            *(u32x4*)(tile + off) = w;
        } else {
            typedef typename std::conditional<OP == kOpQ8, u32x2, unsigned>::type Word;
            Word w;
            if constexpr (OP == kOpQ8) w = none ? Word{} : r[q];
            else w = none ? 0u : nibbles(q);
            if constexpr (EDGE && KC) {
                if (left < BK && some < V) {
                    const int bits = (some > 0 ? some : 0) * (OP == kOpQ8 ? 8 : 4);
                    if constexpr (OP == kOpQ8) {
                        w[0] &= bits >= 32 ? ~0u : (1u << bits) - 1;
                        w[1] &= bits >= 64 ? ~0u : bits > 32 ? (1u << (bits - 32)) - 1 : 0u;
                    } else {
                        w &= (1u << bits) - 1;
                    }
                }
            }
            u32x4 h;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = 2 * i;
                if constexpr (OP == kOpQ8)
                    h[i] = pk_half<ST>((float)((int)(w[e >> 2] << (24 - 8 * (e & 3))) >> 24),
                                       (float)((int)(w[e >> 2] << (16 - 8 * (e & 3))) >> 24));
                else
                    h[i] = pk_half<ST>((float)((int)(w << (28 - 4 * e)) >> 28), (float)((int)(w << (24 - 4 * e)) >> 28));
            }
            *(u32x4*)(tile + off) = h;
        }
    }
    __device__ __forceinline__ void store(char* tile, int left) const {
#pragma unroll
        for (int q = 0; q < NV; ++q) store1(tile, q, left);
    }
    // plane p's 32x32x16 fragment: lane holds k = kk + 8 (lane >> 5) .. + 8 of
    // row base + (lane & 31)
    __device__ static __forceinline__ u32x4 frag(const char* tile, int p, int base, int kk, int lane) {
        const char* xs = tile + p * PLANE;
        if constexpr (KC) {
            const int row = base + (lane & 31), c = (kk >> 3) + (lane >> 5);
            return *(const u32x4*)(xs + row * BK * 2 + ((c ^ rswz(row)) << 4));
        } else {
            const int L = lane & 15, g = lane >> 4;
            const int k = kk + 8 * (g >> 1) + (L >> 2), col = base + 16 * (g & 1) + 4 * (L & 3);
            const int off = k * ROWS * 2 + (((col >> 3) ^ swz(k)) << 4) + (col & 7) * 2;
            // k-row k + 4 has k's swizzle
            const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(xs + off));
            const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(xs + off + 4 * ROWS * 2));
            return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

template <int ST>
__device__ __forceinline__ f32x16 mm(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (ST == kF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// NW waves, WAN of them along the columns, each WM x WN tiles of 32 x 32;
// ST the storage of the output (and of 16-bit operands).
template <int OA, int OB, int ST, bool AK, bool BKC, int WM, int WN, int NW, int WAN, int BK, bool EDGE>
__global__ void __launch_bounds__(64 * NW, 2) staged_gemm_kernel(GemmArgs g) {
    constexpr int NTH = 64 * NW, WAM = NW / WAN, BM = WAM * WM * 32, BN = WAN * WN * 32;
    typedef StageLoader<OA, ST, AK, BM, NTH, BK, EDGE> LA;
    typedef StageLoader<OB, ST, BKC, BN, NTH, BK, EDGE> LB;
    constexpr int PA = LA::PLANES, PB = LB::PLANES;
    constexpr bool QUANT = OB == kOpQ8 || OB == kOpQ4;
    constexpr int STAGE = LA::BYTES + LB::BYTES;
    // a k-split's ranges are whole blocks of UNIT, whatever the tile
    constexpr int UNIT = OA == kOpF32 ? 32 : 64;
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];

    // the work order of gemm_kernel: one line of (split, batch, tile) items,
    // each XCD a contiguous run of them, 8 row-tiles at a time
    const unsigned tiles = (unsigned)g.tiles_m * (unsigned)g.tiles_n;
    const unsigned total = gridDim.x, nb = (unsigned)g.batch;
    const unsigned xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const unsigned q8 = total / 8, r8 = total % 8;
    const unsigned item = xcd * q8 + (xcd < r8 ? xcd : r8) + local;
    const unsigned tb = item / tiles;
    const int split = (int)(tb / nb);
    const unsigned batch = tb - (unsigned)split * nb;
    const unsigned bid = item - tb * tiles;
    constexpr unsigned GROUP = 8;
    const unsigned tiles_m = (unsigned)g.tiles_m;
    const unsigned group_size = GROUP * (unsigned)g.tiles_n;
    const unsigned grp = bid / group_size;
    const unsigned first_m = grp * GROUP;
    const unsigned gm = (tiles_m - first_m) < GROUP ? (tiles_m - first_m) : GROUP;
    const unsigned in_grp = bid - grp * group_size;
    const unsigned tn_idx = in_grp / gm;
    const unsigned tm_idx = first_m + (in_grp - tn_idx * gm);
    const int m0 = (int)(tm_idx * BM), n0 = (int)(tn_idx * BN);

    long long a_off = 0, b_off = 0, c_off = 0, s_off = 0;
    {
        unsigned rest = batch;
        for (int d = g.nbatch - 1; d >= 0; --d) {
            const unsigned dim = (unsigned)g.bdim[d], q = rest / dim, i = rest - q * dim;
            rest = q;
            a_off += (long long)i * g.sa_b[d];
            b_off += (long long)i * g.sb_b[d];
            c_off += (long long)i * g.sc_b[d];
            if (QUANT) s_off += (long long)i * g.ss_b[d];
        }
    }
    // split s of S takes the blocks [s*nkb/S, (s+1)*nkb/S)
    const unsigned nkb = (unsigned)((g.K + UNIT - 1) / UNIT), ns = (unsigned)g.splits;
    const int kbeg = (int)((unsigned)split * nkb / ns * UNIT);
    int kend = (int)(((unsigned)split + 1) * nkb / ns * UNIT);
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
    la.init(g.A, a_off, M, g.sa_m, g.sa_k, m0, kbeg, g.K);
    lb.init(g.B, b_off + (QUANT ? g.b_elem : 0), N, g.sb_n, g.sb_k, n0, kbeg, g.K);
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
    u32x4 a0[WM], b0[WN];
    auto read0 = [&](const char* st, int kk) {
#pragma unroll
        for (int i = 0; i < WM; ++i) a0[i] = LA::frag(st, 0, wm + i * 32, kk, lane);
#pragma unroll
        for (int j = 0; j < WN; ++j) b0[j] = LB::frag(st + LA::BYTES, 0, wn + j * 32, kk, lane);
    };
    if (nk > 0) read0(smem, 0);
    // block kt: STORE, the next block (loaded during block kt - 1) converted
    // into the other stage, one vector after every few MFMAs; LOAD, the loads
    // of the block after it, `lleft` of its k existing
    auto block = [&](int kt, auto store, auto load, int sleft, int lleft) {
        constexpr bool STORE = decltype(store)::value, LOAD = decltype(load)::value > 0, SURE = decltype(load)::value > 1;
        char* const cur = smem + (kt & 1) * STAGE;
        char* const nx = smem + ((kt & 1) ^ 1) * STAGE;
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            u32x4 a1[WM], b1[WN], a2[WM], b2[WN];
            if constexpr (PA == 3) {
#pragma unroll
                for (int i = 0; i < WM; ++i) a1[i] = LA::frag(cur, 1, wm + i * 32, kk, lane);
            }
            if constexpr (PB == 3) {
#pragma unroll
                for (int j = 0; j < WN; ++j) b1[j] = LB::frag(cur + LA::BYTES, 1, wn + j * 32, kk, lane);
            }
            if constexpr (PA == 3) {
#pragma unroll
                for (int i = 0; i < WM; ++i) a2[i] = LA::frag(cur, 2, wm + i * 32, kk, lane);
            }
            if constexpr (PB == 3) {
#pragma unroll
                for (int j = 0; j < WN; ++j) b2[j] = LB::frag(cur + LA::BYTES, 2, wn + j * 32, kk, lane);
            }
            // the vectors converted beside this step's MFMAs: all of them
            // before the products that follow the block's barrier
            constexpr int NVT = LA::NV + LB::NV, STEPS = BK / 16, SPAN = (PA == 3 ? PB == 3 ? 4 : 2 : 0) * WM * WN;
            const int v0 = NVT * (kk / 16) / STEPS, v1 = NVT * (kk / 16 + 1) / STEPS;
            int done = v0, mi = 0;
            auto vector = [&]() {
                __builtin_amdgcn_sched_barrier(0);
                if (done < LA::NV) {
                    la.store1(nx, done, sleft);
                    if (LOAD) la.template load1<SURE>(done, lleft);
                } else {
                    lb.store1(nx + LA::BYTES, done - LA::NV, sleft);
                    if (LOAD) lb.template load1<SURE>(done - LA::NV, lleft);
                }
                ++done;
            };
            // roles exchanged (D = B^T A^T): a lane holds runs of four
            // consecutive columns of one output row
            auto mul = [&](f32x16 (&acc)[WM][WN], const u32x4 (&bb)[WN], const u32x4 (&aa)[WM]) {
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j) {
                        acc[i][j] = mm<ST>(bb[j], aa[i], acc[i][j]);
                        ++mi;
                        if (STORE && SPAN > 0 && done < v1 && (done - v0) * SPAN <= (mi - 1) * (v1 - v0)) vector();
                    }
            };
            if constexpr (PA == 3) {
                mul(big, b0, a0);
                mul(small, b0, a1);
                if constexpr (PB == 3) {
                    mul(small, b1, a0);
                    mul(small, b1, a1);
                }
            }
#pragma unroll
            for (int left = 0; left < NVT; ++left)
                if (STORE && done < v1) vector();
            u32x4 pa[WM], pb[WN];
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
            if constexpr (PA == 3) {
                mul(small, pb, a2);
                if constexpr (PB == 3) mul(small, b2, pa);
            } else {
                mul(big, pb, pa);
            }
        }
        if (LOAD) {
            la.origin += la.step;
            lb.origin += lb.step;
        }
    };
    const std::integral_constant<int, 0> no;
    const std::integral_constant<int, 1> yes;
    const std::integral_constant<int, 2> sure;
    int kt = 0;
    // All blocks but the last are whole, and a vector that runs past its row
    // there ends inside the next k's, unless those lie closer than a vector:
    // then, and for the last, the loads are checked.
    const bool close = EDGE && ((!AK && la.kstr < LA::V) || (!BKC && lb.kstr < LB::V));
    if (!close)
        for (; kt + 3 < nk; ++kt) block(kt, yes, sure, BK, BK);
    if constexpr (EDGE) {
        for (; kt + 2 < nk; ++kt) block(kt, yes, yes, BK, kend - kbeg - (kt + 2) * BK);
    } else if (kt + 2 < nk) {
        block(kt, yes, yes, BK, kend - kbeg - (kt + 2) * BK);
        ++kt;
    }
    if (kt + 1 < nk) {
        block(kt, yes, no, kend - kbeg - (kt + 1) * BK, 0);
        ++kt;
    }
    if (kt < nk) block(kt, no, no, 0, 0);

    // The sums: split operands' back at their scale, an integer weight's
    // times its scale (before, so that only the result can be subnormal).
    // Where operands were split or unscaled, an infinite or NaN sum (an
    // infinite or NaN operand, whose split is NaN, or a sum past f32's range
    // here) is taken again by f32 MFMAs over the same k of the elements
    // themselves.
    if constexpr (PA == 3 || QUANT) {
        const float* const scales = QUANT ? g.scales + s_off : nullptr;
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                f32x16 v = PA == 3 ? big[i][j] + small[i][j] : big[i][j];
                if constexpr (QUANT) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int n = n0 + wn + j * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                        v[e] = v[e] * scales[(n < N ? n : N - 1) * g.ss_n];
                    }
                }
                if constexpr (PA == 3) {
                    constexpr float down = PB == 3 ? kSplitDown * kSplitDown : kSplitDown;
#pragma unroll
                    for (int e = 0; e < 16; ++e) v[e] = v[e] * down;
                }
                bool bad = false;
#pragma unroll
                for (int e = 0; e < 16; ++e) bad |= !__builtin_isfinite(v[e]);
                if (__any(bad)) {
                    int m = m0 + wm + i * 32 + (lane & 31), n = n0 + wn + j * 32 + (lane & 31);
                    m = m < M ? m : M - 1;
                    n = n < N ? n : N - 1;
                    const long long ea = a_off + (long long)m * g.sa_m, eb = b_off + (QUANT ? g.b_elem : 0) + (long long)n * g.sb_n;
                    const float sc = QUANT ? scales[n * g.ss_n] : 1.f;
                    f32x16 s = {};
                    for (int k = kbeg; k < kend; k += 2) {
                        const int kl = k + (lane >> 5);
                        const bool in = kl < kend;
                        const float x = in ? element<OA, ST>(g.A, ea + (long long)kl * g.sa_k) : 0.f;
                        float y = in ? element<OB, ST>(g.B, eb + (long long)kl * g.sb_k) : 0.f;
                        if (QUANT && in) y = y * sc;
                        s = __builtin_amdgcn_mfma_f32_32x32x2f32(y, x, s, 0, 0, 0);
                    }
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        if (!__builtin_isfinite(v[e])) v[e] = s[e];
                }
                big[i][j] = v;
            }
    }

    typedef typename std::conditional<ST == kF32, float, unsigned short>::type S;
    S* const C = (S*)g.C + c_off;
    bool ovf = false;
    float bcol[WN][16];          // a bias by columns, the lane's
    // the lane's outputs in runs of four columns: to the split's partials, or
    // stored with the bias (BIAS: there is one)
    auto store = [&](auto partial, auto biased) {
        constexpr bool PARTIAL = decltype(partial)::value, BIAS = decltype(biased)::value;
        typedef typename std::conditional<PARTIAL, float, S>::type T;
        typedef T T4 __attribute__((ext_vector_type(4)));
        const float bscalar = BIAS && g.bias_kind == 3 ? load_bias<ST>(g.bias, 0) : 0.f;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const int m = m0 + wm + i * 32 + (lane & 31);
            if (m >= M) continue;
            T* const row = PARTIAL ? (T*)g.work + ((long long)split * M + m) * N : (T*)C + (long long)m * g.sc_m;
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int n = n0 + wn + j * 32 + 8 * q + 4 * (lane >> 5);
                    if (n >= N) continue;
                    T4 out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = big[i][j][4 * q + e];
                        if constexpr (PARTIAL) {
                            out[e] = v;
                        } else {
                            float b = bscalar;
                            if (BIAS && g.bias_kind == 1) b = bcol[j][4 * q + e];
                            if (BIAS && g.bias_kind == 2 && n + e < N) b = load_bias<ST>(g.bias, (long long)m * N + n + e);
                            bool o = false;
                            out[e] = round_out<ST>(v, BIAS, b, o);
                            ovf |= o && n + e < N;
                        }
                    }
                    if (n + 4 <= N) {
                        __builtin_memcpy(row + n, &out, sizeof out);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (n + e < N) row[n + e] = out[e];
                    }
                }
        }
    };
    const std::integral_constant<bool, true> with;
    const std::integral_constant<bool, false> without;
    if (g.splits > 1) {
        store(with, without);
    } else if (!g.bias) {
        store(without, without);
    } else {
        // every load of a bias by columns in flight at once (beside the stores
        // each run's was waited for, a third of a short call: 5056 x 128 x 41 in
        // bf16 11.1 us, now 7.2)
        if (g.bias_kind == 1) {
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // four that end inside the bias, moved to where they belong
                    const int n = n0 + wn + j * 32 + 8 * q + 4 * (lane >> 5), first = n + 4 <= N || N < 4 ? n : N - 4, past = n - first;
                    float x[4];
                    if (N >= 4) {
                        typedef S S4 __attribute__((ext_vector_type(4)));
                        S4 b;
                        __builtin_memcpy(&b, (const S*)g.bias + first, sizeof b);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const S one = b[e];
                            x[e] = load_bias<ST>(&one, 0);
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[e] = load_bias<ST>(g.bias, e < N ? e : N - 1);
                    }
                    bcol[j][4 * q] = past == 1 ? x[1] : past == 2 ? x[2] : past == 3 ? x[3] : x[0];
                    bcol[j][4 * q + 1] = past == 1 ? x[2] : past == 2 ? x[3] : x[1];
                    bcol[j][4 * q + 2] = past == 1 ? x[3] : x[2];
                    bcol[j][4 * q + 3] = x[3];
                }
        }
        store(without, with);
    }
    if (ST == kF16 && ovf && g.flag) atomicOr(g.flag, 1u);
}

template <int OA, int OB, int ST, int WM, int WN, int NW, int WAN, int BK, bool EDGE>
hipError_t staged_launch(const GemmArgs& g0, hipStream_t stream) {
    constexpr int BM = NW / WAN * WM * 32, BN = WAN * WN * 32;
    GemmArgs g = g0;
    g.tiles_m = (int)((g.M + BM - 1) / BM);
    g.tiles_n = (int)((g.N + BN - 1) / BN);
    const long long items = (long long)g.tiles_m * g.tiles_n * g.batch * g.splits;
    if (items <= 0) return hipSuccess;
    if (items > 0x7fffffffLL) return hipErrorInvalidValue;
    const unsigned n = (unsigned)items;
#define PRESK_STAGED(a, b) staged_gemm_kernel<OA, OB, ST, a, b, WM, WN, NW, WAN, BK, EDGE><<<n, 64 * NW, 0, stream>>>(g)
    if (g.a_kcontig) {
        if (g.b_kcontig) PRESK_STAGED(true, true);
        else PRESK_STAGED(true, false);
    } else if constexpr (OB == kOpF32 || OB == kOpHalf) {
        if (g.b_kcontig) PRESK_STAGED(false, true);
        else PRESK_STAGED(false, false);
    } else {
        return hipErrorInvalidValue;
    }
#undef PRESK_STAGED
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? split_reduce<ST>(g, stream) : e;
}

// each operand one run of elements along k, or along its rows, at strides
// that keep a tile's offsets in 32 bits
inline bool staged_strides(const GemmArgs& g) {
    const long long lim = 1ll << 22;
    return (g.sa_k == 1 || g.sa_m == 1) && (g.sb_k == 1 || g.sb_n == 1) && g.sa_m < lim && g.sa_k < lim && g.sb_k < lim &&
           g.sb_n < lim;
}
// every vector of V elements whole
inline bool staged_whole(const GemmArgs& g, int va, int vb) {
    return (g.a_kcontig ? g.K : g.M) % va == 0 && (g.b_kcontig ? g.K : g.N) % vb == 0;
}

}  // namespace

}  // namespace presk
