// EXACT mode's contractions: every output the running sum of its products in
// index order from zero, the product and the sum each rounded to f32 as the
// interpreter rounds them (crates/presk-kernel/src/exec.rs:619-896) -- the
// printed nest's bits, computed tile by tile.
//
// Bound: two VALU instructions a product (mul, add; binary16's products are
// exact in f32, so one fma).  256 threads hold a 64 x 64 (32 x 32, 16 x 16) tile,
// 4 x 4 (2 x 2, 1) outputs each, and 32-deep blocks of both operands as f32 in
// LDS; a k's operands are read while the k before is multiplied, the next
// block's loads are in flight while one is multiplied (16-bit elements widened
// on their way to LDS: on arrival, each load was waited for, 43 ns a k against
// 32 in f32).  Elements are loaded one by one through general strides, along
// whichever axis is contiguous, so any size and alignment takes the same path.  Rows and columns past the operands
// repeat the last, k past them are zero: a sum from +0 is never -0, so adding
// +0 changes no bit.
//
// Against the printed nest, f32: 2048 x 384 x 384 54 -> 22 us, 4096 x 1024 x
// 1024 567 -> 178 us (48 TFLOP/s), 16384 x 384 x 1536 with k-contiguous
// operands 5.0 -> 0.38 ms, [384 x 1536] over K 16384 11.9 -> 0.79 ms, 2048 x 65
// x 384 (a row-wise nest, its row in one thread) 2.15 ms -> 17 us.  The course
// GPT's forward at B 8 x T 256: 9.17 -> 2.24 ms.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_store.hpp"

namespace presk {

namespace {

template <int ST>
__device__ __forceinline__ float widen(typename std::conditional<ST == kF32, float, unsigned short>::type x) {
    if constexpr (ST == kF32) return x;
    else return ST == kBF16 ? pk_bf16_to_f32(x) : pk_f16_to_f32(x);
}

// One operand's block (ROWS x BK) as f32 in LDS, [k][ROWS + 4]: KC takes BK k
// of a row side by side, else ROWS rows of a k.  Offsets from the block's
// first element are 32-bit and fixed (the plan bounds the strides); a block
// moves the uniform origin.  Rows past the operand read its last one (their
// sums are never stored), k past K are zero.
template <int ST, bool KC, int ROWS, int BK>
struct SeqLoader {
    static constexpr int LD = ROWS + 4, NV = ROWS * BK / 256, ESZ = ST == kF32 ? 4 : 2;
    const char* origin;
    long long step;
    unsigned voff[NV];
    typedef typename std::conditional<ST == kF32, float, unsigned short>::type S;
    S r[NV];                     // as stored: widened on arrival they would be waited for there
    __device__ __forceinline__ static int row_of(int q) { return KC ? (q * 256 + threadIdx.x) / BK : (q * 256 + threadIdx.x) % ROWS; }
    __device__ __forceinline__ static int k_of(int q) { return KC ? (q * 256 + threadIdx.x) % BK : (q * 256 + threadIdx.x) / ROWS; }
    __device__ __forceinline__ void init(const void* p, long long base, int rows, long long rs, long long ks, int row0) {
        origin = (const char*)p + ESZ * (base + (long long)row0 * rs);
        step = (long long)ESZ * BK * ks;
        const int last = rows - 1 - row0;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int row = row_of(q);
            voff[q] = (unsigned)ESZ * ((unsigned)(row < last ? row : last) * (unsigned)rs + (unsigned)k_of(q) * (unsigned)ks);
        }
    }
    // the block at the origin, `left` of whose k exist
    __device__ __forceinline__ void load(int left) {
        if (left >= BK) {
#pragma unroll
            for (int q = 0; q < NV; ++q) r[q] = *(const S*)(origin + voff[q]);
        } else {
#pragma unroll
            for (int q = 0; q < NV; ++q) r[q] = k_of(q) < left ? *(const S*)(origin + voff[q]) : S(0);
        }
        origin += step;
    }
    __device__ __forceinline__ void store(float* tile) const {
#pragma unroll
        for (int q = 0; q < NV; ++q) tile[k_of(q) * LD + row_of(q)] = widen<ST>(r[q]);
    }
};

// a thread's R elements of a LDS row
template <int R>
__device__ __forceinline__ void take(const float* row, int t, float (&v)[R]) {
    typedef float vec __attribute__((ext_vector_type(R)));
    const vec x = *(const vec*)&row[t * R];
#pragma unroll
    for (int e = 0; e < R; ++e) v[e] = x[e];
}

// 256 threads as 16 x 16, thread (tx, ty) holding RM x RN outputs
template <int ST, bool AK, bool BKC, int RM, int RN>
__global__ void __launch_bounds__(256, 4) seq_gemm_kernel(GemmArgs g) {
    constexpr int BM = 16 * RM, BN = 16 * RN, BK = 32;
    typedef SeqLoader<ST, AK, BM, BK> LA;
    typedef SeqLoader<ST, BKC, BN, BK> LB;
    __shared__ __attribute__((aligned(16))) float smem[2][BK * (LA::LD + LB::LD)];
    const unsigned tiles = (unsigned)g.tiles_m * (unsigned)g.tiles_n;
    const unsigned batch = blockIdx.x / tiles, bid = blockIdx.x - batch * tiles;
    const unsigned tm = bid / (unsigned)g.tiles_n, tn = bid - tm * (unsigned)g.tiles_n;
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
    const int M = (int)g.M, N = (int)g.N, K = (int)g.K;
    const int m0 = (int)tm * BM, n0 = (int)tn * BN;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    float acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) acc[i][j] = 0.f;

    LA la;
    LB lb;
    la.init(g.A, a_off, M, g.sa_m, g.sa_k, m0);
    lb.init(g.B, b_off, N, g.sb_n, g.sb_k, n0);
    la.load(K);
    lb.load(K);
    la.store(smem[0]);
    lb.store(smem[0] + BK * LA::LD);
    __syncthreads();
    int cur = 0;
    for (int kb = 0; kb < K; kb += BK, cur ^= 1) {
        const bool more = kb + BK < K;
        if (more) {
            la.load(K - kb - BK);
            lb.load(K - kb - BK);
        }
        const float* const as = smem[cur];
        const float* const bs = smem[cur] + BK * LA::LD;
        // G k's operands are read while the G before are multiplied (left
        // alone the compiler reads the whole block ahead, 256 registers of
        // it, and one wave a SIMD remains); a 16 x 16 tile's products of one
        // k are over long before the next k's operands are there
        constexpr int G = RM == 1 ? 4 : 1;
        float a[2][G][RM], b[2][G][RN];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            take<RM>(as + k * LA::LD, ty, a[0][k]);
            take<RN>(bs + k * LB::LD, tx, b[0][k]);
        }
#pragma unroll
        for (int k0 = 0; k0 < BK; k0 += G) {
            const int now = k0 / G & 1;
#pragma unroll
            for (int k = 0; k < G; ++k)
                if (k0 + G < BK) {
                    take<RM>(as + (k0 + G + k) * LA::LD, ty, a[now ^ 1][k]);
                    take<RN>(bs + (k0 + G + k) * LB::LD, tx, b[now ^ 1][k]);
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < G; ++k)
#pragma unroll
                for (int i = 0; i < RM; ++i)
#pragma unroll
                    for (int j = 0; j < RN; ++j)
                        acc[i][j] = ST == kF16 ? __builtin_fmaf(a[now][k][i], b[now][k][j], acc[i][j])
                                               : acc[i][j] + a[now][k][i] * b[now][k][j];
            __builtin_amdgcn_sched_barrier(0);
        }
        // the sums belong to this block: without this they are moved past the
        // stores below, and every operand with them is kept in a register
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j) asm volatile("" : "+v"(acc[i][j]));
        if (more) {
            la.store(smem[cur ^ 1]);
            lb.store(smem[cur ^ 1] + BK * LA::LD);
        }
        __syncthreads();
    }

    bool ovf = false;
#pragma unroll
    for (int i = 0; i < RM; ++i) {
        const int m = m0 + ty * RM + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < RN; ++j) {
            const int n = n0 + tx * RN + j;
            if (n >= N) continue;
            float b = 0.f;
            if (g.bias)
                b = load_bias<ST>(g.bias, g.bias_kind == 1 ? n : g.bias_kind == 2 ? (long long)m * N + n : 0);
            store_out<ST>(g.C, c_off + (long long)m * g.sc_m + n, acc[i][j], g.bias != nullptr, b, ovf);
        }
    }
    if (ovf && g.flag) atomicOr(g.flag, 1u);
}

template <int ST, int RM, int RN>
hipError_t launch(const GemmArgs& g0, hipStream_t stream) {
    GemmArgs g = g0;
    g.tiles_m = (int)((g.M + 16 * RM - 1) / (16 * RM));
    g.tiles_n = (int)((g.N + 16 * RN - 1) / (16 * RN));
    const long long items = (long long)g.tiles_m * g.tiles_n * g.batch;
    if (items <= 0) return hipSuccess;
    if (items > 0x7fffffffLL) return hipErrorInvalidValue;
    const unsigned n = (unsigned)items;
    if (g.a_kcontig && g.b_kcontig) seq_gemm_kernel<ST, true, true, RM, RN><<<n, 256, 0, stream>>>(g);
    else if (g.a_kcontig) seq_gemm_kernel<ST, true, false, RM, RN><<<n, 256, 0, stream>>>(g);
    else if (g.b_kcontig) seq_gemm_kernel<ST, false, true, RM, RN><<<n, 256, 0, stream>>>(g);
    else seq_gemm_kernel<ST, false, false, RM, RN><<<n, 256, 0, stream>>>(g);
    return hipGetLastError();
}

template <int ST>
hipError_t launch_st(const GemmArgs& g, hipStream_t stream) {
    // 64 x 64 tiles where they are three a CU or more, else 32 x 32 (2048 x
    // 384 x 384: 38 us on 192 of the former, 22 on 768 of the latter; 4096 x
    // 1024 x 1024: 178 and 204).  Larger tiles gain nothing a product and
    // leave waves too few to cover their latency (128 x 64: 195 us).
    const long long t = ((g.M + 63) / 64) * ((g.N + 63) / 64) * g.batch;
    // And 16 x 16 where even the 32 x 32 ones leave CUs idle, since a workgroup
    // is one serial chain over K, bound by latency: against the printed nest,
    // whose threads hold one output each in such shapes, 32 x 32 tiles took up
    // to 2.4x as long in 16-bit storage (256 x 128 x 11552, bf16, k-contiguous:
    // printed 274 us, 32 x 32 651) and 16 x 16 ones take 0.1-1.0x (of 900 shapes
    // all but two of 4 us, K 56 and 112).  From 192 of the 32 x 32 ones on those
    // are level or ahead (16 x 16 against them: 128-191 0.83-0.97x, 192-255
    // 0.95-1.14x).
    const long long t2 = ((g.M + 31) / 32) * ((g.N + 31) / 32) * g.batch;
    if (t2 < 192) return launch<ST, 1, 1>(g, stream);
    return t >= 768 ? launch<ST, 4, 4>(g, stream) : launch<ST, 2, 2>(g, stream);
}

}  // namespace

hipError_t gemm_seq_launch(const GemmArgs& g, hipStream_t stream) {
    switch (g.storage) {
        case kF32: return launch_st<kF32>(g, stream);
        case kBF16: return launch_st<kBF16>(g, stream);
        case kF16: return launch_st<kF16>(g, stream);
    }
    return hipErrorInvalidValue;
}

}  // namespace presk
