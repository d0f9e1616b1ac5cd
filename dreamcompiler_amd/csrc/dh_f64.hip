// dh_f64.hip -- the fp64 half of the hot path: the products and attention the reference
// computes in double precision.
//
// The reference runs `@` below its dispatch threshold (M*N < gpu_dispatch_threshold()) in
// fp64 with dream_gemm_d (runtime/ops/elementwise.inc:1033-1040, 593-638), flash attention
// outside B*S*S >= 262144 && dk <= 128 with its fp64 online-softmax loop
// (runtime/nn/training.inc:307-308, 336, 366-399), and standard attention always in fp64
// (training.inc:178-263).  This file gives those results on the GPU in fp64.
//
// GEMM.  dream_gemm_d zeroes C and, per 256-deep k block (its KC), adds to every element the
// sum of that block's products, each block's sum being one fused multiply-add chain in k
// order started from zero (the 4x8 AVX2 micro-kernel, elementwise.inc:547-585).  Here the
// fp64 matrix cores run exactly those chains: v_mfma_f64_16x16x4f64 performs the four
// products of each output as sequential IEEE fused multiply-adds in k order (round to nearest
// even, as _mm256_fmadd_pd), so an accumulator started from zero and fed the k-steps in order
// is the chain; it is added to a running total at every 256-boundary of k.  With beta = 0 and
// alpha = 1 the result is therefore bit-identical to the reference's fp64 `@`.  Grids too
// small for the chip split K at those 256-boundaries and sum the block sums in k order in a
// second launch, which keeps the identity.
//
// Attention.  The standard form of training.inc:178-263 on fp64 GEMMs: scores = Q K^T
// (one batched NT product per chunk of slices), a row kernel applies the scale, the causal
// mask and the softmax (max, exp, sum, divide), O = P V; the backward
// (runtime/ops/autograd.inc:675-778) recomputes P, then dV += P^T dO, dP = dO V^T,
// dS = P (dP - rowsum(dP P)), dQ += scale dS K, dK += scale dS^T Q.  Causal products leave out
// what the mask zeroes (F64_SCORES ...).  Score buffers come from the pool in chunks of slices
// (at most 256 MB per buffer).
//
// Bound by the fp64 matrix cores.  16 causal slices of 1024 x 256, forward + backward: 1520 ->
// 721 us (30 GFLOP visible, 42 TFLOP/s); 4096^3 53.5 -> 60.8 (NN), 65.0 (TN) TFLOP/s of the
// 70 that a library product reaches here.
#include "dh_common.hpp"

#include <math.h>
#include <cstdlib>
#include <type_traits>

namespace dh {
namespace {

constexpr int F64_KC = 256;       // the reference's KC: chains restart every 256 k
constexpr int F64_THREADS = 256;  // four waves as 2 x 2, each WB x WB blocks of 16 x 16

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// Which part of a product a causal attention needs (query row0 + m or key k visible up to the
// diagonal), so that masked blocks are neither computed nor read:
//   F64_SCORES     C[m][n]: tiles whose keys n all lie past their queries row0 + m are left out;
//   F64_TO_DIAG    A[m][k] masked past k = row0 + m: k stops at the end of the tile's queries;
//   F64_FROM_DIAG  A^T[m][k] (m a key, k a query row0 + k): k starts at the tile's first key.
// A masked product of finite values is an exact zero, and adding it changes no chain.  Within a
// tile and a stage of the diagonal it is formed all the same: a masked zero times an infinity or
// NaN makes a NaN there, and outputs that are NaN are formed again from their visible k
// (f64_visible).  So every output depends on what its queries and keys see, as in the
// reference's loops, whatever the tile.  The row kernels write zeros up to F64_PAD keys past the diagonal, as
// far as a tile's edge and a stage's start reach.
enum { F64_ALL = 0, F64_SCORES, F64_TO_DIAG, F64_FROM_DIAG };
constexpr int F64_PAD = 80;       // 64-wide tile + 16-deep stage (or 32 + 32)

// Explicitly global pointers: through the argument struct they would become flat loads.
typedef const double __attribute__((address_space(1)))* GlobalF64;
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));
typedef const f64x2u __attribute__((address_space(1)))* GlobalF64x2;
typedef const char __attribute__((address_space(1)))* GlobalBytes;
__device__ double g_zero64;   // zero-initialised, never written

__device__ inline __amdgpu_buffer_rsrc_t f64_rsrc(GlobalBytes p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(const void*)p, 0, bytes, 0x00020000);
}
// Two doubles at byte offset off; words past the resource's range (F64_OOB always is) read zero.
// The opaque offset keeps the four 32-bit loads at constant distances, so that the backend
// merges them into one 128-bit load.
constexpr int F64_OOB = -16;
__device__ inline f64x2 f64_load2(__amdgpu_buffer_rsrc_t rs, int off) {
    asm volatile("" : "+v"(off));
    float v[4];
    buf_load_floats<4>(rs, off, v);
    return __builtin_bit_cast(f64x2, f32x4{v[0], v[1], v[2], v[3]});
}

struct F64Args {
    int M, N, K;
    double alpha;
    const double* A;
    int lda;
    long long sA;
    const double* B;
    int ldb;
    long long sB;
    double beta;
    double* C;
    int ldc;
    long long sC;
    int tilesN;
    double* part;                 // split mode: the chain sums' buffer
    int causal, row0, snake;
};

// One output of a causal product from its visible k alone, k0 .. k1 - 1: the chains and block sums
// of the kernel below.
template <int TA>
__device__ inline double f64_visible(const F64Args& ar, long long b, int m, int n, int k0, int k1) {
    GlobalF64 A = (GlobalF64)(ar.A + b * ar.sA), B = (GlobalF64)(ar.B + b * ar.sB);
    double sum = 0.0;
    for (int kb = k0 / F64_KC * F64_KC; kb < k1; kb += F64_KC) {
        double c = 0.0;
        for (int k = max(k0, kb); k < min(k1, kb + F64_KC); ++k)
            c = __builtin_fma(A[TA == 0 ? (long long)m * ar.lda + k : (long long)k * ar.lda + m],
                              B[(long long)k * ar.ldb + n], c);
        sum = sum + c;
    }
    return sum;
}

template <int WB, int KT>
struct F64Cfg {
    static constexpr int TILE = 32 * WB;                    // work-group tile side
    static constexpr int NLD = TILE * KT / 2 / F64_THREADS; // A (and B) pairs per thread
    // LDS copy of an operand tile in its global order, so the stores from global memory
    // are conflict-free as well as the MFMA operand reads (16 consecutive rows or columns
    // of one k, times 4 k, per wave):
    //   k-contiguous (A untransposed, B transposed): [row][k], row pitch KT + 2 doubles (16
    //   rows start 4 banks apart, the 2 k of a half-wave fill the gaps);
    //   row-contiguous (A transposed, B untransposed): [k][row], odd k with halves of 16 rows
    //   swapped (the 2 k of a half-wave on opposite halves of the 64 banks).
    static constexpr int KP = KT + 2, RP = TILE;
    __device__ static int at_k(int row, int k) { return row * KP + k; }
    __device__ static int at_r(int row, int k) { return k * RP + (row ^ (16 * (k & 1))); }
    static constexpr int SZ_K = TILE * KP, SZ_R = KT * RP;
};

// One TILE x TILE output tile.  Products run on v_mfma_f64_16x16x4f64, which performs its four
// products of an output as sequential IEEE fused multiply-adds in k order (a GPU probe over 7 M
// outputs -- integers, N(0,1), exponents over 2^+-30, subnormals, infinities and NaNs, 64-step
// chains -- found it bitwise equal to the fma chain), so each accumulator is exactly the
// reference's chain.  Operand layout: lane l holds A[l % 16][k0 + l / 16] and
// B[k0 + l / 16][l % 16]; result register r holds D[l / 16 + 4 r][l % 16].  k past the range
// is zero in both operands, and fma(0, 0, c) = c for every chain value (a chain started at +0
// never holds -0), so padded k-steps change nothing.
//
// G groups of four waves share the tile: group g runs the chains of the 256-deep blocks
// g, g + G, ... and the chain sums meet in LDS, where group 0 adds them in k order.  A
// small grid is bound by the chain of memory latencies of a work-group's k-stages; G groups
// run G such chains at a time without a second launch and its partials.  Each group stages its
// own operands: KT k per stage, double-buffered in LDS.  DEEP: stages in pairs, two in flight in
// registers (a load has two stages' products to land); else stage by stage, one in flight, in
// the compiler's schedule.  With `part`, blockIdx.z takes G blocks and every
// group writes its chain sum there instead.
template <int TA, int TB, int WB, int KT, int G, bool WIDE, bool DEEP>
__global__ __launch_bounds__(F64_THREADS * G, WB == 2 ? 4 : 1) void gemm_f64_kernel(F64Args ar) {
    using Cf = F64Cfg<WB, KT>;
    constexpr int TILE = Cf::TILE, NLD = Cf::NLD;
    constexpr int SZA = TA == 0 ? Cf::SZ_K : Cf::SZ_R, SZB = TB == 1 ? Cf::SZ_K : Cf::SZ_R;
    constexpr int SPB = F64_KC / KT;             // stages per block
    static_assert(SPB % 2 == 0, "stages run in pairs");
    static_assert(DEEP || G == 1, "stage by stage: no groups");
    static_assert(G == 1 || SZA + SZB >= TILE * TILE, "a stage buffer holds a group's chain sums");
    __shared__ __attribute__((aligned(16))) double lds[G][2][SZA + SZB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    const int g = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const int t = tid & (F64_THREADS - 1);
    const int wr = 16 * WB * (wave & 1), wc = 16 * WB * (wave >> 1);   // wave's sub-tile
    const int M = ar.M, N = ar.N, K = ar.K;
    int tile = blockIdx.x;
    long long b = blockIdx.y;
    if (ar.causal >= F64_TO_DIAG) {
        // Unequal k-ranges: the tiles of every member by length, longest first, in runs of
        // `snake` (the CU count) that alternate direction, so that the work-groups a CU is dealt
        // (one of each run) add up to about the same length.  Causal P V of 16 slices
        // of 1024 x 256, same box: 142 us in tile order, 100 us so.
        const int lin = blockIdx.y * gridDim.x + blockIdx.x, all = gridDim.x * gridDim.y;
        const int run = lin / ar.snake, base = run * ar.snake;
        const int len = min(ar.snake, all - base);
        const int rank = run & 1 ? base + len - 1 - (lin - base) : lin;
        tile = rank / gridDim.y;
        b = rank - tile * gridDim.y;
        if (ar.causal == F64_TO_DIAG) tile = gridDim.x - 1 - tile;
    }
    int tm, tn;
    if (ar.causal == F64_SCORES) {
        // the grid holds the visible tiles only: tile row tm has tm + 1 + o of them (the last one
        // may lie past N), tm (tm + 1) / 2 + tm o before it
        const int o = (ar.row0 + TILE - 1) / TILE;
        const float h = o + 0.5f;
        tm = (int)(sqrtf(h * h + 2.f * tile) - h);
        while (tm * (tm + 1) / 2 + tm * o > tile) --tm;
        while ((tm + 1) * (tm + 2) / 2 + (tm + 1) * o <= tile) ++tm;
        tn = tile - (tm * (tm + 1) / 2 + tm * o);
        if (tn >= ar.tilesN) return;
    } else if (ar.causal == F64_ALL) {
        // each XCD a 4-row block of tiles: its work-groups share operand rows in its L2
        xcd_tile_order(tile, gridDim.x, (M + TILE - 1) / TILE, ar.tilesN, 4, tm, tn);
    } else {
        tm = tile / ar.tilesN;
        tn = tile % ar.tilesN;
    }
    // scalar registers (the tile search goes through the vector ALU)
    const int m0 = __builtin_amdgcn_readfirstlane(tm) * TILE;
    const int n0 = __builtin_amdgcn_readfirstlane(tn) * TILE;
    int kbeg = 0, kend = K;
    if (ar.causal == F64_TO_DIAG) kend = min(K, ar.row0 + m0 + TILE);
    if (ar.causal == F64_FROM_DIAG) kbeg = max(0, m0 - ar.row0) / KT * KT;
    // blocks from blk0 on, G of them a round; stage q of group g starts at k_of(q)
    int blk0 = kbeg / F64_KC * F64_KC;
    if (ar.part) {
        blk0 = blockIdx.z * (G * F64_KC);
        kend = min(kend, blk0 + G * F64_KC);
    }
    const int left = kend - blk0;
    const int rounds = left > 0 ? (left + G * F64_KC - 1) / (G * F64_KC) : 0;
    const int last = left - (rounds - 1) * (G * F64_KC);     // k of the last round
    const int nq = rounds ? (rounds - 1) * SPB + (min(last, F64_KC) + KT - 1) / KT : 0;
    const int q0 = G == 1 && kbeg > blk0 ? (kbeg - blk0) / KT & ~1 : 0;
    auto k_of = [&](int q) { return blk0 + (q / SPB * G + g) * F64_KC + q % SPB * KT; };

    // This thread's NLD pairs of values per operand, two consecutive along the contiguous index
    // (a load instruction costs its issue whatever its width), as loop-invariant byte offsets
    // from a base that moves with the stage: a stage spends next to no vector ALU time, which
    // fp64 products need, on addresses.  k outside the range (the ragged last stage, a stage past
    // the end, masked values before kbeg that nobody wrote) reads zero through an offset or a
    // buffer range that excludes it, or is dropped by stash(): no branch, so nothing waits for
    // a load before its stash.  kbeg is a multiple of KT: no stage straddles it.  A row past the
    // edge reads the last row: its values reach only results that are not stored.  The buffer
    // range ends with the operand's last valid value.
    int ak[NLD], bk[NLD], arow[NLD], brow[NLD];
    size_t ao[NLD], bo[NLD];
    const int ma = min(TILE, M - m0), nb = min(TILE, N - n0);   // valid rows of the tile
#pragma unroll
    for (int r = 0; r < NLD; ++r) {
        const int f = t + F64_THREADS * r;
        ak[r] = TA == 0 ? 2 * (f % (KT / 2)) : f / (TILE / 2);
        arow[r] = TA == 0 ? f / (KT / 2) : 2 * (f % (TILE / 2));
        bk[r] = TB == 1 ? 2 * (f % (KT / 2)) : f / (TILE / 2);
        brow[r] = TB == 1 ? f / (KT / 2) : 2 * (f % (TILE / 2));
        const size_t am = min(arow[r], ma - 1), bn = min(brow[r], nb - 1);
        ao[r] = 8 * (TA == 0 ? am * ar.lda + ak[r] : ak[r] * (size_t)ar.lda + am);
        bo[r] = 8 * (TB == 1 ? bn * ar.ldb + bk[r] : bk[r] * (size_t)ar.ldb + bn);
    }
    const GlobalBytes abase = (GlobalBytes)(ar.A + b * ar.sA + (TA == 0 ? (long long)m0 * ar.lda : m0));
    const GlobalBytes bbase = (GlobalBytes)(ar.B + b * ar.sB + (TB == 1 ? (long long)n0 * ar.ldb : n0));
    auto valid_of = [&](int q) {   // k of stage q inside the range
        const int k0 = k_of(q);
        return q < nq && k0 >= kbeg && k0 < kend ? min(kend - k0, KT) : 0;
    };
    f64x2 ra[2][NLD], rb[2][NLD];
    auto fetch = [&](auto set_c, int q) {
        constexpr int set = decltype(set_c)::value;
        const int k0 = k_of(q), valid = valid_of(q);
        const GlobalBytes pa = abase + 8LL * (TA == 0 ? k0 : (long long)k0 * ar.lda);
        const GlobalBytes pb = bbase + 8LL * (TB == 1 ? k0 : (long long)k0 * ar.ldb);
        if (WIDE && valid == KT && ma == TILE && nb == TILE) {   // 64-bit offsets
#pragma unroll
            for (int r = 0; r < NLD; ++r) {
                ra[set][r] = *(GlobalF64x2)(pa + ao[r]);
                rb[set][r] = *(GlobalF64x2)(pb + bo[r]);
            }
        } else if constexpr (WIDE) {   // the same at an edge, value by value
            const GlobalBytes zero = (GlobalBytes)&g_zero64;
#pragma unroll
            for (int r = 0; r < NLD; ++r)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const bool ain = TA == 0 ? ak[r] + e < valid : ak[r] < valid && arow[r] + e < ma;
                    const bool bin = TB == 1 ? bk[r] + e < valid : bk[r] < valid && brow[r] + e < nb;
                    ra[set][r][e] = *(GlobalF64)(ain ? pa + ao[r] + 8 * e : zero);
                    rb[set][r][e] = *(GlobalF64)(bin ? pb + bo[r] + 8 * e : zero);
                }
        } else {
            const int lasta = TA == 0 ? (ma - 1) * ar.lda + valid : (valid - 1) * ar.lda + ma;
            const int lastb = TB == 1 ? (nb - 1) * ar.ldb + valid : (valid - 1) * ar.ldb + nb;
            const __amdgpu_buffer_rsrc_t sa = f64_rsrc(pa, __builtin_amdgcn_readfirstlane(valid ? 8 * lasta : 0));
            const __amdgpu_buffer_rsrc_t sb = f64_rsrc(pb, __builtin_amdgcn_readfirstlane(valid ? 8 * lastb : 0));
#pragma unroll
            for (int r = 0; r < NLD; ++r) {
                ra[set][r] = f64_load2(sa, TA == 1 || ak[r] < valid ? (int)ao[r] : F64_OOB);
                rb[set][r] = f64_load2(sb, TB == 0 || bk[r] < valid ? (int)bo[r] : F64_OOB);
            }
        }
    };
    auto stash = [&](auto set_c, int q) {
        constexpr int set = decltype(set_c)::value;
        double* d = lds[g][DEEP ? set : q & 1];
        const int valid = valid_of(q);
#pragma unroll
        for (int r = 0; r < NLD; ++r) {
            f64x2 va = ra[set][r], vb = rb[set][r];
            // k along a row: the pair that holds the range's end read the next value with it
            if (TA == 0) va[1] = ak[r] + 1 < valid ? va[1] : 0.0;
            if (TB == 1) vb[1] = bk[r] + 1 < valid ? vb[1] : 0.0;
            *reinterpret_cast<f64x2*>(d + (TA == 0 ? Cf::at_k(arow[r], ak[r]) : Cf::at_r(arow[r], ak[r]))) = va;
            *reinterpret_cast<f64x2*>(d + SZA + (TB == 1 ? Cf::at_k(brow[r], bk[r]) : Cf::at_r(brow[r], bk[r]))) = vb;
        }
    };

    f64x4 tot[WB][WB], acc[WB][WB];
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) tot[i][j][r] = acc[i][j][r] = 0.0;
    const int kr0 = lane >> 4, c0 = lane & 15;
    auto step = [&](auto set_c, int q) {   // stage q from LDS buffer q % 2 = set
        constexpr int set = decltype(set_c)::value;
        fetch(set_c, q + (DEEP ? 2 : 1));
        if (DEEP) __builtin_amdgcn_sched_barrier(0);
        const double* as = lds[g][DEEP ? set : q & 1];
        const double* bs = as + SZA;
        double a[KT / 4][WB], bb[KT / 4][WB];
#pragma unroll
        for (int k4 = 0; k4 < KT / 4; ++k4) {
            const int kr = 4 * k4 + kr0;
#pragma unroll
            for (int i = 0; i < WB; ++i) {
                const int row = wr + 16 * i + c0, col = wc + 16 * i + c0;
                a[k4][i] = as[TA == 0 ? Cf::at_k(row, kr) : Cf::at_r(row, kr)];
                bb[k4][i] = bs[TB == 1 ? Cf::at_k(col, kr) : Cf::at_r(col, kr)];
            }
        }
        // One block per wave: a dependent chain of products; with the reads between them each
        // pair waited for its own LDS latency (200 cycles a product instead of 64), so a
        // stage's reads all go first.
        if (DEEP && WB == 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k4 = 0; k4 < KT / 4; ++k4)
#pragma unroll
            for (int i = 0; i < WB; ++i)
#pragma unroll
                for (int j = 0; j < WB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k4][i], bb[k4][j], acc[i][j], 0, 0, 0);
        // stage q + 1, fetched a step ago; kept behind the products (the scheduler would move its
        // wait to the front, and the loads would have one stage to land instead of two)
        if (DEEP) __builtin_amdgcn_sched_barrier(0);
        stash(std::integral_constant<int, DEEP ? set ^ 1 : 0>{}, q + 1);
        __syncthreads();
    };
    // A pair's second stage past the end multiplies zeros, so the loop has no branch around the
    // accumulators; the blocks of 256 k are an outer loop, which adds their chain sums in k order.
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    if (q0 < nq) {
        fetch(even, q0);
        if (DEEP) fetch(odd, q0 + 1);
        stash(even, q0);
        __syncthreads();
    }
    for (int q = q0; q < nq;) {
        const int qe = min(nq, (q / SPB + 1) * SPB);
        if constexpr (DEEP) {
            for (; q < qe; q += 2) {
                step(even, q);
                step(odd, q + 1);
            }
        } else {
            for (; q < qe; ++q) step(even, q);
        }
        if (G > 1 && !ar.part) {
            // lds[.][1] was read in the last step and is not written before the next round
            auto at = [&](int grp, int i, int j, int r) -> double& {
                return lds[grp][1][(((wave * WB + i) * WB + j) * 4 + r) * 64 + lane];
            };
            if (g > 0) {
#pragma unroll
                for (int i = 0; i < WB; ++i)
#pragma unroll
                    for (int j = 0; j < WB; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) at(g, i, j, r) = acc[i][j][r];
            }
            __syncthreads();
            if (g == 0) {
#pragma unroll
                for (int i = 0; i < WB; ++i)
#pragma unroll
                    for (int j = 0; j < WB; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            double s = tot[i][j][r] + acc[i][j][r];
                            for (int x = 1; x < G; ++x) s = s + at(x, i, j, r);
                            tot[i][j][r] = s;
                        }
            }
            __syncthreads();
        } else {
#pragma unroll
            for (int i = 0; i < WB; ++i)
#pragma unroll
                for (int j = 0; j < WB; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) tot[i][j][r] = tot[i][j][r] + acc[i][j][r];
        }
#pragma unroll
        for (int i = 0; i < WB; ++i)
#pragma unroll
            for (int j = 0; j < WB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0;
    }
    const int block = blockIdx.z * G + g;   // split mode: this group's block
    if (ar.part ? block * F64_KC >= K : g > 0) return;
    // lane l, register r of block (i, j): row wr + 16 i + l / 16 + 4 r, column wc + 16 j + l % 16
    if (TB == 0 && ar.causal >= F64_TO_DIAG) {
#pragma unroll
        for (int i = 0; i < WB; ++i)
#pragma unroll
            for (int j = 0; j < WB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int gm = m0 + wr + 16 * i + kr0 + 4 * r, gn = n0 + wc + 16 * j + c0;
                    if (tot[i][j][r] == tot[i][j][r] || gm >= M || gn >= N) continue;
                    int k0 = ar.causal == F64_TO_DIAG ? 0 : max(0, gm - ar.row0);
                    int k1 = ar.causal == F64_TO_DIAG ? min(K, ar.row0 + gm + 1) : K;
                    if (ar.part) {
                        k0 = max(k0, block * F64_KC);
                        k1 = min(k1, (block + 1) * F64_KC);
                    }
                    tot[i][j][r] = f64_visible<TA>(ar, b, gm, gn, k0, k1);
                }
    }
    double* out = ar.part ? ar.part + ((long long)block * gridDim.y + b) * ((long long)M * N)
                          : ar.C + b * ar.sC;
    const long long ld = ar.part ? N : ar.ldc;
    const double alpha = ar.alpha, beta = ar.beta;
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j) {
            const int gn = n0 + wc + 16 * j + c0;
            if (gn >= N) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gm = m0 + wr + 16 * i + kr0 + 4 * r;
                if (gm >= M) continue;
                double* c = out + (long long)gm * ld + gn;
                if (ar.part) {          // this block's chain sum, compact M x N per (block, member)
                    *c = tot[i][j][r];
                } else {
                    const double v = alpha == 1.0 ? tot[i][j][r] : alpha * tot[i][j][r];
                    *c = beta == 0.0 ? v : beta * *c + v;
                }
            }
        }
}

// Split-K finish: C = alpha * (((0 + s_0) + s_1) + ...) over the per-block chain sums in k
// order -- the reference's accumulation of its block sums into a zeroed C -- then beta.
__global__ __launch_bounds__(256) void gemm_f64_reduce(int M, int N, int nkb, int batch,
                                                       const double* __restrict__ part,
                                                       double alpha, double beta,
                                                       double* __restrict__ C, int ldc,
                                                       long long sC) {
    const long long mn = (long long)M * N, total = mn * batch;
    for (long long idx = (long long)blockIdx.x * 256 + threadIdx.x; idx < total;
         idx += (long long)gridDim.x * 256) {
        const long long b = idx / mn, rem = idx - b * mn;
        double tot = 0.0;
        for (int z = 0; z < nkb; ++z) tot = tot + part[((long long)z * batch + b) * mn + rem];
        double* c = C + b * sC + (rem / N) * (long long)ldc + rem % N;
        const double v = alpha == 1.0 ? tot : alpha * tot;
        *c = beta == 0.0 ? v : beta * *c + v;
    }
}

// Row softmax of one chunk of attention scores, in place: row r is query i = r mod S of its
// slice; x_j = s_j * scale over the row's visible keys (j <= i when causal), then
// p_j = exp(x_j - max x) / sum exp(x - max x), and exact zeros for masked keys (up to F64_PAD
// past the diagonal: no product reads further) (training.inc:193-201, 240-247).  One wave per
// row.  P holds `rows` score rows of S keys: consecutive groups of R rows are query rows
// row0 .. row0 + R - 1 of a slice (R = S, row0 = 0 for whole slices).
// Bound by memory: with NV > 0 (S <= 64 NV) the row stays in registers, so it is read and
// written once.
template <int NV>
__global__ __launch_bounds__(256) void attn_softmax_f64(double* __restrict__ P, int S,
                                                        long long rows, int R, int row0,
                                                        double scale, int causal) {
    // x = s * scale is rounded before the subtraction, as the reference stores it first.
#pragma clang fp contract(off)
    const long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    const int i = row0 + (int)(r % R);
    const int n = causal ? i + 1 : S, fill = causal ? min(S, i + F64_PAD) : S;
    double* row = P + r * (long long)S;
    double mx = -1e30, sum = 0.0;
    if constexpr (NV > 0) {
        double x[NV];
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            x[t] = row[min(lane + 64 * t, n - 1)] * scale;   // no branch: the loads overlap
        }
#pragma unroll
        for (int t = 0; t < NV; ++t)
            if (lane + 64 * t < n) mx = fmax(mx, x[t]);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) mx = fmax(mx, __shfl_xor(mx, d));
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            if (64 * t >= n) continue;   // wave-uniform
            if (lane + 64 * t < n) {
                x[t] = exp(x[t] - mx);
                sum += x[t];
            }
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d);
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            const int j = lane + 64 * t;
            if (j < fill) row[j] = j < n ? x[t] / sum : 0.0;
        }
    } else {
        for (int j = lane; j < n; j += 64) mx = fmax(mx, row[j] * scale);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) mx = fmax(mx, __shfl_xor(mx, d));
        for (int j = lane; j < n; j += 64) {
            const double e = exp(row[j] * scale - mx);
            row[j] = e;
            sum += e;
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d);
        for (int j = lane; j < fill; j += 64) row[j] = j < n ? row[j] / sum : 0.0;
    }
}

// dS = P o (dP - rowsum(dP o P)) in place of dP, zeros on masked keys up to F64_PAD past the
// diagonal (the softmax JVP of autograd.inc:711-714, 758-761).
template <int NV>
__global__ __launch_bounds__(256) void attn_softmax_bwd_f64(const double* __restrict__ P,
                                                            double* __restrict__ dP, int S,
                                                            long long rows, int R, int row0,
                                                            int causal) {
    const long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    const int i = row0 + (int)(r % R);
    const int n = causal ? i + 1 : S, fill = causal ? min(S, i + F64_PAD) : S;
    const double* p = P + r * (long long)S;
    double* g = dP + r * (long long)S;
    double rd = 0.0;
    if constexpr (NV > 0) {
        double pv[NV], gv[NV];
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            const int j = min(lane + 64 * t, n - 1);   // no branch: the loads overlap
            pv[t] = p[j];
            gv[t] = g[j];
        }
#pragma unroll
        for (int t = 0; t < NV; ++t)
            if (lane + 64 * t < n) rd = __builtin_fma(gv[t], pv[t], rd);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) rd += __shfl_xor(rd, d);
#pragma unroll
        for (int t = 0; t < NV; ++t) {
            const int j = lane + 64 * t;
            if (j < fill) g[j] = j < n ? pv[t] * (gv[t] - rd) : 0.0;
        }
    } else {
        for (int j = lane; j < n; j += 64) rd = __builtin_fma(g[j], p[j], rd);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) rd += __shfl_xor(rd, d);
        for (int j = lane; j < fill; j += 64) g[j] = j < n ? p[j] * (g[j] - rd) : 0.0;
    }
}

template <int WB, int KT, int G, bool WIDE = false, bool DEEP = true>
void launch_f64(int transA, int transB, dim3 grid, const F64Args& ar) {
#define DH_F64_LAUNCH(TA, TB) \
    gemm_f64_kernel<TA, TB, WB, KT, G, WIDE, DEEP><<<grid, F64_THREADS * G, 0, stream()>>>(ar)
    if (!transA && !transB) DH_F64_LAUNCH(0, 0);
    else if (!transA) DH_F64_LAUNCH(0, 1);
    else if (!transB) DH_F64_LAUNCH(1, 0);
    else DH_F64_LAUNCH(1, 1);
#undef DH_F64_LAUNCH
}

int gemm_f64_launch(int transA, int transB, int M, int N, int K, double alpha, const double* A,
                    int lda, long long sA, const double* B, int ldb, long long sB, double beta,
                    double* C, int ldc, long long sC, int batch, int causal = F64_ALL,
                    int row0 = 0) {
    // 64 x 64 tiles (2 x 2 blocks per wave) when they fill the chip twice over (from 1.6 times on for K
    // of one block), else 32 x 32.  K of few stages, and 32 x 32 tiles without groups, run stage by
    // stage: a pair of stages multiplies up to a whole stage of zeros, and with several
    // work-groups on a CU they cover each other's loads (us, pairs / stage by stage: 2048^2 x 11 14.4 /
    // 11.0, x 130 30.5 / 28.8, x 257 48.4 / 47.6; 1292 x 1395 x 34 13.2 / 10.3, 490 x 1561 x 11 8.2 / 6.4, 1000 x 700 x
    // 513 26.5 / 23.3, 1000 x 700 x 1030 49.5 / 45.9; but one block per work-group and CU, 1024 x 128 x 511, 11.9 /
    // 13.1).
    // A small grid is bound by the latencies of its work-groups' k-stages, so it runs the
    // 256-deep blocks of k side by side: one work-group per block, whose chain sums gemm_f64_reduce
    // adds in k order, where the tiles leave half the CUs idle (64^2 x 4096 77.7 -> 15.3, 300^2 x 1000
    // 21.8 -> 15.6), or up to four groups of waves in a work-group, as many as fit the CUs at once
    // (four take 135 KB of LDS, two 68 KB), whichever takes less by the two estimates below (in
    // us, fitted to tiles of 137 to 512 and 2 to 16 blocks; one group / groups / blocks: 511^3
    // 13.6 / 12.4 / 17.9, 500 x 300 x 1500 - / 31.7 / 22.8, 1756 x 149 x 2000 - / 51.0 / 37.4, 700^2 x 2000 - / 51.9 / 58.2).
    // Every form leaves the results bit-identical.  Leading dimensions that take a tile past
    // 32-bit offsets (2^22 to 2^24, see `wide`) have forms with 64-bit ones.
    const long long cus = num_cus();
    const long long tiles64 = ((M + 63) / 64) * (long long)((N + 63) / 64) * batch;
    const bool short2 = causal == F64_ALL && (tiles64 >= 2 * cus ? K <= 160 : K <= 256 && 5 * tiles64 >= 8 * cus);
    const int wb = tiles64 >= 2 * cus || short2 ? 2 : 1;
    // rows of a tile and stage: the tile's, or its k
    const int rows_a = transA ? (wb == 2 ? 16 : 32) : 32 * wb, rows_b = transB ? 32 * wb : wb == 2 ? 16 : 32;
    const bool wide = 8LL * rows_a * lda > 0x7fffffffLL || 8LL * rows_b * ldb > 0x7fffffffLL;
    const long long tilesM = (M + 32 * wb - 1) / (32 * wb), tilesN = (N + 32 * wb - 1) / (32 * wb);
    const long long tiles = tilesM * tilesN * batch;
    const long long nkb = ((long long)K + F64_KC - 1) / F64_KC;
    int G = 1;
    if (wb == 1 && !wide)
        while (G < 4 && G < nkb && tiles * G <= 2 * cus) G *= 2;
    const double blocks_us = 7.7 + 3.8 * (double)(tiles * nkb) / (double)cus;
    const double groups_us = G == 4 ? 5.5 + 13.2 * (double)(nkb / 4) + (nkb % 4 > 1 ? 13.2 : 3.7 * (nkb % 4))
                           : tiles <= cus ? 12.0 : 6.2 + 11.3 * (double)(nkb / 2) + (nkb % 2 ? 3.5 + 0.028 * ((K - 1) % F64_KC) : 0.0);
    const size_t pbytes = (size_t)nkb * batch * M * N * sizeof(double);
    double* part = nullptr;
    if (nkb > 1 && nkb <= 65535 && pbytes <= ((size_t)512 << 20) &&
        (2 * tiles <= cus || (G > 1 && blocks_us < groups_us && !capturing())))
        part = static_cast<double*>(dh_malloc(pbytes));   // none: the unsplit grid
    if (part) G = 1;
    const long long o = (row0 + 32 * wb - 1) / (32 * wb);   // F64_SCORES: visible tiles only
    const dim3 grid((unsigned)(causal == F64_SCORES ? tilesM * (tilesM + 1) / 2 + tilesM * o
                                                    : tilesM * tilesN),
                    (unsigned)batch,
                    part ? (unsigned)nkb : 1u);
    const F64Args ar{M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, (int)tilesN, part,
                     causal, row0, (int)cus};
    if (wide && wb == 2) launch_f64<2, 16, 1, true, false>(transA, transB, grid, ar);
    else if (wide) launch_f64<1, 32, 1, true, false>(transA, transB, grid, ar);
    else if (short2) launch_f64<2, 16, 1, false, false>(transA, transB, grid, ar);
    else if (wb == 2) launch_f64<2, 16, 1>(transA, transB, grid, ar);
    else if (G == 1 && !part && causal == F64_ALL && (K <= 16 || (K > 32 && K <= 48)))
        launch_f64<1, 16, 1, false, false>(transA, transB, grid, ar);
    else if (part && tiles * nkb <= cus) launch_f64<1, 32, 1>(transA, transB, grid, ar);
    else if (G == 1) launch_f64<1, 32, 1, false, false>(transA, transB, grid, ar);
    else if (G == 2) launch_f64<1, 32, 2>(transA, transB, grid, ar);
    else launch_f64<1, 32, 4>(transA, transB, grid, ar);
    if (part) {
        const long long total = (long long)M * N * batch;
        long long blocks = (total + 255) / 256;
        if (blocks > 8LL * num_cus()) blocks = 8LL * num_cus();
        gemm_f64_reduce<<<(unsigned)blocks, 256, 0, stream()>>>(M, N, (int)nkb, batch, part,
                                                                 alpha, beta, C, ldc, sC);
        dh_free(part);   // pooled: stream order keeps the buffer alive for the queued work
    }
    return check_launch("dh_gemm_f64");
}

int check_gemm_f64(const char* op, int transA, int transB, int M, int N, int K, const void* A,
                   int lda, long long sA, const void* B, int ldb, long long sB, const void* C,
                   int ldc, long long sC, int batch) {
    if (M < 0 || N < 0 || K < 0 || batch < 0)
        return set_error(DH_ERR_INVALID, "%s: negative shape (M=%d N=%d K=%d batch=%d)", op, M, N,
                         K, batch);
    if (M == 0 || N == 0 || batch == 0) return DH_OK;
    if (!C || (K > 0 && (!A || !B))) return set_error(DH_ERR_INVALID, "%s: null pointer", op);
    if ((K > 0 && (lda < (transA ? M : K) || ldb < (transB ? K : N))) || ldc < N)
        return set_error(DH_ERR_INVALID, "%s: leading dimension too small (lda=%d ldb=%d ldc=%d)",
                         op, lda, ldb, ldc);
    if (sA < 0 || sB < 0 || sC < 0)
        return set_error(DH_ERR_INVALID, "%s: negative batch stride", op);
    if (batch > 1 && sC < (long long)(M - 1) * ldc + N)
        return set_error(DH_ERR_INVALID, "%s: batch members of C overlap (strideC=%lld)", op, sC);
    if (batch > 65535)
        return set_error(DH_ERR_UNSUPPORTED, "%s: batch %d above 65535", op, batch);
    const long long tiles = (long long)((M + 31) / 32) * ((N + 31) / 32);
    if (tiles > 0x7fffffffLL)
        return set_error(DH_ERR_UNSUPPORTED, "%s: %lld output tiles", op, tiles);
    return DH_OK;
}

// Bytes one fp64 score buffer may take: 256 MB (DH_ATTN_F64_SCORE_BYTES overrides it, for
// tests of the row-block path at small S).
size_t attn_budget() {
    const char* e = std::getenv("DH_ATTN_F64_SCORE_BYTES");
    const long long v = e && *e ? std::atoll(e) : 0;
    return v > 0 ? (size_t)v : ((size_t)256 << 20);
}

// Work per pass over the scores: `chunk` whole slices of S x S scores when one slice fits the
// budget, else (chunk = 1) blocks of `rows` query rows of one slice, rows x S scores each.
struct AttnPass {
    int chunk, rows;
};
AttnPass attn_pass(int BH, int S) {
    const size_t budget = attn_budget();
    const size_t per = (size_t)S * S * sizeof(double);
    if (per <= budget) {
        size_t c = budget / (per ? per : 1);
        if (c > (size_t)BH) c = BH;
        if (c > 65535) c = 65535;
        return {(int)c, S};
    }
    size_t r = budget / ((size_t)S * sizeof(double));
    if (r < 1) r = 1;
    return {1, (int)r};
}

int check_attn_f64(const char* op, int BH, int S, int D) {
    if (BH < 0 || S < 0 || D < 0)
        return set_error(DH_ERR_INVALID, "%s: negative shape (BH=%d S=%d D=%d)", op, BH, S, D);
    if ((long long)S * D > 0x7fffffffLL)
        return set_error(DH_ERR_UNSUPPORTED, "%s: S*D = %lld above 2^31", op, (long long)S * D);
    if (S > 46340)
        return set_error(DH_ERR_UNSUPPORTED, "%s: S = %d (S*S above 2^31)", op, S);
    return DH_OK;
}

void launch_softmax(double* P, int S, long long rows, int R, int row0, double scale,
                    int causal) {
    const unsigned grid = (unsigned)((rows + 3) / 4);
    if (S <= 256) attn_softmax_f64<4><<<grid, 256, 0, stream()>>>(P, S, rows, R, row0, scale, causal);
    else if (S <= 1024) attn_softmax_f64<16><<<grid, 256, 0, stream()>>>(P, S, rows, R, row0, scale, causal);
    else attn_softmax_f64<0><<<grid, 256, 0, stream()>>>(P, S, rows, R, row0, scale, causal);
}

void launch_softmax_bwd(const double* P, double* G, int S, long long rows, int R, int row0,
                        int causal) {
    const unsigned grid = (unsigned)((rows + 3) / 4);
    if (S <= 256) attn_softmax_bwd_f64<4><<<grid, 256, 0, stream()>>>(P, G, S, rows, R, row0, causal);
    else if (S <= 1024) attn_softmax_bwd_f64<16><<<grid, 256, 0, stream()>>>(P, G, S, rows, R, row0, causal);
    else attn_softmax_bwd_f64<0><<<grid, 256, 0, stream()>>>(P, G, S, rows, R, row0, causal);
}

}  // namespace
}  // namespace dh

using namespace dh;

extern "C" {

int dh_gemm_f64_ex(int transA, int transB, int M, int N, int K, double alpha, const double* d_A,
                   int lda, long long strideA, const double* d_B, int ldb, long long strideB,
                   double beta, double* d_C, int ldc, long long strideC, int batch) {
    DH_TRY(ensure_init());
    DH_TRY(check_gemm_f64("dh_gemm_f64", transA, transB, M, N, K, d_A, lda, strideA, d_B, ldb,
                          strideB, d_C, ldc, strideC, batch));
    if (M == 0 || N == 0 || batch == 0) return DH_OK;
    return gemm_f64_launch(transA ? 1 : 0, transB ? 1 : 0, M, N, K, alpha, d_A, lda, strideA, d_B,
                           ldb, strideB, beta, d_C, ldc, strideC, batch);
}

int dh_gemm_f64(int transA, int transB, int M, int N, int K, const double* d_A, int lda,
                const double* d_B, int ldb, double beta, double* d_C, int ldc) {
    return dh_gemm_f64_ex(transA, transB, M, N, K, 1.0, d_A, lda, 0, d_B, ldb, 0, beta, d_C, ldc,
                          0, 1);
}

int dh_attention_f64_fwd(int BH, int S, int D, double scale, int causal, const double* d_Q,
                         const double* d_K, const double* d_V, double* d_O) {
    DH_TRY(ensure_init());
    DH_TRY(check_attn_f64("dh_attention_f64_fwd", BH, S, D));
    if (BH == 0 || S == 0 || D == 0) return DH_OK;
    if (!d_Q || !d_K || !d_V || !d_O)
        return set_error(DH_ERR_INVALID, "dh_attention_f64_fwd: null pointer");
    if (!(scale > 0.0) || !isfinite(scale))
        return set_error(DH_ERR_INVALID, "dh_attention_f64_fwd: scale must be positive and finite");
    const AttnPass ps = attn_pass(BH, S);
    const long long SD = (long long)S * D;
    const long long RS = (long long)ps.rows * S;   // scores per slice and pass
    double* P = static_cast<double*>(dh_malloc((size_t)ps.chunk * RS * sizeof(double)));
    if (!P)
        return set_error(DH_ERR_OOM, "dh_attention_f64_fwd: %d score blocks of %d x %d",
                         ps.chunk, ps.rows, S);
    int st = DH_OK;
    for (int b0 = 0; b0 < BH && st == DH_OK; b0 += ps.chunk) {
        const int nb = BH - b0 < ps.chunk ? BH - b0 : ps.chunk;
        for (int r0 = 0; r0 < S && st == DH_OK; r0 += ps.rows) {
            const int nr = S - r0 < ps.rows ? S - r0 : ps.rows;
            const long long off = (long long)b0 * SD, qoff = off + (long long)r0 * D;
            // scores of query rows r0 .. r0 + nr - 1 = Q K^T
            st = gemm_f64_launch(0, 1, nr, S, D, 1.0, d_Q + qoff, D, SD, d_K + off, D, SD, 0.0,
                                 P, S, RS, nb, causal ? F64_SCORES : F64_ALL, r0);
            if (st != DH_OK) break;
            launch_softmax(P, S, (long long)nb * nr, nr, r0, scale, causal);
            st = check_launch("dh_attention_f64_fwd");
            if (st != DH_OK) break;
            // O = P V
            st = gemm_f64_launch(0, 0, nr, D, S, 1.0, P, S, RS, d_V + off, D, SD, 0.0,
                                 d_O + qoff, D, SD, nb, causal ? F64_TO_DIAG : F64_ALL, r0);
        }
    }
    dh_free(P);   // pooled: stream order keeps the buffer alive for the queued work
    return st;
}

int dh_attention_f64_bwd(int BH, int S, int D, double scale, int causal, const double* d_Q,
                         const double* d_K, const double* d_V, const double* d_dO, double* d_dQ,
                         double* d_dK, double* d_dV, int accumulate) {
    DH_TRY(ensure_init());
    DH_TRY(check_attn_f64("dh_attention_f64_bwd", BH, S, D));
    if (BH == 0 || S == 0 || D == 0) return DH_OK;
    if (!d_Q || !d_K || !d_V || !d_dO || !d_dQ || !d_dK || !d_dV)
        return set_error(DH_ERR_INVALID, "dh_attention_f64_bwd: null pointer");
    if (!(scale > 0.0) || !isfinite(scale))
        return set_error(DH_ERR_INVALID, "dh_attention_f64_bwd: scale must be positive and finite");
    const long long SD = (long long)S * D;
    const size_t gbytes = (size_t)BH * SD * sizeof(double);
    // Shared gradient buffers (one tensor passed as several of Q, K, V) receive the sum of
    // their gradients: every product then adds into its output, after one clearing pass.
    // Buffers of their own are written by the first product that reaches them.
    const bool shared = d_dQ == d_dK || d_dQ == d_dV || d_dK == d_dV;
    const bool add = accumulate || shared;
    if (!accumulate && shared) {
        double* outs[3] = {d_dQ, d_dK, d_dV};
        for (int x = 0; x < 3; ++x) {
            bool seen = false;
            for (int y = 0; y < x; ++y) seen |= outs[y] == outs[x];
            if (!seen) DH_TRY(dh_memset(outs[x], 0, gbytes));
        }
    }
    const AttnPass ps = attn_pass(BH, S);
    const long long RS = (long long)ps.rows * S;   // scores per slice and pass
    double* P = static_cast<double*>(dh_malloc((size_t)ps.chunk * RS * sizeof(double)));
    double* G = static_cast<double*>(dh_malloc((size_t)ps.chunk * RS * sizeof(double)));
    if (!P || !G) {
        if (P) dh_free(P);
        if (G) dh_free(G);
        return set_error(DH_ERR_OOM, "dh_attention_f64_bwd: %d score blocks of %d x %d",
                         ps.chunk, ps.rows, S);
    }
    int st = DH_OK;
    for (int b0 = 0; b0 < BH && st == DH_OK; b0 += ps.chunk) {
        const int nb = BH - b0 < ps.chunk ? BH - b0 : ps.chunk;
        const long long off = (long long)b0 * SD;
        const double *Q = d_Q + off, *K = d_K + off, *V = d_V + off, *dO = d_dO + off;
        // Query rows r0 .. r0 + nr - 1 per pass (whole slices when they fit the budget).
        for (int r0 = 0; r0 < S && st == DH_OK; r0 += ps.rows) {
            const int nr = S - r0 < ps.rows ? S - r0 : ps.rows;
            const long long ro = (long long)r0 * D;
            const double beta = add || r0 > 0 ? 1.0 : 0.0;   // dV, dK: summed over the passes
            // P recomputed from Q, K exactly as the forward computes it
            st = gemm_f64_launch(0, 1, nr, S, D, 1.0, Q + ro, D, SD, K, D, SD, 0.0, P, S, RS, nb,
                                 causal ? F64_SCORES : F64_ALL, r0);
            if (st != DH_OK) break;
            launch_softmax(P, S, (long long)nb * nr, nr, r0, scale, causal);
            if ((st = check_launch("dh_attention_f64_bwd")) != DH_OK) break;
            // dV += P^T dO
            st = gemm_f64_launch(1, 0, S, D, nr, 1.0, P, S, RS, dO + ro, D, SD, beta, d_dV + off,
                                 D, SD, nb, causal ? F64_FROM_DIAG : F64_ALL, r0);
            if (st != DH_OK) break;
            // dP = dO V^T, then dS in its place
            st = gemm_f64_launch(0, 1, nr, S, D, 1.0, dO + ro, D, SD, V, D, SD, 0.0, G, S, RS, nb,
                                 causal ? F64_SCORES : F64_ALL, r0);
            if (st != DH_OK) break;
            launch_softmax_bwd(P, G, S, (long long)nb * nr, nr, r0, causal);
            if ((st = check_launch("dh_attention_f64_bwd")) != DH_OK) break;
            // dQ += scale dS K ;  dK += scale dS^T Q
            st = gemm_f64_launch(0, 0, nr, D, S, scale, G, S, RS, K, D, SD, add ? 1.0 : 0.0,
                                 d_dQ + off + ro, D, SD, nb, causal ? F64_TO_DIAG : F64_ALL, r0);
            if (st != DH_OK) break;
            st = gemm_f64_launch(1, 0, S, D, nr, scale, G, S, RS, Q + ro, D, SD, beta,
                                 d_dK + off, D, SD, nb, causal ? F64_FROM_DIAG : F64_ALL, r0);
        }
    }
    dh_free(P);
    dh_free(G);
    return st;
}

}  // extern "C"
