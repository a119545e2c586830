// sgemm_x3.hip -- fp32 GEMM on the bf16 matrix instructions, every operand
// split into three bf16 pieces (split_bf16.hpp):
// C = alpha * op(A) . op(B) (+ beta C) (+ bias) with A [m, k] or, transposed,
// [k, m] and B [k, n] (NN: Tensor::matmul, ghostflow-core/src/ops/matmul.rs:
// 91-119) or [n, k] (NT: Linear::forward, ghostflow-nn/src/linear.rs:56-69),
// all four combinations (matmul_backward's a^T . grad among them,
// ghostflow-autograd/src/backward.rs:131-160), batches with batched_matmul's
// modulo slice indexing (matmul.rs:122-170), and groups of products of one
// shape in one launch.
//
// Why: v_mfma_f32_32x32x2_f32 peaks at 157 TFLOP/s, and the fp32 tile kernels
// before this one ran 4096^3 at 0.93 of it (935 us).  Six v_mfma_f32_16x16x32
// _bf16 per 32 k do the same product: a register-only loop of them on split
// N(0, 1) data sustains 1920 TFLOP/s (320 of fp32 product; 1570 with the
// 32x32x16 form) at about 1.8 GHz, the power limit.  Measured, before -> now
// (us; NT / NN / TN): 4096^3 938 / 956 / 959 -> 604 / 608 / 623; 2048^3 NN
// 131 -> 93; 1000 x 1500 x 784 NN 42.6 -> 24.3; 64 x 11008 x 4096 NT 90 -> 56.
// Relative error against 64 bits: 4096^3 1.1e-6 -> 2.2e-7, 512 x 512 x 64
// 1.1e-7 -> 4.7e-8 (no shape of the sweep came out larger than before).
//
// Precision: a stage's six piece products (smallest first) go into an
// accumulator that starts at zero, which is then added to the running one, so
// the running sum is rounded once per 32 k where the f32 instructions round
// it 16 times.  Straight chaining of all products measured 545 us at 4096^3
// but 1.0e-6, above what split-K launches of the f32 tiles had.
//
// Design (one BM x BN tile per workgroup of 8 waves, 4 at 32 rows):
//  * Both operands pass through registers: 4 consecutive k of one row per
//    unit, requested two stages ahead, split and written to LDS one stage
//    ahead (two LDS buffers, one barrier per stage).  So any leading
//    dimension, alignment and K is served; a last stage that K cuts short
//    moves its 8-k groups down to end at K and zeroes the repeated k of A.
//  * LDS: three planes per operand, four chunks of 8 k (16 bytes) per row.
//    Row r of chunk c sits at r ^ {0, 14, 4, 10}[c] of its 16-row block:
//    conflict-free for the 16-byte fragment reads (whose 16-lane groups mix
//    two chunks) and for the 8-byte writes of a k-contiguous operand (with
//    padding between chunks instead, 89e6 conflict cycles at 4096^3 and
//    568 us against 556).
//  * The stage's splits are spread between the MFMAs (609 us with the
//    splits in one block, 573 spread, before the summing order above).
//    After the barrier the last row block's MFMAs, whose operands are in
//    registers, cover the next stage's first fragment reads.
//  * MFMA operands are swapped (B first), so a lane holds 4 consecutive
//    columns of C and stores them as one 16-byte store.
//  * 65% of all cycles are MFMA-busy at 4096^3 (1.97 GHz); wider prefetch
//    (2 and 4 stages) and a 2 x 4 wave grid measured the same.
//  * Both operands are scaled by 2^16 before they are split, so that every
//    fp32 value down to the subnormals keeps its 24 bits beside elements of
//    any size (unscaled, an element below 2^-110 lost its low bits, and rows
//    and columns of such values had to be found and redone); the sums are
//    scaled back at the end of K.  Infinities, NaN, elements of 2^112 and
//    sums of 2^96 and more are computed again on the f32 instructions
//    (sgemm_x3_kernel's end).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "split_bf16.hpp"

#pragma clang fp contract(off)

namespace gfh {
namespace {

constexpr int kBK = 32;  // k per stage: one 16x16x32 MFMA step

// Geometry of a BM x BN tile on an NWM x NWN wave grid.  A stage of an
// operand with R rows is three bf16 planes, each four chunks of 8 k: row r of
// chunk c is 16 bytes at c * kChunk(R) + 16 r.
// WIDE: leading dimensions beyond the 32-bit offsets inside a tile.
template <int BM_, int BN_, int NWM_, int NWN_, bool AK_, bool BK_, bool WIDE_ = false>
struct X3Geo {
    static constexpr int BM = BM_, BN = BN_, NWM = NWM_, NWN = NWN_;
    static constexpr bool AK = AK_, BK = BK_;  // operand k-contiguous in memory
    static constexpr bool WIDE = WIDE_;
    static constexpr int NT = 64 * NWM * NWN;
    static constexpr int WM = BM / NWM, WN = BN / NWN;
    static constexpr int FM = WM / 16, FN = WN / 16;
    static_assert(FM % 2 == 0 && FN >= 1, "row blocks alternate between two register sets");
    static constexpr int chunk(int rows) { return rows * 16; }
    static constexpr int plane(int rows) { return 4 * chunk(rows); }
    static constexpr int kABytes = 3 * plane(BM), kBBytes = 3 * plane(BN);
    static constexpr int kStage = kABytes + kBBytes;
    static constexpr int kLds = 2 * kStage;
    static_assert(kLds <= 160 * 1024, "LDS per workgroup");
    // workgroups per CU that the LDS leaves room for, and the register bound
    // that lets all of them in
    static constexpr int kPerCu = (160 * 1024) / kLds;
    static constexpr int kWavesPerSimd = std::max(1, kPerCu * NT / 256);
};

struct X3Params {
    // the products of one launch: a batch (slices of product 0, indexed
    // modulo batch_a / batch_b) or a group of separate ones
    const float *a[kNtMaxGroups], *b[kNtMaxGroups];
    float *c[kNtMaxGroups];
    const float *bias[kNtMaxGroups];
    int64_t ldc[kNtMaxGroups];
    int64_t m, n, k, lda, ldb;
    int64_t stride_a, stride_b, stride_c;
    int batch_a, batch_b;
    int count;  // products
    bool grouped;
    float alpha, beta;
    int tiles_m, tiles_n;
    int slices, kslice;  // split K: slice z covers stages [z kslice, (z + 1) kslice)
    float *part;
    int *counters;
};

// Row r of chunk c sits at r ^ swz(c) of its 16-row block.
__device__ __forceinline__ constexpr int swz(int c) { return (c & 1 ? 14 : 0) ^ (c & 2 ? 4 : 0); }

// One operand's share of a stage in registers.
template <int R, int NT, bool KC, bool WIDE>
struct X3Loader {
    using Off = std::conditional_t<WIDE, uint64_t, uint32_t>;
    // A unit is 4 consecutive k of one row: one 16-byte load of a k-contiguous
    // operand (8 lanes cover a row's stage, 128 bytes), four 4-byte loads of a
    // k-major one (64 lanes on adjacent rows).
    static constexpr int F = 4;
    static constexpr int U = R * (kBK / F) / NT;
    static_assert(U >= 1 && U * NT * F == R * kBK, "whole units per thread");
    float v[U][F];
    Off off[U];   // byte offset of the unit, from one stage before the one it is loaded from
    uint32_t at;  // where unit 0's pieces go in a plane

    // Unit u lies kRows rows (k-contiguous) or kChunks chunks of 8 k (k-major)
    // after unit u - 1.
    static constexpr int kRows = NT / 8, kChunks = NT / (2 * R);
    static_assert(KC ? kRows % 16 == 0 : U == 1 || ((kChunks & (kChunks - 1)) == 0 && kChunks > 0),
                  "unit 0's address serves all units");

    // first k of unit id inside a stage
    static __device__ __forceinline__ int first_k(int id) { return KC ? 4 * (id % 8) : F * (id / R); }
    __device__ __forceinline__ void init(int tid, int64_t ld, int64_t row0, int64_t rows) {
        const int r0 = KC ? tid / 8 : tid % R, c0 = first_k(tid) / 8;
        at = (uint32_t)(c0 * R * 16 + (r0 ^ swz(c0)) * 16 + (first_k(tid) & 4) * 2);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int id = tid + u * NT;
            if (KC) {
                const int64_t r = min((int64_t)(id / 8), rows - 1 - row0);
                off[u] = (Off)((r * ld + first_k(id) + kBK) * 4);
            } else {
                const int64_t r = min((int64_t)(id % R), rows - 1 - row0);
                off[u] = (Off)(((first_k(id) + kBK) * ld + r) * 4);
            }
        }
    }
    // k positions the 8-k group at k is moved down by in a last stage with
    // `left` < 32 k, so that it ends at K (the moved group repeats earlier k:
    // keep() drops those from one operand)
    static __device__ __forceinline__ int moved(int k, int left) { return max(0, (k & ~7) + 8 - left); }
    // Moves the offsets for that stage.  (tid through an empty asm: what these
    // two rare steps need is not kept in registers over the whole loop.)
    __device__ __forceinline__ void move_down(int tid, int64_t ld, int left) {
        asm volatile("" : "+v"(tid));
#pragma unroll
        for (int u = 0; u < U; ++u) off[u] -= (Off)(moved(first_k(tid + u * NT), left) * (KC ? 1 : ld) * 4);
    }
    // Requests unit u of a stage.  `base` is one stage before it (k-contiguous:
    // the tile's first row at that k; k-major: that k row), so that the
    // offsets stay unsigned when the last stage moves down.
    // (Buffer loads: a uniform base and row offset in scalar registers, the
    // lane's offset in one vector register.)
    __device__ __forceinline__ void load(int u, const char *base, int64_t ld) {
        if constexpr (WIDE) {
            typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
            const float *from = reinterpret_cast<const float *>(base + off[u]);
            if constexpr (KC) {
                const f32x4 x = *reinterpret_cast<const f32x4_any *>(from);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[u][e] = x[e];
            } else {
#pragma unroll
                for (int e = 0; e < F; ++e) v[u][e] = from[e * ld];
            }
            return;
        }
        const __amdgpu_buffer_rsrc_t buf = coherent_buffer(base, 0xffffffffu);
        if constexpr (KC) {
            const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buf, (int)off[u], 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[u][e] = x[e];
        } else {
#pragma unroll
            for (int e = 0; e < F; ++e)
                v[u][e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(buf, (int)off[u], e * (int)ld * 4, 0));
        }
    }
    // Zeroes what load() repeated in that stage.
    __device__ __forceinline__ void keep(int tid, int left) {
        asm volatile("" : "+v"(tid));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = first_k(tid + u * NT);
            const int drop = moved(k, left) - (k & 7);  // leading floats of the unit
#pragma unroll
            for (int e = 0; e < F; ++e) v[u][e] = e < drop ? 0.f : v[u][e];
        }
    }
    __device__ __forceinline__ void store(int u, char *planes) {
        constexpr int CH = R * 16, PL = 4 * CH;
        uint32_t p[3][F / 2];
#pragma unroll
        for (int e = 0; e < F; e += 2)
            split2(v[u][e] * kPieceUp, v[u][e + 1] * kPieceUp, p[0][e / 2], p[1][e / 2], p[2][e / 2]);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            // (k-major: unit 0's chunk is below kChunks, so the chunk bits and
            // with them the XORs of both combine)
            char *dst = KC ? planes + at + u * kRows * 16 : planes + (at ^ (swz(u * kChunks) * 16)) + u * kChunks * CH;
            *reinterpret_cast<uint2 *>(dst + q * PL) = make_uint2(p[q][0], p[q][1]);
        }
    }
};

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// NM MFMAs with NV VALU instructions, ND LDS reads, NW LDS writes and NL
// global loads spread between them.
template <int NL, int NV, int ND, int NW, int NM, int I = 0>
__device__ __forceinline__ void mix() {
    if constexpr (I < NM) {
        constexpr int l = (I + 1) * NL / NM - I * NL / NM, v = (I + 1) * NV / NM - I * NV / NM;
        constexpr int d = (I + 1) * ND / NM - I * ND / NM, w = (I + 1) * NW / NM - I * NW / NM;
        if constexpr (d > 0) __builtin_amdgcn_sched_group_barrier(0x100, d, 0);
        if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x002, v, 0);
        if constexpr (w > 0) __builtin_amdgcn_sched_group_barrier(0x200, w, 0);
        if constexpr (l > 0) __builtin_amdgcn_sched_group_barrier(0x020, l, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        mix<NL, NV, ND, NW, NM, I + 1>();
    }
}

template <int N, int I = 0, class F>
__device__ __forceinline__ void unrolled(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<N, I + 1>(f);
    }
}

template <class G>
__global__ __launch_bounds__(G::NT, G::kWavesPerSimd) void sgemm_x3_kernel(X3Params p) {
    constexpr int BM = G::BM, BN = G::BN, FM = G::FM, FN = G::FN, NT = G::NT;
    constexpr int CHA = G::chunk(BM), CHB = G::chunk(BN), PLA = G::plane(BM), PLB = G::plane(BN);
    // (two arrays: the compiler then knows that splitting into one does not
    // touch the fragments read from the other)
    __shared__ __attribute__((aligned(1024))) char lds0[G::kStage];
    __shared__ __attribute__((aligned(1024))) char lds1[G::kStage];
    auto ring = [&](int buf) __attribute__((always_inline)) { return buf ? lds1 : lds0; };
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm0 = (wave / G::NWN) * G::WM, wn0 = (wave % G::NWN) * G::WN;

    // workgroup -> (K slice, product, tile)
    const int nblk = p.tiles_m * p.tiles_n;
    int bid = xcd_chunked(blockIdx.x, gridDim.x);
    const int outer = bid / nblk;
    bid -= outer * nblk;
    const int slice = outer / p.count, prod = outer - slice * p.count;
    const int slot = prod * nblk + bid;  // this tile among all products' tiles
    constexpr int kGroupM = 4;
    const int group_size = kGroupM * p.tiles_n;
    const int group = bid / group_size;
    const int first_m = group * kGroupM;
    const int gm = min(p.tiles_m - first_m, kGroupM);
    const int in_group = bid - group * group_size;
    const int64_t m0 = (int64_t)(first_m + in_group % gm) * BM;
    const int64_t n0 = (int64_t)(in_group / gm) * BN;
    const int g = p.grouped ? prod : 0, bz = p.grouped ? 0 : prod;
    const float *pa = p.a[g] + (bz % p.batch_a) * p.stride_a;
    const float *pb = p.b[g] + (bz % p.batch_b) * p.stride_b;
    float *pc = p.c[g] + bz * p.stride_c;
    const float *bias = p.bias[g];
    const int64_t ldc = p.ldc[g];

    const int64_t k_lo = (int64_t)slice * p.kslice * kBK;
    const int64_t k_hi = min(p.k, k_lo + (int64_t)p.kslice * kBK);
    const int nk = (int)((k_hi - k_lo + kBK - 1) / kBK);
    const char *a_base = reinterpret_cast<const char *>(G::AK ? pa + m0 * p.lda + k_lo : pa + k_lo * p.lda + m0);
    const char *b_base = reinterpret_cast<const char *>(G::BK ? pb + n0 * p.ldb + k_lo : pb + k_lo * p.ldb + n0);
    // (the loads' bases, one stage early)
    const int64_t a_step = G::AK ? kBK * 4 : kBK * 4 * p.lda, b_step = G::BK ? kBK * 4 : kBK * 4 * p.ldb;
    a_base -= a_step;
    b_base -= b_step;

    X3Loader<BM, NT, G::AK, G::WIDE> ga;
    X3Loader<BN, NT, G::BK, G::WIDE> gb;
    ga.init(tid, p.lda, m0, p.m);
    gb.init(tid, p.ldb, n0, p.n);
    constexpr int UA = decltype(ga)::U, UB = decltype(gb)::U;
    auto left_of = [&](int t) __attribute__((always_inline)) { return (int)(p.k - k_lo) - t * kBK; };
    const int left_last = left_of(nk - 1);  // < 32: the last stage is cut short
    auto load = [&](int t) __attribute__((always_inline)) {
        const int64_t tt = min(t, nk - 1);
#pragma unroll
        for (int u = 0; u < UA; ++u) ga.load(u, a_base + tt * a_step, p.lda);
#pragma unroll
        for (int u = 0; u < UB; ++u) gb.load(u, b_base + tt * b_step, p.ldb);
    };
    // before stage t is loaded / split: a last stage that is cut short
    auto before_load = [&](int t) __attribute__((always_inline)) {
        if (t == nk - 1 && left_last < kBK) {
            ga.move_down(tid, p.lda, left_last);
            gb.move_down(tid, p.ldb, left_last);
        }
    };
    auto before_store = [&](int t) __attribute__((always_inline)) {
        if (t == nk - 1 && left_last < kBK) ga.keep(tid, left_last);
    };

    bf16x8 af[2][3], bf[2][FN][3];
    const int fo_a = (lane >> 4) * CHA + (wm0 + ((lane & 15) ^ swz(lane >> 4))) * 16;
    const int fo_b = (lane >> 4) * CHB + (wn0 + ((lane & 15) ^ swz(lane >> 4))) * 16;
    auto read_a = [&](int set, int buf, int i) __attribute__((always_inline)) {
        const char *s = ring(buf) + fo_a + i * 256;
#pragma unroll
        for (int q = 0; q < 3; ++q) af[set][q] = *reinterpret_cast<const bf16x8 *>(s + q * PLA);
    };
    auto read_b = [&](int set, int buf) __attribute__((always_inline)) {
        const char *s = ring(buf) + G::kABytes + fo_b;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 3; ++q) bf[set][j][q] = *reinterpret_cast<const bf16x8 *>(s + q * PLB + j * 256);
    };
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Product s of the six of row block i, smallest first, into a sum of the
    // stage's own.  Each sum is added to its accumulators while the next row
    // block's products run (the last block's in the next stage): with four or
    // more column blocks one after another as the next products take their
    // place, which needs one set of registers, and otherwise from a second set
    // after the third product, so that no add waits for its MFMA.
    constexpr int SB = FN >= 4 ? 1 : 2;
    f32x4 sum[SB][FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) sum[SB - 1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto add_sum = [&](int i, int j) __attribute__((always_inline)) { acc[i][j] = acc[i][j] + sum[i % SB][j]; };
    auto step = [&](int i, int s, int aset, int bset) __attribute__((always_inline)) {
        constexpr int P[6] = {2, 1, 0, 1, 0, 0}, Q[6] = {0, 1, 2, 0, 1, 0};
        const int before = i == 0 ? FM - 1 : i - 1;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            if (SB == 1 && s == 0) add_sum(before, j);
            sum[i % SB][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                bf[bset][j][Q[s]], af[aset][P[s]], s == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sum[i % SB][j], 0, 0, 0);
        }
        if (SB == 2 && s == 2) {
#pragma unroll
            for (int j = 0; j < FN; ++j) add_sum(before, j);
        }
    };

    before_load(0);
    load(0);
    before_store(0);
#pragma unroll
    for (int u = 0; u < UA; ++u) ga.store(u, ring(0));
#pragma unroll
    for (int u = 0; u < UB; ++u) gb.store(u, ring(0) + G::kABytes);
    if (nk > 1) {
        before_load(1);
        load(1);
    }
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
    read_b(0, 0);
    read_a(0, 0, 0);
    auto stage = [&](int t, auto par) __attribute__((always_inline)) {
        constexpr int P = decltype(par)::value;
        before_store(t + 1);
        before_load(t + 2);
        __builtin_amdgcn_sched_barrier(0);
        // product steps of row blocks 0 .. FM - 2, with the next stage's
        // units split (and the one after's requested) in between
        constexpr int NU = UA + UB;
        const int64_t tt = min(t + 2, nk - 1);
        const char *a_next = a_base + tt * a_step, *b_next = b_base + tt * b_step;
        unrolled<FM - 1>([&](auto rc) __attribute__((always_inline)) {
            constexpr int r = decltype(rc)::value;
            constexpr int u0 = r * NU / (FM - 1), n = (r + 1) * NU / (FM - 1) - u0;  // this row's units
            read_a((r + 1) & 1, P, r + 1);
            unrolled<n == 0 ? 1 : n>([&](auto pc) __attribute__((always_inline)) {
                constexpr int i = decltype(pc)::value, pieces = n == 0 ? 1 : n, u = u0 + i;
                constexpr int s0 = i * 6 / pieces, s1 = (i + 1) * 6 / pieces;
#pragma unroll
                for (int s = s0; s < s1; ++s) step(r, s, r & 1, P);
                constexpr bool isa = u < UA;
                if constexpr (n > 0 && isa) {
                    ga.store(u, ring(P ^ 1));
                    ga.load(u, a_next, p.lda);
                } else if constexpr (n > 0) {
                    gb.store(u - UA, ring(P ^ 1) + G::kABytes);
                    gb.load(u - UA, b_next, p.ldb);
                }
                if constexpr (SB == 1 && i == 0) mix<0, 4 * FN, 0, 0, FN>();
                mix<n == 0 ? 0 : (isa ? G::AK : G::BK) ? 1 : 4, n == 0 ? 0 : 26 + (SB == 2 ? 4 * FN / pieces : 0),
                    i == 0 ? 3 : 0, n == 0 ? 0 : 3, (s1 - s0 - (SB == 1 && i == 0 ? 1 : 0)) * FN>();
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        wait_lgkm0();
        __builtin_amdgcn_s_barrier();
        read_b(P ^ 1, P ^ 1);
        read_a(0, P ^ 1, 0);
#pragma unroll
        for (int s = 0; s < 6; ++s) step(FM - 1, s, (FM - 1) & 1, P);
        if constexpr (SB == 1) mix<0, 4 * FN, 0, 0, FN>();
        mix<0, 0, 3 + 3 * FN, 0, (SB == 1 ? 5 : 6) * FN>();
        __builtin_amdgcn_sched_barrier(0);
        // The stage's adds stay in the stage: left to itself the compiler
        // moves them into the blocks after the next branch, past the
        // scheduling barriers, and every row block's sums stay in registers
        // until then (256 and 26 to 44 spilled, 1027 us at 4096^3; with this
        // and the loop in pairs 226 to 246 and none).
#pragma unroll
        for (int i = 0; i + 1 < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                f32x4 &x = acc[i][j];
                asm volatile("" : "+v"(x));
            }
    };
    // The last stage has nothing to split, request or wait for.  (As a stage
    // like the others it split and loaded itself once more: NN 64 x 64 x
    // 3000000 483 us instead of 406, 96 x [500, 64] x [64, 500] 41.1 instead
    // of 38.9, 4096^3 618 instead of 604.)
    auto last = [&](auto par) __attribute__((always_inline)) {
        constexpr int P = decltype(par)::value;
        unrolled<FM>([&](auto rc) __attribute__((always_inline)) {
            constexpr int r = decltype(rc)::value;
            if constexpr (r + 1 < FM) read_a((r + 1) & 1, P, r + 1);
#pragma unroll
            for (int s = 0; s < 6; ++s) step(r, s, r & 1, P);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    int t = 0;
    for (; t + 2 < nk; t += 2) {
        stage(t, Even{});
        stage(t + 1, Odd{});
    }
    if (t + 1 < nk) {
        stage(t, Even{});
        last(Odd{});
    } else {
        last(Even{});
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) add_sum(FM - 1, j);

    // Values the pieces cannot carry: an infinity splits into inf and NaN, an
    // element of 2^112 or a sum of 2^96 becomes inf scaled.  Where a sum is
    // not finite the tile is computed again on the f32 matrix instructions,
    // straight from memory (4096^3 NN 671 us, with an infinity in one row of
    // A 2590, in every tile 2680; NT 639, 4077, 4123).
    {
        int odd = 0;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) odd |= !(fabsf(acc[i][j][r]) <= 3.402823466e38f);
        if (__syncthreads_or(odd)) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int64_t k = k_lo; k < k_hi; k += 4) {
                const int64_t kk = k + (lane >> 4);
                const bool in = kk < k_hi;
                float a[FM], b[FN];
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    const int64_t r = min(m0 + wm0 + i * 16 + (lane & 15), p.m - 1);
                    a[i] = in ? pa[G::AK ? r * p.lda + kk : kk * p.lda + r] : 0.f;
                }
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    const int64_t r = min(n0 + wn0 + j * 16 + (lane & 15), p.n - 1);
                    b[j] = in ? pb[G::BK ? r * p.ldb + kk : kk * p.ldb + r] : 0.f;
                }
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j], a[i], acc[i][j], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = acc[i][j] * kPieceDown;
        }
    }

    if (p.slices > 1) {
        constexpr int R4 = FM * FN;
        const uint32_t part_bytes = (uint32_t)((int64_t)p.slices * p.count * nblk * R4 * NT * 16);
        const __amdgpu_buffer_rsrc_t part_buf = coherent_buffer(p.part, part_bytes);
        auto part_off = [&](int sl, int q) { return (uint32_t)((((int64_t)sl * p.count * nblk + slot) * R4 + q) * NT + tid) * 16; };
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, acc[i][j]), part_buf,
                                                       part_off(slice, i * FN + j), 0, kScDevice);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        wait_vmcnt<0>();
        __syncthreads();
        int *last_flag = reinterpret_cast<int *>(lds0);
        if (tid == 0)
            *last_flag =
                __hip_atomic_fetch_add(p.counters + slot, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.slices - 1;
        __syncthreads();
        if (!*last_flag) return;
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        constexpr int GS = 8;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                f32x4 tot = {0.f, 0.f, 0.f, 0.f};
                for (int s0 = 0; s0 < p.slices; s0 += GS) {
                    i32x4 t[GS];
#pragma unroll
                    for (int g = 0; g < GS; ++g)
                        t[g] = s0 + g < p.slices
                                   ? __builtin_amdgcn_raw_buffer_load_b128(part_buf, part_off(s0 + g, i * FN + j), 0, kScDevice)
                                   : i32x4{0, 0, 0, 0};
#pragma unroll
                    for (int g = 0; g < GS; ++g) {
                        const f32x4 v = __builtin_bit_cast(f32x4, t[g]);
                        if (s0 + g == 0)
                            tot = v;
                        else if (s0 + g < p.slices)
                            tot = tot + v;
                    }
                }
                acc[i][j] = tot;
            }
        if (tid == 0) __hip_atomic_store(p.counters + slot, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // Epilogue: lane l holds row l % 16 of block i and columns 4 (l / 16) ..
    // + 3 of block j.
    const bool vec_out = (ldc % 4) == 0 && (reinterpret_cast<uintptr_t>(pc) & 15) == 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int64_t r = m0 + wm0 + i * 16 + (lane & 15);
        if (r >= p.m) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t col = n0 + wn0 + j * 16 + 4 * (lane >> 4);
            float *dst = pc + r * ldc + col;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = p.alpha * acc[i][j][e];
            if (vec_out && col + 3 < p.n) {
                if (p.beta != 0.f) {
                    const f32x4 c0 = *reinterpret_cast<const f32x4 *>(dst);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = v[e] + p.beta * c0[e];
                }
                if (bias) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = v[e] + bias[col + e];
                }
                *reinterpret_cast<f32x4 *>(dst) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (col + e >= p.n) continue;
                    float x = v[e];
                    if (p.beta != 0.f) x = x + p.beta * dst[e];
                    if (bias) x = x + bias[col + e];
                    dst[e] = x;
                }
            }
        }
    }
}

// Tiles and what they take (us): a stage of 32 k where a workgroup has its CU
// to itself, the same per workgroup of a filled GPU (less where several share
// a CU and hide each other's latency; more at 256x128 and 128x128, one per CU,
// where the matrix units then run at the power limit), a tile's prologue and
// stores; and how many of its workgroups share a CU.  Fitted to 4096^3,
// 2048^3 and 110 products of 33-3000 rows, K 64-11008, N 128-11008 timed on
// every tile and split: the choice is on average 1.1% slower than the fastest
// of them.  (With every workgroup counted as a CU's only one, and without the
// last arriver's reads below, 2.9%: 337 x 1152 x 1024 NN 22.5 us for 16.1,
// 72 x 1702 x 3554 28.4 for 20.8.)
struct X3Tile {
    int bm, bn, per_cu;
    double alone, full, ends;
    constexpr int threads() const { return bm == 32 ? 256 : 512; }
    int64_t tiles(const SgemmDesc &d, int64_t count) const {
        return ((d.m + bm - 1) / bm) * ((d.n + bn - 1) / bn) * count;
    }
};
constexpr X3Tile kTiles[] = {{256, 128, 1, 1.75, 2.20, 4.5},
                             {128, 128, 1, 1.00, 1.32, 2.2},
                             {128, 64, 2, 0.64, 0.71, 1.1},
                             {64, 64, 3, 0.48, 0.44, 0.5},
                             {32, 64, 4, 0.44, 0.30, 0.3}};

// Tile I of the table on an NWM x NWN wave grid, in the layout of d.
template <int I, int NWM, int NWN, bool WIDE = false>
void launch_tile(const SgemmDesc &d, const X3Params &p, dim3 grid, hipStream_t s) {
    constexpr int BM = kTiles[I].bm, BN = kTiles[I].bn;
    static_assert(X3Geo<BM, BN, NWM, NWN, true, true>::kPerCu == kTiles[I].per_cu &&
                      64 * NWM * NWN == kTiles[I].threads(),
                  "the plan's figures are the kernel's");
    auto go = [&](auto ak, auto bk) {
        hipLaunchKernelGGL((sgemm_x3_kernel<X3Geo<BM, BN, NWM, NWN, decltype(ak)::value, decltype(bk)::value, WIDE>>), grid,
                           dim3(64 * NWM * NWN), 0, s, p);
    };
    using Y = std::true_type;
    using N = std::false_type;
    if (d.trans_a)
        d.trans_b ? go(N{}, Y{}) : go(N{}, N{});
    else
        d.trans_b ? go(Y{}, Y{}) : go(Y{}, N{});
}

struct X3Plan {
    int tile;  // index into kTiles
    int slices;
};

// Whether the offsets inside a tile fit 32 bits: up to 256 rows of a
// k-contiguous operand, 32 k and the stage before of a k-major one (and the
// three k that the loads' scalar offsets add).
bool x3_offsets_fit(const SgemmDesc &d) {
    constexpr int64_t kRows = (int64_t)1 << 22, kMajor = (int64_t)1 << 23;
    return d.lda <= (d.trans_a ? kMajor : kRows) && d.ldb <= (d.trans_b ? kRows : kMajor);
}
constexpr int kWideTile = 3;  // 64-bit offsets: one tile size

// Work items of a launch: 32 bits.
bool x3_grid_fits(const X3Tile &t, int64_t workgroups) { return workgroups * t.threads() < (int64_t)1 << 32; }

// The tile and K split with the shortest estimated time for `count` products
// of one shape: workgroups in rounds of per_cu on every CU.  K slices add the
// partial tiles' stores, at 6 TB/s, and the last arriver's reads of a tile's
// partials, which one workgroup takes in at 100 GB/s.  The operands arrive no
// faster than 5 TB/s, nor than the resident workgroups' two requested stages
// per 3 us: with few rows one workgroup per CU keeps too little in flight (NT
// 33 x 4096 x 4096 in 4 slices 30.1 us, in 8 26.3; of 85 products of 33-1500
// rows whose operands lie beyond the MALL the choice is 3.6% slower than the
// fastest on average and 28% at worst, 4.2% without this, and up to 128 rows
// 2.4 for 3.9).  (A batch splits like a
// group: a few slices of a long K otherwise leave most CUs idle, 2 x [4096,
// 4096] x [4096, 64] 84 us, split 44; 29 batches of 2-64 with K 281-7981:
// 20% less time over all, none more than 2% slower.)
X3Plan plan_x3(const SgemmDesc &d, int64_t count) {
    const int64_t stages = (d.k + kBK - 1) / kBK, cus = device_cu_count();
    const bool wide = !x3_offsets_fit(d);
    const double operands = 4.0 * (double)d.k * (double)(d.m + d.n) * (double)count;
    X3Plan best{0, 1};
    double least = 1e30;
    for (int i = 0; i < (int)(sizeof kTiles / sizeof kTiles[0]); ++i) {
        const X3Tile &t = kTiles[i];
        const int64_t tiles = t.tiles(d, count);
        if (!x3_grid_fits(t, tiles) || (wide && i != kWideTile)) continue;
        const int64_t round = t.per_cu * cus;
        for (int sl = 1; sl <= 256; sl += sl < 16 ? 1 : sl / 4) {
            const double one = (double)t.bm * t.bn * 4, part = (double)sl * (double)tiles * one;
            if (sl > 1 && (stages / sl < 4 || part > 64e6)) break;
            const int64_t tasks = tiles * sl, rem = tasks % round;
            const double st = (double)((stages + sl - 1) / sl);
            auto shared = [&](double n) { return std::max(st * t.alone, n * st * t.full) + n * t.ends; };
            double us = (double)(tasks / round) * shared(t.per_cu);
            if (rem) us += 4 * rem <= 3 * cus ? st * t.alone + t.ends : shared((double)((rem + cus - 1) / cus));
            const double flight = (double)std::min(tasks, round) * 2 * (t.bm + t.bn) * kBK * 4;
            us = std::max(us, operands / std::min(5e6, flight / 3));
            if (sl > 1) us += 2.5 + part / 6e6 + sl * one / 1e5;
            if (us < least) {
                least = us;
                best = {i, sl};
            }
        }
    }
    return best;
}

bool x3_takes(const SgemmDesc &d, int64_t count) {
    const X3Tile &t = kTiles[x3_offsets_fit(d) ? 0 : kWideTile];
    return d.k >= 32 && d.k <= (int64_t)1 << 30 && d.m >= 1 && d.n >= 1 && x3_grid_fits(t, t.tiles(d, count));
}

// d[0] gives the shape and layout of all products.
int launch_products(const SgemmDesc *d, X3Params &p, hipStream_t s) {
    p.m = d->m;
    p.n = d->n;
    p.k = d->k;
    p.lda = d->lda;
    p.ldb = d->ldb;
    p.alpha = d->alpha;
    p.beta = d->beta;
    const X3Plan plan = plan_x3(*d, p.count);
    const X3Tile &t = kTiles[plan.tile];
    p.tiles_m = (int)((d->m + t.bm - 1) / t.bm);
    p.tiles_n = (int)((d->n + t.bn - 1) / t.bn);
    const int64_t nblk = (int64_t)p.tiles_m * p.tiles_n * p.count, stages = (d->k + kBK - 1) / kBK;
    p.kslice = (int)((stages + plan.slices - 1) / plan.slices);
    p.slices = (int)((stages + p.kslice - 1) / p.kslice);
    if (p.slices > 1) {
        // one partial tile per slice
        void *ws = nullptr;
        GFH_TRY(stream_workspace(s, sizeof(float) * (size_t)(p.slices * nblk) * t.bm * t.bn, &ws));
        p.part = static_cast<float *>(ws);
        GFH_TRY(stream_counters(s, (size_t)nblk, &p.counters));
    }
    const dim3 grid((unsigned)(nblk * p.slices));
    switch (plan.tile) {
        case 0: launch_tile<0, 4, 2>(*d, p, grid, s); break;
        case 1: launch_tile<1, 2, 4>(*d, p, grid, s); break;
        case 2: launch_tile<2, 4, 2>(*d, p, grid, s); break;
        case 3:
            if (x3_offsets_fit(*d))
                launch_tile<3, 2, 4>(*d, p, grid, s);
            else
                launch_tile<3, 2, 4, true>(*d, p, grid, s);
            break;
        default: launch_tile<4, 1, 4>(*d, p, grid, s); break;
    }
    return check_launch("sgemm (bf16 pieces)");
}

}  // namespace

// Whether this kernel takes the product.  K >= 32: below that the fp32 chain
// is short enough for its rounding to be smaller than the pieces'.  The
// number of threads of the launch is 32-bit: from 2^29 rows on the smaller
// tiles drop out (128 x 64 has four threads a row), at 2^31 the largest.
bool sgemm_x3_fits(const SgemmDesc &d) { return x3_takes(d, std::max<int64_t>(d.batch, 1)); }

int launch_sgemm_x3(const SgemmDesc &d, hipStream_t s) {
    X3Params p{};
    p.a[0] = d.a;
    p.b[0] = d.b;
    p.c[0] = d.c;
    p.bias[0] = d.bias;
    p.ldc[0] = d.ldc;
    p.stride_a = d.stride_a;
    p.stride_b = d.stride_b;
    p.stride_c = d.stride_c;
    // (a slice count above the batch indexes like the batch itself)
    const int64_t nb = std::max<int64_t>(d.batch, 1);
    p.batch_a = (int)std::min(std::max<int64_t>(d.batch_a, 1), nb);
    p.batch_b = (int)std::min(std::max<int64_t>(d.batch_b, 1), nb);
    p.count = (int)nb;
    return launch_products(&d, p, s);
}

bool sgemm_x3_group_fits(const SgemmDesc *d, int count) {
    if (count < 1 || count > kNtMaxGroups) return false;
    for (int g = 0; g < count; ++g) {
        const SgemmDesc &e = d[g];
        if (!x3_takes(e, count) || e.batch > 1 || e.batch_a > 1 || e.batch_b > 1 || e.trans_a != d[0].trans_a ||
            e.trans_b != d[0].trans_b || e.m != d[0].m || e.n != d[0].n || e.k != d[0].k || e.lda != d[0].lda ||
            e.ldb != d[0].ldb || e.alpha != d[0].alpha || e.beta != d[0].beta)
            return false;
    }
    return true;
}

int launch_sgemm_x3_group(const SgemmDesc *d, int count, hipStream_t s) {
    X3Params p{};
    for (int g = 0; g < count; ++g) {
        p.a[g] = d[g].a;
        p.b[g] = d[g].b;
        p.c[g] = d[g].c;
        p.bias[g] = d[g].bias;
        p.ldc[g] = d[g].ldc;
    }
    p.batch_a = p.batch_b = 1;
    p.count = count;
    p.grouped = count > 1;
    return launch_products(d, p, s);
}

}  // namespace gfh

// What the plan gives an [m, k] x [k, n] product: out = {tile rows, tile
// columns, K slices, threads of the launch}; returns 0 where the kernel does
// not take it.  Not part of the API: it lets the tests say which tile a shape
// runs on, without a GPU.
extern "C" __attribute__((visibility("default"))) int gfh_internal_sgemm_x3_plan(int trans_a, int trans_b, int64_t m,
                                                                                 int64_t n, int64_t k, int64_t batch,
                                                                                 int64_t *out) {
    gfh::SgemmDesc d;
    d.trans_a = trans_a != 0;
    d.trans_b = trans_b != 0;
    d.m = m;
    d.n = n;
    d.k = k;
    d.lda = trans_a ? m : k;
    d.ldb = trans_b ? k : n;
    d.batch = batch;
    if (!gfh::sgemm_x3_fits(d)) return 0;
    const gfh::X3Plan plan = gfh::plan_x3(d, batch);
    const gfh::X3Tile &t = gfh::kTiles[plan.tile];
    out[0] = t.bm;
    out[1] = t.bn;
    out[2] = plan.slices;
    out[3] = t.tiles(d, batch) * plan.slices * t.threads();
    return 1;
}
