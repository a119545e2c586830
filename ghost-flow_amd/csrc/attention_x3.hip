// attention_x3.hip -- scaled-dot-product attention with both products on the
// bf16 matrix units, every operand as three bf16 pieces (split_bf16.hpp).
//
// softmax(mask(Q K^T * scale)) V per (batch, head), online over 32-key tiles;
// semantics as listed in attention.hip.  fp32 in, fp32 out, fp32 sums: an
// f32 MFMA does 1/16 of the bf16 rate, a product of pieces takes six bf16
// MFMAs, and the six together are closer to the exact product than one chain
// of f32 MFMAs (64-bit comparison, B = 4, H = 32, S = 1000, D = 128 causal:
// 3.9e-7 -> 2.4e-7 of the norm; weights 2.1e-7 -> 1.0e-7).
//
// Layout: eight waves per workgroup, SETS sets of 16 queries per wave.
//  * S^T = K . Q^T on 16x16x32: lane (c = l % 16, h = l / 16) holds keys
//    16 kb + 4 h + r of query c, so the softmax is per lane plus two
//    cross-quarter swaps, and a tile's eight probabilities of a lane are
//    exactly its B operand of O^T = V^T . P^T when the A operand takes the
//    32 keys in the order chunk h = (4h .. 4h + 3, 16 + 4h .. 16 + 4h + 3):
//    P never moves between lanes.  V is staged in that order.
//  * K and V tiles go through registers (buffer loads two tiles ahead, zero
//    past the last key), are split there and stored as three planes; the
//    XOR of the row with its chunk keeps both the 8-byte stores and the
//    16-byte fragment reads on distinct banks.
//  * K has two buffers and V three: waves 4 .. 7 take a tile's P.V one
//    iteration later, so that the softmax (VALU) of one wave of a SIMD meets
//    the products (MFMA) of the other instead of its softmax.
//
// What bounds it: the six-fold products (3.1 TFLOP of pieces per 1e9 scores at
// D = 128) and, between them, the softmax and splitting each tile of K and V,
// which every workgroup repeats for its own queries: B = 4, H = 32, D = 128
// causal the MFMAs are busy 30 / 36 / 50% of the cycles at S = 512 / 1000 /
// 2048, VALU issue takes another 25% at S = 1000.  us on f32 MFMAs -> here, B =
// 4, H = 32: D = 128 causal S = 512 92 -> 74, 1000 303 -> 200, 2048 1143 -> 705,
// not causal 1000 540 -> 316; D = 64 causal 165 -> 103; with weights and a mask
// B = 4, H = 16, S = 512, D = 64 201 -> 57.  The two-set forms of D = 128 spill
// 2 to 26 registers.
//
// V and the probabilities are scaled by 2^16 before they are split (and the
// sums scaled back), so that small ones keep their 24 bits: a weight of 2^-120
// can be the output where V is zero at the larger ones.  Q and K need no
// scale, as a score enters by its absolute size: their lost bits move it by
// less than 2^-134 2^60 2^20 d (the bounds below), nothing.
//
// Inputs beyond the pieces: a workgroup that meets an element of Q, K or V
// that is not finite or above 2^60, or a scale above 2^20, and a wave whose
// result is not finite redo their queries on f32 MFMAs (set_f32).
// (Bounds of buffers: the loads of a tile's last keys rely on a raw buffer
// load returning zero where voffset + soffset passes num_records.)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "split_bf16.hpp"

#pragma clang fp contract(off)

namespace gfh {
namespace {

constexpr int kKeys = 32;      // keys per tile: one 16x16x32 MFMA step of P.V
constexpr int kWaves = 8;     // per workgroup; kFewWaves for launches of few queries
constexpr int kFewWaves = 4;

struct X3Attn {
    const float *q, *k, *v;
    float *out;
    float *weights;
    const float *mask;
    int64_t mask_numel;
    int64_t q_bs, q_hs, q_rs, kv_bs, kv_hs, kv_rs, o_bs, o_hs, o_rs;
    int64_t h;
    int sq, skv, d;
    int off;  // causal keeps key j for query i when j <= i + off
    float scale;
    bool mask_rows;  // mask_numel is a multiple of skv
    bool mask_vec;   // and its rows are 16-byte aligned
    bool w_vec;      // rows of weights are 16-byte aligned
};

__device__ __forceinline__ int swz(int c) { return (c & 1 ? 14 : 0) ^ (c & 2 ? 4 : 0); }

// Sizes of a tile's pieces in LDS.  K: plane, 32-dim step u, 8-dim chunk c,
// key r at r ^ swz(c) ^ u of its 16-key block (16 bytes each).  V: plane,
// key chunk c (keys 4c .. 4c + 3, 16 + 4c .. 16 + 4c + 3), dim r at
// r ^ swz(c) of its 16-dim block.
template <int DP, int NW = kWaves>
struct Tile {
    static constexpr int kThreads = 64 * NW;
    static constexpr int NU = DP / 32, NB = DP / 16;
    static constexpr int kPlane = kKeys * DP * 2;
    static constexpr int kBuf = 3 * kPlane;  // one tile of K or V
    static constexpr int kUnits = kKeys * DP / 4;  // 4-element units of one operand
    static constexpr int U = (kUnits + kThreads - 1) / kThreads;
    static constexpr bool kAll = kUnits % kThreads == 0;
};

// A thread's share of a K/V tile in registers.
template <int DP, int NW>
struct KvRegs {
    using T = Tile<DP, NW>;
    static constexpr int kThreads = T::kThreads;
    float k[T::U][4], v[T::U][4];

    __device__ __forceinline__ void load(const X3Attn &p, const float *K, const float *V, int k0, int tid) {
        // rows past the last key read as zero (the buffers end there)
        const int n = min(kKeys, p.skv - k0), rs = (int)p.kv_rs;
        const uint32_t bytes = n > 0 ? (uint32_t)(((n - 1) * rs + p.d) * 4) : 0u;
        const int64_t at = (int64_t)(n > 0 ? k0 : 0) * rs;
        const __amdgpu_buffer_rsrc_t kb = coherent_buffer(K + at, bytes), vb = coherent_buffer(V + at, bytes);
#pragma unroll
        for (int u = 0; u < T::U; ++u) {
            const int id = T::kAll ? tid + u * kThreads : min(tid + u * kThreads, T::kUnits - 1);
            const int key = id / (DP / 4), dim = 4 * (id % (DP / 4));
            const f32x4 x = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(kb, (key * rs + (dim < p.d ? dim : 0)) * 4, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) k[u][e] = x[e];
            const int vd = min(id % DP, p.d - 1), vk = 4 * (id / DP);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[u][e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(vb, (vk * rs + vd) * 4, e * rs * 4, 0));
        }
    }
    // The largest magnitude held, NaN if any is.
    __device__ __forceinline__ float largest() const {
        float x = 0.f;
#pragma unroll
        for (int u = 0; u < T::U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) x = max_nan(max_nan(fabsf(k[u][e]), fabsf(v[u][e])), x);
        return x;
    }
    static __device__ __forceinline__ void put(char *at, const float (&x)[4], float up) {
        uint2 p[3];
        split2(x[0] * up, x[1] * up, p[0].x, p[1].x, p[2].x);
        split2(x[2] * up, x[3] * up, p[0].y, p[1].y, p[2].y);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2 *>(at + q * T::kPlane) = p[q];
    }
    __device__ __forceinline__ void store_k(int u, char *lds, int tid) const {
        const int id = tid + u * kThreads;
        if (!T::kAll && id >= T::kUnits) return;
        const int key = id / (DP / 4), q = id % (DP / 4), st = q / 8, c = (q % 8) >> 1;
        put(lds + st * (kKeys * 64) + c * (kKeys * 16) + (key & 16) * 16 + ((key & 15) ^ swz(c) ^ st) * 16 + (q & 1) * 8,
            k[u], 1.f);
    }
    __device__ __forceinline__ void store_v(int u, char *lds, int tid) const {
        const int id = tid + u * kThreads;
        if (!T::kAll && id >= T::kUnits) return;
        const int dim = id % DP, kq = id / DP, c = kq & 3;
        put(lds + c * (DP * 16) + (dim & ~15) * 16 + ((dim & 15) ^ swz(c)) * 16 + (kq >> 2) * 8, v[u], kPieceUp);
    }
};

constexpr float kBig = 0x1p60f;  // the pieces' range, with slack for the products

constexpr float kLog2e = 0x1.715476p+0f;
__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Whether the mask keeps key `key` (< skv) for a query whose first flattened
// score is `base` (reduced modulo mask_numel when mask_rows).
__device__ __forceinline__ float mask_at(const X3Attn &p, int64_t base, int key) {
    const int64_t f = base + key;
    return p.mask[p.mask_rows ? f : f % p.mask_numel];
}

// The scores' products of one 32-key tile for SETS sets of 16 queries: lane
// (c, h), register r of key block kb holds key 16 kb + 4 h + r of query c.
template <int DP, int SETS>
__device__ __forceinline__ void scores(const char *lds, const bf16x8 (&qf)[SETS][DP / 32][3], int c, int h,
                                       f32x4 (&s)[SETS][2]) {
    using T = Tile<DP>;
    constexpr int P[6] = {2, 1, 0, 1, 0, 0}, Q[6] = {0, 1, 2, 0, 1, 0};
    f32x4 lo[SETS][2];
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[i][kb] = lo[i][kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const char *at = lds + h * (kKeys * 16);
    const int row = (c ^ swz(h)) * 16;
#pragma unroll
    for (int u = 0; u < T::NU; ++u) {
        bf16x8 kf[2][3];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int q = 0; q < 3; ++q)
                kf[kb][q] = *reinterpret_cast<const bf16x8 *>(at + (row ^ (u * 16)) + q * T::kPlane + u * (kKeys * 64) +
                                                              kb * 256);
#pragma unroll
        for (int n = 0; n < 6; ++n)
#pragma unroll
            for (int i = 0; i < SETS; ++i)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    f32x4 &acc = n < 5 ? lo[i][kb] : s[i][kb];
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][P[n]], qf[i][u][Q[n]], acc, 0, 0, 0);
                }
    }
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            s[i][kb] = s[i][kb] + lo[i][kb];
            // (The sums are taken here: the compiler would move them behind
            // the next branch, with both addends in registers until then: 13
            // instead of 8 spilled at D = 128 causal, B = 4, H = 32, S = 1000
            // 199 us instead of 193.5.  It waits for the matrix results either
            // way: at least 8 states between an MFMA and the first use of its
            // result on every path of every form of this kernel, 10 for the
            // f32 ones.)
            asm volatile("" : "+v"(s[i][kb]));
        }
}

// f32 attention of one 16-query set straight from memory, for inputs the
// pieces cannot carry: seven to nine times the time of the pieces (B = 4, H =
// 32, S = 1000, D = 128 causal 244 us, with one element beyond in one head 1659,
// in all 2192).
template <int DP, bool CAUSAL, bool MASK, bool WEIGHTS>
__device__ __forceinline__ void set_f32(const X3Attn &p, const float *Q, const float *K, const float *V, float *O,
                                        int64_t wrow0, int q0, int lane) {
    constexpr int NB = DP / 16;
    const int c = lane & 15, h = lane >> 4;
    const int q = q0 + c;
    const float *qrow = Q + (int64_t)min(q, p.sq - 1) * p.q_rs;
    const int64_t mbase = MASK ? (p.mask_rows ? (wrow0 + q) * p.skv % p.mask_numel : (wrow0 + q) * p.skv) : 0;
    const int last = min(p.skv - 1, CAUSAL ? q + p.off : p.skv - 1);
    auto score = [&](int k0) __attribute__((always_inline)) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        const float *krow = K + (int64_t)min(k0 + c, p.skv - 1) * p.kv_rs;
        for (int dim = 0; dim < p.d; dim += 4) s = __builtin_amdgcn_mfma_f32_16x16x4f32(krow[dim + h], qrow[dim + h], s, 0, 0, 0);
        s = s * p.scale;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int key = k0 + 4 * h + r;
            bool keep = key <= last;
            if (MASK && keep) keep = mask_at(p, mbase, key) > 0.5f;
            s[r] = keep ? s[r] : -INFINITY;
        }
        return s;
    };
    f32x4 o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) o[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    const int end = CAUSAL ? min(p.skv, q0 + 16 + p.off) : p.skv;
    for (int k0 = 0; k0 < end; k0 += 16) {
        f32x4 s = score(k0);
        const float m_new = max_nan(m, quarter_max_nan(max_nan(max_nan(s[0], s[1]), max_nan(s[2], s[3]))));
        const bool dead = m_new == -INFINITY;
        const float alpha = dead ? 1.f : __expf(m - m_new);
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = dead ? 0.f : __expf(s[r] - m_new);
            sum += s[r];
        }
        l = l * alpha + quarter_sum(sum);
        m = m_new;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            o[b] *= alpha;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float *vrow = V + (int64_t)min(k0 + 4 * h + r, p.skv - 1) * p.kv_rs;
                o[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vrow[min(16 * b + c, p.d - 1)], s[r], o[b], 0, 0, 0);
            }
        }
    }
    const float inv_l = 1.0f / l;
    if constexpr (WEIGHTS) {
        float *w = p.weights + (wrow0 + q) * p.skv;
        for (int k0 = 0; k0 < p.skv; k0 += 16) {
            const f32x4 s = score(k0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (q < p.sq && k0 + 4 * h + r < p.skv) w[k0 + 4 * h + r] = __expf(s[r] - m) * inv_l;
        }
    }
    // (last: out may be q)
    if (q < p.sq) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
            if (16 * b + 4 * h < p.d) *reinterpret_cast<f32x4 *>(O + (int64_t)q * p.o_rs + 16 * b + 4 * h) = o[b] * inv_l;
    }
}

// NW = kFewWaves: four waves and one V buffer, so that two workgroups share a
// CU at D > 64 (launch_sdpa_x3 has the rule).
template <int DP, int SETS, bool CAUSAL, bool MASK, bool WEIGHTS, int NW>
__global__ __launch_bounds__(64 * NW, SETS == 1 && DP <= 64 ? 4 : 2) void sdpa_x3_kernel(X3Attn p) {
    using T = Tile<DP, NW>;
    constexpr int NU = T::NU, NB = T::NB;
    constexpr bool FEW = NW < kWaves;
    constexpr int kQ = 16 * SETS * NW;  // queries per workgroup
    __shared__ __attribute__((aligned(1024))) char lds[(FEW ? 3 : 5) * T::kBuf];  // K, K, V (, V, V)
    char *const ldsv = lds + 2 * T::kBuf;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, h = lane >> 4;
    const int64_t bh = blockIdx.x;
    const int64_t bb = bh / p.h, hh = bh % p.h;
    const float *Q = p.q + bb * p.q_bs + hh * p.q_hs;
    const float *K = p.k + bb * p.kv_bs + hh * p.kv_hs;
    const float *V = p.v + bb * p.kv_bs + hh * p.kv_hs;
    float *O = p.out + bb * p.o_bs + hh * p.o_hs;
    const int blk = CAUSAL ? (int)gridDim.y - 1 - (int)blockIdx.y : (int)blockIdx.y;  // heaviest first
    const int wq0 = blk * kQ + wave * 16 * SETS;  // this wave's first query

    KvRegs<DP, NW> kv;
    kv.load(p, K, V, 0, tid);
    // (lanes that met an element beyond the pieces; a scale this large could
    // raise scores out of the pieces' last bits)
    uint64_t beyond = fabsf(p.scale) <= 0x1p20f ? 0 : 1;
    float qmax = 0.f;
    bf16x8 qf[SETS][NU][3];
    f32x4 o[SETS][NB];
    float m[SETS], l[SETS];
    int64_t mbase[SETS];
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
        const int q = wq0 + 16 * i + c;
        const float *row = Q + (int64_t)min(q, p.sq - 1) * p.q_rs;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            uint32_t pk[3][4];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int dim = 32 * u + 8 * h + 4 * e;
                const f32x4 x = *reinterpret_cast<const f32x4 *>(row + (dim < p.d ? dim : 0));
                const f32x4 v = dim < p.d ? x : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int r = 0; r < 4; ++r) qmax = max_nan(qmax, fabsf(v[r]));
                split2(v[0], v[1], pk[0][2 * e], pk[1][2 * e], pk[2][2 * e]);
                split2(v[2], v[3], pk[0][2 * e + 1], pk[1][2 * e + 1], pk[2][2 * e + 1]);
            }
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const i32x4 w = {(int)pk[t][0], (int)pk[t][1], (int)pk[t][2], (int)pk[t][3]};
                qf[i][u][t] = __builtin_bit_cast(bf16x8, w);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) o[i][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        m[i] = -INFINITY;
        l[i] = 0.f;
        mbase[i] = MASK ? (p.mask_rows ? (bh * p.sq + q) * p.skv % p.mask_numel : (bh * p.sq + q) * p.skv) : 0;
    }

    const int kv_end = CAUSAL ? min(p.skv, min(blk * kQ + kQ, p.sq) + p.off) : p.skv;
    const int wave_end = CAUSAL ? min(p.skv, min(wq0 + 16 * SETS, p.sq) + p.off) : p.skv;
    const int ntiles = (kv_end + kKeys - 1) / kKeys;
    const bool live = wq0 < p.sq;

    beyond |= __ballot(!(max_nan(qmax, kv.largest()) <= kBig));
#pragma unroll
    for (int u = 0; u < T::U; ++u) {
        kv.store_k(u, lds, tid);
        kv.store_v(u, ldsv, tid);
    }
    kv.load(p, K, V, kKeys, tid);
    __syncthreads();

    // The mask's values for this lane's scores of a tile, requested a tile
    // ahead; bit 4 kb + r: key 16 kb + 4 h + r is kept.
    float mv[MASK ? SETS : 1][8];
    auto load_mask = [&](int k0) __attribute__((always_inline)) {
        if constexpr (MASK) {
#pragma unroll
            for (int i = 0; i < SETS; ++i)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const int key = k0 + 16 * kb + 4 * h;
                    if (p.mask_vec) {
                        const f32x4 x = *reinterpret_cast<const f32x4 *>(p.mask + mbase[i] + min(key, p.skv - 4));
#pragma unroll
                        for (int r = 0; r < 4; ++r) mv[i][4 * kb + r] = x[r];
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) mv[i][4 * kb + r] = mask_at(p, mbase[i], min(key + r, p.skv - 1));
                    }
                }
        }
    };
    uint32_t kept[SETS];
    // Whether any score of the wave's tile is kept.
    auto any_kept = [&]() __attribute__((always_inline)) {
        bool any = !MASK;
        if constexpr (MASK) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                kept[i] = 0;
#pragma unroll
                for (int e = 0; e < 8; ++e) kept[i] |= (mv[i][e] > 0.5f ? 1u : 0u) << e;
                any |= kept[i] != 0 && wq0 + 16 * i + c < p.sq;
            }
            any = __any(any);
        }
        return any;
    };
    auto mask_tile = [&](int i, int k0, f32x4 (&s)[2]) __attribute__((always_inline)) {
        const int q = wq0 + 16 * i + c;
        const int lim = min(p.skv - 1, CAUSAL ? q + p.off : p.skv - 1) - k0;
        // (uniform: every query of the set sees the whole tile)
        const bool full = !MASK && k0 + kKeys <= (CAUSAL ? min(p.skv, wq0 + 16 * i + p.off + 1) : p.skv);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[kb][r] = s[kb][r] * p.scale;
                if (!full) {
                    bool keep = 16 * kb + 4 * h + r <= lim;
                    if (MASK) keep = keep && ((kept[i] >> (4 * kb + r)) & 1);
                    s[kb][r] = keep ? s[kb][r] : -INFINITY;
                }
            }
        }
    };
    load_mask(0);

    // P.V of one tile, with the probabilities' pieces in pf.
    bf16x8 pf[SETS][3];
    auto weigh = [&](const char *vt) __attribute__((always_inline)) {
        constexpr int P[6] = {2, 1, 0, 1, 0, 0}, R[6] = {0, 1, 2, 0, 1, 0};
        const char *at = vt + h * (DP * 16) + (c ^ swz(h)) * 16;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            bf16x8 vf[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) vf[q] = *reinterpret_cast<const bf16x8 *>(at + q * T::kPlane + b * 256);
#pragma unroll
            for (int n = 0; n < 6; ++n)
#pragma unroll
                for (int i = 0; i < SETS; ++i)
                    o[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[P[n]], pf[i][R[n]], o[i][b], 0, 0, 0);
        }
    };
    // The online softmax of one tile: m and l, O's rescale, the pieces of P.
    auto soften = [&](f32x4 (&s)[SETS][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < SETS; ++i) {
            float mb = max_nan(max_nan(s[i][0][0], s[i][0][1]), max_nan(s[i][0][2], s[i][0][3]));
            mb = max_nan(mb, max_nan(max_nan(s[i][1][0], s[i][1][1]), max_nan(s[i][1][2], s[i][1][3])));
            const float m_new = max_nan(m[i], quarter_max_nan(mb));
            // (every score so far masked: any finite maximum gives weights of 0)
            const float ml = -kLog2e * (m_new == -INFINITY ? 0.f : m_new);
            // (the rounded products of both maxima, as the weights use them)
            const float alpha = exp2_fast(ml - -kLog2e * m[i]);
            float pv[8], sum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                pv[e] = exp2_fast(__builtin_fmaf(s[i][e >> 2][e & 3], kLog2e, ml));
                sum += pv[e];
            }
            l[i] = l[i] * alpha + sum;
            m[i] = m_new;
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int b = 0; b < NB; ++b) o[i][b] *= alpha;
            }
            uint32_t pk[3][4];
#pragma unroll
            for (int e = 0; e < 4; ++e) split2(pv[2 * e] * kPieceUp, pv[2 * e + 1] * kPieceUp, pk[0][e], pk[1][e], pk[2][e]);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const i32x4 w = {(int)pk[q][0], (int)pk[q][1], (int)pk[q][2], (int)pk[q][3]};
                pf[i][q] = __builtin_bit_cast(bf16x8, w);
            }
        }
    };

    const bool late = !FEW && wave >= NW / 2;
    bool pending = false;
    int vc = 0, vp = 2;  // V buffers of this tile and the one before
    for (int t = 0; t < ntiles; ++t) {
        const int k0 = t * kKeys, vn = FEW || vc == 2 ? 0 : vc + 1;
        if (pending) weigh(ldsv + vp * T::kBuf);
        pending = false;
        if (live && k0 < wave_end && any_kept()) {
            f32x4 s[SETS][2];
            scores<DP, SETS>(lds + (t & 1) * T::kBuf, qf, c, h, s);
#pragma unroll
            for (int i = 0; i < SETS; ++i) mask_tile(i, k0, s[i]);
            soften(s);
            if (late)
                pending = true;
            else
                weigh(ldsv + vc * T::kBuf);
        }
        load_mask(k0 + kKeys);
        beyond |= __ballot(!(kv.largest() <= kBig));
#pragma unroll
        for (int u = 0; u < T::U; ++u) {
            kv.store_k(u, lds + ((t + 1) & 1) * T::kBuf, tid);
            if (!FEW) kv.store_v(u, ldsv + vn * T::kBuf, tid);
        }
        if constexpr (FEW) {
            __syncthreads();  // every wave is done with this tile's V
#pragma unroll
            for (int u = 0; u < T::U; ++u) kv.store_v(u, ldsv, tid);
        }
        kv.load(p, K, V, k0 + 2 * kKeys, tid);
        __syncthreads();
        vp = vc;
        vc = vn;
    }
    if (pending) weigh(ldsv + vp * T::kBuf);
#pragma unroll
    for (int i = 0; i < SETS; ++i) l[i] = quarter_sum(l[i]);

    bool odd = __syncthreads_or(beyond != 0);
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
        const int q = wq0 + 16 * i + c;
        const float inv_l = 1.0f / l[i];
        bool bad = !(l[i] <= 3.402823466e38f);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = fabsf(o[i][b][r]);
                bad |= !(x <= 3.402823466e38f);
            }
        odd |= bad && m[i] != -INFINITY && q < p.sq;
        l[i] = inv_l;
#pragma unroll
        for (int b = 0; b < NB; ++b) o[i][b] = o[i][b] * kPieceDown * inv_l;
    }
    odd = __any(odd);
    if (live && !odd) {
#pragma unroll
        for (int i = 0; i < SETS; ++i) {
            const int q = wq0 + 16 * i + c;
            if (q >= p.sq) continue;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (16 * b + 4 * h < p.d)
                    *reinterpret_cast<f32x4 *>(O + (int64_t)q * p.o_rs + 16 * b + 4 * h) = o[i][b];
        }
    }

    if constexpr (WEIGHTS) {
        // Second pass: the normalized probabilities of every key (masked ones
        // are 0), with the same scores.
        const int wtiles = (p.skv + kKeys - 1) / kKeys;
        kv.load(p, K, K, 0, tid);
#pragma unroll
        for (int u = 0; u < T::U; ++u) kv.store_k(u, lds, tid);
        kv.load(p, K, K, kKeys, tid);
        load_mask(0);
        __syncthreads();
        for (int t = 0; t < wtiles; ++t) {
            const int k0 = t * kKeys;
            if (live) {
                f32x4 s[SETS][2];
                if (k0 < wave_end && any_kept()) {
                    scores<DP, SETS>(lds + (t & 1) * T::kBuf, qf, c, h, s);
#pragma unroll
                    for (int i = 0; i < SETS; ++i) mask_tile(i, k0, s[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < SETS; ++i)
#pragma unroll
                        for (int kb = 0; kb < 2; ++kb)
                            s[i][kb] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
                }
#pragma unroll
                for (int i = 0; i < SETS; ++i) {
                    const int q = wq0 + 16 * i + c;
                    const float ml = -kLog2e * m[i];
                    float *w = p.weights + (bh * p.sq + q) * p.skv;
                    if (q >= p.sq) continue;
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) {
                        const int key = k0 + 16 * kb + 4 * h;
                        f32x4 x;
#pragma unroll
                        for (int r = 0; r < 4; ++r) x[r] = exp2_fast(__builtin_fmaf(s[i][kb][r], kLog2e, ml)) * l[i];
                        if (p.w_vec) {
                            if (key < p.skv) *reinterpret_cast<f32x4 *>(w + key) = x;
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (key + r < p.skv) w[key + r] = x[r];
                        }
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < T::U; ++u) kv.store_k(u, lds + ((t + 1) & 1) * T::kBuf, tid);
            load_mask(k0 + kKeys);
            kv.load(p, K, K, k0 + 2 * kKeys, tid);
            __syncthreads();
        }
    }
    if (odd) {
        for (int i = 0; i < SETS; ++i)
            if (wq0 + 16 * i < p.sq) set_f32<DP, CAUSAL, MASK, WEIGHTS>(p, Q, K, V, O, bh * p.sq, wq0 + 16 * i, lane);
    }
}

template <int DP, int SETS, int NW = kWaves>
void launch_d(const X3Attn &p, int64_t bh, bool causal, hipStream_t s) {
    const dim3 grid((unsigned)bh, (unsigned)((p.sq + 16 * SETS * NW - 1) / (16 * SETS * NW)));
    const bool mask = p.mask != nullptr, weights = p.weights != nullptr;
    auto go = [&](auto cc, auto mc, auto wc) {
        hipLaunchKernelGGL((sdpa_x3_kernel<DP, SETS, decltype(cc)::value, decltype(mc)::value, decltype(wc)::value, NW>),
                           grid, dim3(64 * NW), 0, s, p);
    };
    using Y = std::true_type;
    using N = std::false_type;
    if constexpr (SETS == 2) {
        if (causal)
            mask ? go(Y{}, Y{}, N{}) : go(Y{}, N{}, N{});
        else
            mask ? go(N{}, Y{}, N{}) : go(N{}, N{}, N{});
    } else if (causal)
        mask ? (weights ? go(Y{}, Y{}, Y{}) : go(Y{}, Y{}, N{})) : (weights ? go(Y{}, N{}, Y{}) : go(Y{}, N{}, N{}));
    else
        mask ? (weights ? go(N{}, Y{}, Y{}) : go(N{}, Y{}, N{})) : (weights ? go(N{}, N{}, Y{}) : go(N{}, N{}, N{}));
}

}  // namespace

// Tile and row indices are 32-bit, a K/V tile's byte offsets too, and the
// grid is one column per (batch, head).
bool sdpa_x3_fits(const SdpaDesc &d) {
    constexpr int64_t kIndex = ((int64_t)1 << 31) - 512;
    return d.sq < kIndex && d.skv < kIndex && (!d.strided || d.kv_rs < (int64_t)1 << 24) &&
           d.b * d.h < (int64_t)1 << 23;
}

int launch_sdpa_x3(const SdpaDesc &d, hipStream_t s) {
    X3Attn p{};
    p.q = d.q;
    p.k = d.k;
    p.v = d.v;
    p.out = d.out;
    p.weights = d.weights;
    p.mask = d.mask;
    p.mask_numel = d.mask_numel;
    p.mask_rows = d.mask && d.mask_numel % d.skv == 0;
    p.mask_vec = p.mask_rows && d.skv % 4 == 0 && aligned16(d.mask);
    p.w_vec = d.skv % 4 == 0 && aligned16(d.weights);
    p.sq = (int)d.sq;
    p.skv = (int)d.skv;
    p.d = (int)d.d;
    p.h = d.h;
    if (d.strided) {
        p.q_bs = d.q_bs, p.q_hs = d.q_hs, p.q_rs = d.q_rs;
        p.kv_bs = d.kv_bs, p.kv_hs = d.kv_hs, p.kv_rs = d.kv_rs;
        p.o_bs = d.o_bs, p.o_hs = d.o_hs, p.o_rs = d.o_rs;
    } else {
        p.q_hs = d.sq * d.d, p.q_bs = d.h * p.q_hs, p.q_rs = d.d;
        p.kv_hs = d.skv * d.d, p.kv_bs = d.h * p.kv_hs, p.kv_rs = d.d;
        p.o_hs = p.q_hs, p.o_bs = p.q_bs, p.o_rs = d.d;
    }
    p.off = (int)(d.causal ? d.skv - d.sq : 0);
    p.scale = d.scale;
    const int64_t bh = d.b * d.h;
    // Two sets per wave halve the tile splits and fragment reads per query;
    // they pay where the launch still holds two rounds of workgroups, the
    // second set is not empty, and the sets' registers leave no second
    // workgroup per CU anyway (us, two sets / one: B = 4, H = 32 causal, D =
    // 128, S = 512 77 / 63, 1000 187 / 204, 2048 673 / 760; D = 80, S = 1000
    // 139 / 156; D = 64, S = 1000 105 / 99; with weights 2 x 8 x 1000, D = 128
    // 248 / 147; 2048 slices of 128 queries and 700 keys, D = 96 509 / 486).
    const bool two = d.d > 64 && !d.weights && d.sq > 128 && bh * ((d.sq + 255) / 256) >= 512;
    // Few queries leave most waves of a workgroup with tiles to split and
    // nothing to multiply; at D > 64 its LDS also fills the CU.  With four
    // waves and one V buffer two share it: worth it once there are more
    // workgroups than CUs (us, four waves / eight: 2048 slices, 700 keys, D =
    // 96, 1 query 201 / 281, 64 queries 294 / 344, 80 502 / 403; 600 slices,
    // D = 128, 1 query 111 / 119; 200 slices 49 / 40).
    const bool few = d.d > 64 && d.sq <= 16 * kFewWaves && bh > device_cu_count();
    if (few)
        d.d <= 96 ? launch_d<96, 1, kFewWaves>(p, bh, d.causal, s) : launch_d<128, 1, kFewWaves>(p, bh, d.causal, s);
    else if (d.d <= 32)
        launch_d<32, 1>(p, bh, d.causal, s);
    else if (d.d <= 64)
        launch_d<64, 1>(p, bh, d.causal, s);
    else if (d.d <= 96)
        two ? launch_d<96, 2>(p, bh, d.causal, s) : launch_d<96, 1>(p, bh, d.causal, s);
    else
        two ? launch_d<128, 2>(p, bh, d.causal, s) : launch_d<128, 1>(p, bh, d.causal, s);
    return check_launch("sdpa (bf16 pieces)");
}

}  // namespace gfh
