// fp32 matrix products on the bf16 matrix cores, for the tied head's loss
// (chunked_lm_loss.py:29-72: logits, and the gradients of hidden states and
// weight):
//   C[m][n] (+)= sum_k A(m, k) B(n, k)
// Each fp32 operand comes as three bf16 pieces x = x1 + x2 + x3 (each the
// rounded remainder of the ones before: 3 x 8 significant bits hold all 24 of
// x), a bf16 operand as one.  A product of two bf16 pieces is exact in fp32
// and the MFMA accumulates in fp32, so (the splitting is Dekker's, "A floating-point
// technique for extending the available precision", 1971, with bf16 pieces)
//   1 x 3 pieces  x1 (y1 + y2 + y3)                              exact products
//   3 x 3 pieces  x1 y1 + x1 y2 + x1 y3 + x2 y1 + x2 y2 + x3 y1  (the terms left
//                 out are below 2^-26 of |x y|, under fp32's own rounding 2^-24)
// at 3 or 6 bf16 products instead of one fp32 product: the bf16 matrix rate is
// 16 times the fp32 one (155 TFLOP/s reached by the BLAS library's fp32 GEMM,
// which is that unit's peak).  Elements that are not finite go whole into the
// first piece; where infinite elements or overflowing products meet pieces that
// are zero or of the other sign, the sum of the piece products is NaN though the
// fp32 product is not: a wave that finds a NaN among its results forms them
// again in fp32 (exact_tile).
//
// Operand layouts, per operand:
//   K_FAST  element (row, k) at row * ld + k   (K padded with zeros in memory
//           to a multiple of 32)
//   K_SLOW  element (row, k) at k * ld + row   (k past K loads zero)
// K_SLOW fragments come out of LDS through the transposing read
// ds_read_b64_tr_b16 (wgrad_gemm.hip describes it), its 4 x 16 blocks chosen so
// that the K-slots agree with K_FAST's: lane half h, slot q <-> k = 8 h + q.
//
// Tile: 256 rows of A x 64 TNF rows of B (TNF = 2 for B in three pieces, else
// 4), 4 waves of 128 x 32 TNF, v_mfma_f32_32x32x16_bf16 with B as the MFMA's A
// operand (a lane's results are 4 consecutive n of one m: 16-byte stores).
// A stage is 32 of K for every piece of both operands: a fragment is read from
// LDS once and multiplied with every piece of the other operand it meets, so
// the LDS moves 5/8 (1 x 3) to 3/8 (3 x 3) of what separate bf16 GEMMs per
// piece pair would.  LDS traffic is what bounds the bf16 GEMMs of this library
// (swiglu_gemm.hip); here the MFMA does (48 or 96 of 32 cycles a stage and
// wave).  Two stages of 40 - 72 KB in LDS: stage s + 2 is loaded (direct to LDS)
// into stage s's buffer from the middle of stage s on, one barrier a stage.
//
// Epilogues (EPI) of the logits form, one slice only:
//   STORE    C in fp32 (above).
//   CE_FWD   per row and wave (32 TNF columns) the maximum of the logits and the sum
//            of exp(x - max), and the label's logit: the logits are not written.
//            ce_merge_kernel merges a row's pairs into its log-sum-exp and loss.
//   CE_BWD   the gradient block scale * (exp(x - lse) - onehot) as its three bf16
//            pieces (the operand of the two gradient products), from the
//            accumulators: neither the logits nor an fp32 gradient are written.
//
// Split K: the stages are cut into slices so that tiles x slices fill the CUs
// (plan_split); each slice's fp32 partial goes to the workspace and a second
// kernel adds them in slice order, so results do not depend on scheduling.
//
// Measured (4096 rows, D = 768, vocabulary 32000; the library's fp32 GEMM before
// -> here, one profiled run; figures beside the code are of pairs run back to back,
// on cards whose clocks differ by some percent; error of the result against 64 bits,
// normwise):
//   logits, bf16 x fp32        1536 -> 589 us (1.02 PFLOP/s bf16)  5.0e-7 -> 3.0e-7
//     with the loss rows       1650 -> 467 us (1.29)
//     with the gradient block  1720 -> 577 us (1.05; 786 MB of pieces written)
//   logits, fp32 x fp32        1518 -> 998 us (1.21)               5.0e-7 -> 4.3e-7
//   d hidden, fp32 x fp32      1458 -> 997 us (1.21)               3.2e-6 -> 1.4e-6
//   d weight, fp32 x bf16      1448 -> 449 us (1.34)               1.1e-6 -> 7.0e-7
//   d weight, fp32 x fp32      1417 -> 957 us (1.26)               1.1e-6 -> 1.0e-6
#include <math.h>

#include <type_traits>

#include "bf16_pieces.h"
#include "lds_dma.h"

namespace mogt {
namespace {

typedef __bf16 sp_bf16x8 __attribute__((ext_vector_type(8)));
typedef short sp_i16x4 __attribute__((ext_vector_type(4)));
typedef short sp_i16x8 __attribute__((ext_vector_type(8)));
typedef float sp_f32x16 __attribute__((ext_vector_type(16)));
typedef float sp_f32x4 __attribute__((ext_vector_type(4)));
typedef float sp_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 sp_bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t sp_u32x2 __attribute__((ext_vector_type(2)));

constexpr int SP_BM = 256;        // rows of A per work-group
constexpr int SP_BK = 32;         // contraction per stage
constexpr int SP_THREADS = 256;   // 4 waves, 2 x 2
constexpr int SP_GROUP_M = 8;     // row blocks walked together per XCD

struct SplitParams {
    const bf16_t* a;
    const bf16_t* b;
    float* out;                // C (one slice) or the partials [slices][M][N]
    int64_t lda, ldb, ldo;     // elements
    int64_t pa, pb;            // elements between pieces
    int64_t po;                // elements between slices of out
    int M, N, K;               // N: multiple of 4 within ldo
    int nb_valid;              // rows of B that exist (K_FAST loads clamp to them)
    int n_mb, n_nb;            // tiles
    int stages, per_slice;     // in all, per slice
    int accumulate;            // out += (one slice)
    // CE_FWD / CE_BWD
    const int64_t* labels;     // [M]
    int64_t ignore;
    float* pairs;              // CE_FWD: [M][2 n_nb][2] (max, sum)
    float* xlab;               // CE_FWD: [M] the label's logit
    const float* lse;          // CE_BWD: [M]
    const float* scale;        // CE_BWD: one value
    bf16_t* grad;              // CE_BWD: [3][M][ldo]
};

enum SplitEpi { EPI_STORE = 0, EPI_CE_FWD = 1, EPI_CE_BWD = 2 };
constexpr float SP_LOG2E = 1.4426950408889634f;

// B's fragments per wave: 2 where B comes in three pieces.  1 x 3 pieces then
// need 80 KB of LDS and 256 registers, so two work-groups share a CU and one's
// epilogue runs beside the other's products: logits with the cross-entropy
// epilogue 566 -> 481 us, with the gradient epilogue 850 -> 660 us then (one
// work-group of 256 columns before), the written logits unchanged (589 us).
__host__ __device__ constexpr int sp_tnf(int nb) { return nb == 3 ? 2 : 4; }

// block id -> (row block, column block, slice): each XCD (ids mod 8) a
// contiguous run, 8 row blocks walked together so that its L2 keeps them
__device__ __forceinline__ void sp_tile(const SplitParams& p, int& mb, int& nb, int& s) {
    const int tiles = p.n_mb * p.n_nb;
    const int n = static_cast<int>(gridDim.x);
    const int bid = blockIdx.x;
    const int q = n >> 3, rem = n & 7;
    const int xcd = bid & 7, loc = bid >> 3;
    const int v = xcd < rem ? xcd * (q + 1) + loc : rem * (q + 1) + (xcd - rem) * q + loc;
    s = v / tiles;
    const int t = v - s * tiles;
    const int group = SP_GROUP_M * p.n_nb;
    const int g = t / group, first = g * SP_GROUP_M;
    const int gm = (p.n_mb - first) < SP_GROUP_M ? (p.n_mb - first) : SP_GROUP_M;
    const int w = t - g * group;
    mb = first + w % gm;
    nb = w / gm;
}

__device__ __forceinline__ sp_i16x4 sp_read_tr(const char* p) {
    typedef __attribute__((address_space(3))) sp_i16x4 lds_i16x4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_i16x4*)((__attribute__((address_space(3))) char*)(const_cast<char*>(p))));
}

// One operand's side of the tile: ROWS = 64 F rows, F 32-row fragments per wave.
template <bool KS, int F>
struct Operand {
    static constexpr int ROWS = 64 * F;
    static constexpr int BYTES = ROWS * 64;          // one piece of a stage
    static constexpr int LOADS = BYTES / 4096;       // 1 KB load instructions per wave and piece
    static constexpr int CMASK = 2 * F - 1;          // K_SLOW: 64-byte chunks per LDS row - 1
    int vo[LOADS];       // per-lane global byte offsets
    int fo[F];           // per-lane LDS byte offsets of the fragments (K_FAST: of the row)
    int swz;             // K_FAST: chunk swizzle of the lane's row

    // valid: rows of this block that exist (K_FAST); side: the wave's half
    __device__ __forceinline__ void init(int wave, int side, int lane, int64_t ld, int valid) {
        const int l32 = lane & 31;
        if constexpr (KS) {
            // an LDS row is one k: 2 F chunks of 32 rows' values (64 B), chunk c
            // of row r at position c ^ (r mod 2 F)
            constexpr int LPR = ROWS / 8;            // lanes per LDS row
            constexpr int RPI = 64 / LPR;            // LDS rows per instruction
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const int r = (wave * LOADS + i) * RPI + lane / LPR, q = lane % LPR;
                vo[i] = static_cast<int>((r * ld + (((q >> 2) ^ (r & CMASK)) << 5) + ((q & 3) << 3)) * 2);
            }
            const int G = lane >> 4, j = lane & 15, r = 8 * (lane >> 5) + (j >> 2);
#pragma unroll
            for (int f = 0; f < F; ++f)
                fo[f] = r * (ROWS * 2) + (((F * side + f) ^ (r & CMASK)) << 6) + 32 * (G & 1) + 8 * (j & 3);
            swz = 0;
        } else {
            const int lc = (lane & 3) ^ (((lane >> 3) ^ (lane >> 4)) & 3);
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                const int r = 16 * (wave * LOADS + i) + (lane >> 2);
                vo[i] = static_cast<int>((r < valid ? r : valid - 1) * ld * 2) + lc * 16;
            }
#pragma unroll
            for (int f = 0; f < F; ++f) fo[f] = (32 * F * side + 32 * f + l32) * 64;
            swz = ((l32 >> 1) ^ (l32 >> 2)) & 3;
        }
    }
    // instruction i of the wave's loads of stage s into LDS `dst` (the piece's base)
    __device__ __forceinline__ void load(lds_i32x4 rsrc, int i, int s, int64_t ld, uint32_t dst, int wave) const {
        const uint32_t at = dst + (wave * LOADS + i) * 1024;
        if constexpr (KS) lds_dma16(rsrc, vo[i] + s * static_cast<int>(SP_BK * ld * 2), 0, at);
        else lds_dma16(rsrc, vo[i], s * (SP_BK * 2), at);
    }
    // fragment f of K-step ks (16 of K) from the piece at `st`
    __device__ __forceinline__ sp_bf16x8 read(const char* st, int ks, int f, int hb) const {
        if constexpr (KS) {
            // rows 8 h + j / 4 and 4 further: the swizzle's bit 2 flips (F = 4)
            const int o0 = fo[f] + ks * (16 * ROWS * 2);
            const int o1 = (CMASK >= 4 ? o0 ^ 256 : o0) + 4 * (ROWS * 2);
            const sp_i16x8 v = __builtin_shufflevector(sp_read_tr(st + o0), sp_read_tr(st + o1), 0, 1, 2, 3, 4, 5, 6, 7);
            return __builtin_bit_cast(sp_bf16x8, v);
        } else {
            return *reinterpret_cast<const sp_bf16x8*>(st + fo[f] + (((2 * ks + hb) ^ swz) << 4));
        }
    }
};

// Q consecutive k of one row of one piece, as loaded (k: a multiple of Q).
template <bool KS, int Q> struct RawRow {
    Pack<bf16_t, Q> w;
    __device__ __forceinline__ void load(const bf16_t* base, int64_t ld, int row, int k, int) {
        w = *reinterpret_cast<const Pack<bf16_t, Q>*>(base + row * ld + k);
    }
    __device__ __forceinline__ float at(int q, int, int) const { return bf16_to_f32(w.v[q]); }
};
template <int Q> struct RawRow<true, Q> {
    bf16_t v[Q];
    // rows past K repeat the last one: the loads carry no condition, which would
    // make each wait for the one before
    __device__ __forceinline__ void load(const bf16_t* base, int64_t ld, int row, int k, int K) {
#pragma unroll
        for (int q = 0; q < Q; ++q) v[q] = base[min(k + q, K - 1) * ld + row];
    }
    __device__ __forceinline__ float at(int q, int k, int K) const { return k + q < K ? bf16_to_f32(v[q]) : 0.0f; }
};

// The wave's accumulators from fp32 products of the same operands (stages s0 ..
// s0 + T - 1), read from memory and summed from their pieces:
// v_mfma_f32_32x32x2_f32 leaves its results where the bf16 form does; lane half h
// takes k = Q h + q of a step of 2 Q.  Rows past the end repeat the last one; their
// results are not used.  (All inputs NaN, where every wave comes here: a training
// pass over 8192 tokens, vocabulary 32000, 21 ms; the BLAS library's fp32 GEMMs 12.)
template <int NA, int NB, bool KSA, bool KSB, int TNF, bool TR>
__device__ __forceinline__ void exact_tile(sp_f32x16 (&acc)[TNF][4], const SplitParams& p, int m0, int n0, int s0, int T,
                                           int l32, int hb) {
    constexpr int Q = NA == 1 && KSA ? 4 : 8;   // 8 would spill at that form's 256 registers
#pragma unroll
    for (int j = 0; j < TNF; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;
    for (int k0 = s0 * SP_BK; k0 < (s0 + T) * SP_BK; k0 += 2 * Q) {
        const int k = k0 + Q * hb;
        RawRow<KSA, Q> a[4][NA];
        RawRow<KSB, Q> b[TNF][NB];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < NA; ++c) a[i][c].load(p.a + c * p.pa, p.lda, min(m0 + 32 * i + l32, p.M - 1), k, p.K);
#pragma unroll
        for (int j = 0; j < TNF; ++j)
#pragma unroll
            for (int c = 0; c < NB; ++c) b[j][c].load(p.b + c * p.pb, p.ldb, min(n0 + 32 * j + l32, p.nb_valid - 1), k, p.K);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            float x[4], y[TNF];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = a[i][0].at(q, k, p.K);
#pragma unroll
                for (int c = 1; c < NA; ++c) x[i] += a[i][c].at(q, k, p.K);
            }
#pragma unroll
            for (int j = 0; j < TNF; ++j) {
                y[j] = b[j][0].at(q, k, p.K);
#pragma unroll
                for (int c = 1; c < NB; ++c) y[j] += b[j][c].at(q, k, p.K);
            }
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(TR ? x[i] : y[j], TR ? y[j] : x[i], acc[j][i], 0, 0, 0);
        }
    }
}

template <int NA, int NB, bool KSA, bool KSB, int TNF, int EPI, bool TR>
__global__ __launch_bounds__(SP_THREADS, NA == 1 && TNF == 2 ? 2 : 1) void split_gemm_kernel(SplitParams p) {
    static_assert(EPI == EPI_STORE || (!KSA && !KSB && !TR), "cross-entropy epilogues: the logits form");
    using OA = Operand<KSA, 4>;
    using OB = Operand<KSB, TNF>;
    constexpr int STB = NA * OA::BYTES + NB * OB::BYTES;
    constexpr int NP = NA == 3 && NB == 3 ? 6 : NA * NB;   // piece pairs
    constexpr int NM = NP * 4 * TNF;                       // MFMAs per K-step and wave
    constexpr int NR = NA * 4 + NB * TNF;                  // fragments per K-step
    constexpr int NL = NA * OA::LOADS + NB * OB::LOADS;    // loads per stage and wave
    static_assert(2 * NR <= NM && 2 * NL <= NM + 1, "reads and loads interleave with the MFMAs");
    __shared__ __attribute__((aligned(1024))) char smem[2 * STB];
    int mb, nb, sl;
    sp_tile(p, mb, nb, sl);
    const int m0 = mb * SP_BM, n0 = nb * OB::ROWS;
    const int s0 = sl * p.per_slice;
    const int T = min(p.per_slice, p.stages - s0);   // >= 1 (host)
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave >> 1, wn = wave & 1;
    const int l32 = lane & 31, hb = lane >> 5;
    const uint32_t lds0 = lds_addr(smem);

    OA oa;
    OB ob;
    oa.init(wave, wm, lane, p.lda, p.M - m0);
    ob.init(wave, wn, lane, p.ldb, p.nb_valid - n0);
    lds_i32x4 ra[NA], rb[NB];
    // K_FAST: from the block's first row to the block's last element; K_SLOW:
    // from (slice start, block's first row) to the last k's row end, in whole
    // 16-byte pieces (a dword partly past the range would load zero)
    const int kv = p.K - s0 * SP_BK;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        if constexpr (KSA)
            ra[i] = lds_rsrc(p.a + i * p.pa + static_cast<int64_t>(s0) * SP_BK * p.lda + m0,
                             static_cast<uint32_t>(((kv - 1) * p.lda + ((p.M - m0 + 7) & ~7)) * 2));
        else
            ra[i] = lds_rsrc(p.a + i * p.pa + m0 * p.lda + s0 * SP_BK,
                             static_cast<uint32_t>((min(p.M - m0, SP_BM) * p.lda - s0 * SP_BK) * 2));
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        if constexpr (KSB)
            rb[i] = lds_rsrc(p.b + i * p.pb + static_cast<int64_t>(s0) * SP_BK * p.ldb + n0,
                             static_cast<uint32_t>(((kv - 1) * p.ldb + ((p.nb_valid - n0 + 7) & ~7)) * 2));
        else
            rb[i] = lds_rsrc(p.b + i * p.pb + n0 * p.ldb + s0 * SP_BK,
                             static_cast<uint32_t>((min(p.nb_valid - n0, OB::ROWS) * p.ldb - s0 * SP_BK) * 2));
    }
    // load t of stage s (t = 0 .. NL - 1: A's pieces, then B's)
    auto load = [&](int t, int s) {
        const uint32_t st = lds0 + (s & 1) * STB;
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if (t >= i * OA::LOADS && t < (i + 1) * OA::LOADS)
                oa.load(ra[i], t - i * OA::LOADS, s, p.lda, st + i * OA::BYTES, wave);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int u = t - NA * OA::LOADS;
            if (u >= i * OB::LOADS && u < (i + 1) * OB::LOADS)
                ob.load(rb[i], u - i * OB::LOADS, s, p.ldb, st + NA * OA::BYTES + i * OB::BYTES, wave);
        }
    };

    sp_f32x16 acc[TNF][4];
#pragma unroll
    for (int j = 0; j < TNF; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;

    struct Frags {
        sp_bf16x8 a[NA][4], b[NB][TNF];
    };
    // fragment r of a K-step in order of first use: a1, b1, then b2, b3, a2, a3
    auto read = [&](Frags& f, int r, int s, int ks) {
        const char* st = smem + (s & 1) * STB;
        if (r < 4) {
            f.a[0][r] = oa.read(st, ks, r, hb);
        } else if (r < 4 + NB * TNF) {
            const int u = r - 4;
            f.b[u / TNF][u % TNF] = ob.read(st + NA * OA::BYTES + (u / TNF) * OB::BYTES, ks, u % TNF, hb);
        } else {
            const int u = r - 4 - NB * TNF;
            f.a[1 + u / 4][u % 4] = oa.read(st + (1 + u / 4) * OA::BYTES, ks, u % 4, hb);
        }
    };
    // pair q of the piece pairs, A's piece slowest: for 3 x 3 (0,0) (0,1) (0,2)
    // (1,0) (1,1) (2,0)
    auto pair_a = [](int q) { return NP == 6 ? (q < 3 ? 0 : q < 5 ? 1 : 2) : NB == 1 ? q : 0; };
    auto pair_b = [](int q) { return NP == 6 ? (q < 3 ? q : q < 5 ? q - 3 : 0) : NB == 1 ? 0 : q; };
    // One K-step's MFMAs on `cur`, with one fragment read of `next` (K-step kn of
    // stage sn) and one load of stage sld every other MFMA; for 3 x 3 pieces, whose
    // MFMAs leave room, the loads evenly over them (hidden gradient at 4096 x
    // 32000 x 768 1012 -> 997 us; a load every MFMA 1052; the 1 x 3 forms were 1 -
    // 3 % slower with even loads).
    constexpr bool SPREAD = NP == 6;
    auto kstep = [&](const Frags& cur, Frags& next, int sn, int kn, int sld, auto reads, auto loads) {
        int t = 0;
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const sp_bf16x8 fa = cur.a[pair_a(q)][i], fb = cur.b[pair_b(q)][j];
                    acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TR ? fa : fb, TR ? fb : fa, acc[j][i], 0, 0, 0);
                    if constexpr (decltype(reads)::value)
                        if (t % 2 == 0 && t / 2 < NR) read(next, t / 2, sn, kn);
                    if constexpr (decltype(loads)::value)
                        if (SPREAD ? (t + 1) * NL / NM > t * NL / NM : t % 2 == 1 && t / 2 < NL)
                            load(SPREAD ? t * NL / NM : t / 2, sld);
                    __builtin_amdgcn_sched_barrier(0);
                    ++t;
                }
    };
    constexpr std::true_type YES{};
    constexpr std::false_type NO{};

    // stages are numbered within the slice (the descriptors start at it)
#pragma unroll
    for (int t = 0; t < NL; ++t) load(t, 0);
    if (T > 1) {
#pragma unroll
        for (int t = 0; t < NL; ++t) load(t, 1);
        lds_wait_vm<NL>();
    } else {
        lds_wait_vm<0>();
    }
    __syncthreads();
    Frags f0, f1;
#pragma unroll
    for (int r = 0; r < NR; ++r) read(f0, r, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    // Stage s: its first K-step reads its second's fragments; then stage s + 1
    // has landed for every wave and stage s's buffer is free (every wave's
    // reads of it are complete before the barrier).
    int s = 0;
    for (; s + 2 < T; ++s) {
        kstep(f0, f1, s, 1, 0, YES, NO);
        lds_wait_vm<0>();
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        kstep(f1, f0, s + 1, 0, s + 2, YES, YES);
    }
    for (; s + 1 < T; ++s) {
        kstep(f0, f1, s, 1, 0, YES, NO);
        lds_wait_vm<0>();
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        kstep(f1, f0, s + 1, 0, 0, YES, NO);
    }
    kstep(f0, f1, s, 1, 0, YES, NO);
    kstep(f1, f0, 0, 0, 0, NO, NO);

    // a NaN among the wave's results (or infinities of both signs) leaves one in
    // their sum (a training pass of the loss over 8192 tokens, vocabulary 32000:
    // 5124 us without the test, 5132 with it)
    if constexpr (NP > 1) {
        float any = 0.0f;
#pragma unroll
        for (int j = 0; j < TNF; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) any += acc[j][i][r];
        if (__any(any != any))
            exact_tile<NA, NB, KSA, KSB, TNF, TR>(acc, p, m0 + 128 * wm, n0 + 32 * TNF * wn, s0, T, l32, hb);
    }

    // lane (l32, hb), register group q of acc[j][i]: row m0 + 128 wm + 32 i +
    // l32, columns n0 + 32 TNF wn + 32 j + 8 q + 4 hb .. + 3
    if constexpr (EPI == EPI_CE_FWD) {
        const int c0 = n0 + 32 * TNF * wn + 4 * hb;   // column of (j, q, e): c0 + 32 j + 8 q + e
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + 128 * wm + 32 * i + l32;
            const int64_t lab = m < p.M ? p.labels[m] : -1;
            // the label's place among this lane's columns (no match: outside)
            const int at = lab >= 0 && lab < p.nb_valid ? static_cast<int>(lab) - c0 : -1;
            float mx = -INFINITY, xl = 0.0f;
            bool has = false;
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int o = 32 * j + 8 * q + e;
                        float x = acc[j][i][4 * q + e];
                        if (at == o) {
                            xl = x;
                            has = true;
                        }
                        if (c0 + o >= p.nb_valid) x = -INFINITY;
                        acc[j][i][4 * q + e] = x;
                        mx = fmaxf(mx, x);
                    }
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mm = mx == -INFINITY ? 0.0f : mx;   // nothing but -inf: every term is 0
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += __builtin_amdgcn_exp2f((acc[j][i][r] - mm) * SP_LOG2E);
            sum += __shfl_xor(sum, 32, 64);
            if (m < p.M) {
                if (hb == 0) {
                    sp_f32x2* pr = reinterpret_cast<sp_f32x2*>(p.pairs) + (static_cast<int64_t>(m) * p.n_nb + nb) * 2 + wn;
                    *pr = sp_f32x2{mx, sum};
                }
                if (has) p.xlab[m] = xl;   // one lane of the grid per row
            }
        }
        return;
    }
    if constexpr (EPI == EPI_CE_BWD) {
        // 32 rows x the wave's columns of one piece at a time through a wave-private
        // LDS tile (rows padded by 16 bytes), so that every store instruction
        // covers whole rows of the wave's columns: with 8-byte stores into 32 rows
        // the kernel ran 897 us at 4096 x 32000 x 768, with the rows
        // staged 850 us, with two work-groups per CU (sp_tnf) 660 us, and with
        // the arithmetic below (no test per element, no spills) 620 us.
        constexpr int CW = 32 * TNF;              // the wave's columns
        constexpr int RS = CW * 2 + 16;           // LDS row stride
        constexpr int LPR = CW / 8;               // lanes per row of 16-byte stores
        static_assert(4 * 32 * RS <= 2 * STB, "four waves' tiles");
        __syncthreads();                          // every wave's fragment reads are done
        char* tile = smem + wave * (32 * RS);
        const float sc = *p.scale;
        const int64_t plane = static_cast<int64_t>(p.M) * p.ldo;
        const int cw0 = n0 + CW * wn;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int mb0 = m0 + 128 * wm + 32 * i;
            const int m = mb0 + l32;
            const int64_t lab = m < p.M ? p.labels[m] : p.ignore;
            const bool skip = lab == p.ignore;
            const float bad = (!skip && (lab < 0 || lab >= p.nb_valid)) ? __builtin_nanf("") : 0.0f;
            const float lr = m < p.M ? p.lse[m] : 0.0f;
            // the gradient replaces the logits; what concerns few rows or tiles (a
            // label among the wave's columns, ignored rows, the vocabulary's end)
            // under uniform branches
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[j][i][r] = __builtin_amdgcn_exp2f((acc[j][i][r] - lr) * SP_LOG2E);
            const int at = lab >= cw0 && lab < cw0 + CW ? static_cast<int>(lab) - cw0 - 4 * hb : -1;
            if (__any(at >= 0)) {
#pragma unroll
                for (int j = 0; j < TNF; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[j][i][r] -= at == 32 * j + 8 * (r >> 2) + (r & 3) ? 1.0f : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[j][i][r] = acc[j][i][r] * sc + bad;
            if (__any(skip) || cw0 + CW > p.nb_valid) {
#pragma unroll
                for (int j = 0; j < TNF; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int n = cw0 + 32 * j + 8 * (r >> 2) + 4 * hb + (r & 3);
                        if (skip || n >= p.nb_valid) acc[j][i][r] = 0.0f;
                    }
            }
            // Pieces two at a time without the tests of bf16_pieces: an element
            // that needs them (not finite, or rounded up to infinity) leaves a
            // NaN as its last remainder
            sp_u32x2 pc[3][TNF * 4];
            float last = 0.0f;
#pragma unroll
            for (int j = 0; j < TNF; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float x0 = acc[j][i][4 * q + 2 * e], x1 = acc[j][i][4 * q + 2 * e + 1];
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector((sp_f32x2{x0, x1}), sp_bf16x2));
                            pc[k][4 * j + q][e] = w;
                            if (k < 2) {
                                x0 -= __uint_as_float(w << 16);
                                x1 -= __uint_as_float(w & 0xffff0000u);
                            }
                        }
                        last += x0;
                        last += x1;
                    }
            if (__any(last != last)) {
#pragma unroll
                for (int j = 0; j < TNF; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        Pack<bf16_t, 4> w[3];
#pragma unroll
                        for (int e = 0; e < 4; ++e) bf16_pieces(acc[j][i][4 * q + e], w[0].v[e], w[1].v[e], w[2].v[e]);
#pragma unroll
                        for (int k = 0; k < 3; ++k) pc[k][4 * j + q] = __builtin_bit_cast(sp_u32x2, w[k]);
                    }
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
#pragma unroll
                for (int t = 0; t < TNF * 4; ++t)
                    *reinterpret_cast<sp_u32x2*>(tile + l32 * RS + (8 * t + 4 * hb) * 2) = pc[k][t];
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
                for (int t = 0; t < 32 * LPR / 64; ++t) {
                    const int r = t * (64 / LPR) + lane / LPR, c = (lane % LPR) * 8;
                    const Pack<bf16_t, 8> w = *reinterpret_cast<const Pack<bf16_t, 8>*>(tile + r * RS + c * 2);
                    if (mb0 + r < p.M && cw0 + c < p.N)   // N: the padded width here, a multiple of 8
                        *reinterpret_cast<Pack<bf16_t, 8>*>(p.grad + k * plane + static_cast<int64_t>(mb0 + r) * p.ldo + cw0 + c) = w;
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            }
        }
        return;
    }
    float* out = p.out + sl * p.po;
    if constexpr (TR) {
        // A was the MFMA's A operand: a lane's results are 4 consecutive m of one
        // n, and C is stored transposed, out[n][m]
#pragma unroll
        for (int j = 0; j < TNF; ++j) {
            const int n = n0 + 32 * TNF * wn + 32 * j + l32;
            if (n >= p.nb_valid) continue;
            float* row = out + n * p.ldo;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int m = m0 + 128 * wm + 32 * i + 8 * q + 4 * hb;
                    if (m >= p.M) continue;
                    sp_f32x4 v = {acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
                    if (p.accumulate) v += *reinterpret_cast<const sp_f32x4*>(row + m);
                    *reinterpret_cast<sp_f32x4*>(row + m) = v;
                }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + 128 * wm + 32 * i + l32;
        if (m >= p.M) continue;
        float* row = out + m * p.ldo;
#pragma unroll
        for (int j = 0; j < TNF; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + 32 * TNF * wn + 32 * j + 8 * q + 4 * hb;
                if (n >= p.N) continue;
                sp_f32x4 v = {acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
                if (p.accumulate) v += *reinterpret_cast<const sp_f32x4*>(row + n);
                *reinterpret_cast<sp_f32x4*>(row + n) = v;
            }
    }
}

// Per-row log-sum-exp and loss from the row's (max, sum) pairs: one wave per
// row.  Labels: ignore_index gives loss 0, others outside the vocabulary NaN.
__global__ __launch_bounds__(256) void ce_merge_kernel(const float* __restrict__ pairs, const float* __restrict__ xlab,
                                                       const int64_t* __restrict__ labels, int64_t ignore, int M,
                                                       int npair, int64_t vocab, float* __restrict__ loss,
                                                       float* __restrict__ lse) {
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= M) return;
    const sp_f32x2* pr = reinterpret_cast<const sp_f32x2*>(pairs) + static_cast<int64_t>(m) * npair;
    float mx = -INFINITY;
    for (int k = lane; k < npair; k += 64) mx = fmaxf(mx, pr[k][0]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    const float mm = mx == -INFINITY ? 0.0f : mx;
    float sum = 0.0f;
    for (int k = lane; k < npair; k += 64) {
        const sp_f32x2 v = pr[k];
        sum += v[1] * __builtin_amdgcn_exp2f((v[0] - mm) * SP_LOG2E);   // v[0] = -inf: 0 (its sum is 0)
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (lane == 0) {
        const float l = mx + logf(sum);
        const int64_t lab = labels[m];
        loss[m] = lab == ignore ? 0.0f : (lab < 0 || lab >= vocab) ? __builtin_nanf("") : l - xlab[m];
        lse[m] = l;
    }
}

// C (+)= sum over slices of the partials, in slice order
template <bool BF16OUT>
__global__ __launch_bounds__(256) void split_reduce_kernel(const float* __restrict__ part, void* __restrict__ out,
                                                           int64_t ldo, int slices, int M, int N, int accumulate) {
    const int per_row = N >> 2;
    const int64_t n = static_cast<int64_t>(M) * per_row, plane = static_cast<int64_t>(M) * N;
    for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < n;
         g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t m = g / per_row;
        const int c = static_cast<int>(g - m * per_row) << 2;
        const float* src = part + m * N + c;
        sp_f32x4 v = *reinterpret_cast<const sp_f32x4*>(src);
        for (int k = 1; k < slices; ++k) v += *reinterpret_cast<const sp_f32x4*>(src + k * plane);
        if constexpr (BF16OUT) {
            const sp_u32x2 w = {
                __builtin_bit_cast(uint32_t, __builtin_convertvector((sp_f32x2{v[0], v[1]}), sp_bf16x2)),
                __builtin_bit_cast(uint32_t, __builtin_convertvector((sp_f32x2{v[2], v[3]}), sp_bf16x2))};
            *reinterpret_cast<sp_u32x2*>(static_cast<bf16_t*>(out) + m * ldo + c) = w;
        } else {
            float* dst = static_cast<float*>(out) + m * ldo + c;
            if (accumulate) v += *reinterpret_cast<const sp_f32x4*>(dst);
            *reinterpret_cast<sp_f32x4*>(dst) = v;
        }
    }
}

// fp32 [rows, cols] -> three bf16 pieces [3][rows][ldd], columns cols .. ldd - 1
// zero; 4 elements per thread
__global__ __launch_bounds__(256) void split_pieces_kernel(const float* __restrict__ src, int64_t lds,
                                                           bf16_t* __restrict__ dst, int64_t ldd, int64_t plane,
                                                           int64_t rows, int64_t cols) {
    const int64_t per_row = ldd >> 2, n = rows * per_row;
    for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < n;
         g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t r = g / per_row, c = (g - r * per_row) << 2;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = c + e < cols ? src[r * lds + c + e] : 0.0f;
        store_pieces4(v, dst + r * ldd + c, plane);
    }
}

struct SplitPlan {
    int64_t stages, per_slice, slices, n_mb, n_nb;
};

// Slices: the count that makes rounds of work-groups (one per CU) times their
// length, plus the partials' traffic, the least.  A stage is taken for its MFMA
// cycles at 1.9 GHz: 1.6 us for 3 x 3 pieces, which take 2.6 in the hidden
// gradient, so the partials' traffic weighs more here than it does there.
SplitPlan plan_split(int64_t M, int64_t N, int64_t K, int na, int nb, int64_t splits, int64_t cus) {
    SplitPlan pl{};
    const int np = na == 3 && nb == 3 ? 6 : na * nb;
    const int tnf = sp_tnf(nb);
    pl.n_mb = (M + SP_BM - 1) / SP_BM;
    pl.n_nb = (N + 64 * tnf - 1) / (64 * tnf);
    pl.stages = (K + SP_BK - 1) / SP_BK;
    const int64_t tiles = pl.n_mb * pl.n_nb;
    int64_t best = splits > 0 ? splits : 1;
    if (splits <= 0) {
        const double stage = np * 4 * tnf * 2 * 32 / 1.9e3;   // us
        double least = 1e30;
        for (int64_t s = 1; s <= 64 && s <= pl.stages; ++s) {
            const int64_t per = (pl.stages + s - 1) / s;
            const int64_t rounds = (tiles * s + cus - 1) / cus;
            double us = static_cast<double>(rounds) * (per * stage + 8.0);
            if (s > 1) us += 4.0 + static_cast<double>(s + 1) * M * N * 8 / 4.0e6;
            if (us < least * 0.98) {
                least = us;
                best = s;
            }
        }
    }
    if (best > pl.stages) best = pl.stages;
    pl.per_slice = (pl.stages + best - 1) / best;
    pl.slices = (pl.stages + pl.per_slice - 1) / pl.per_slice;
    return pl;
}

template <int NA, int NB, bool KSA, bool KSB, int EPI = EPI_STORE, bool TR = false>
void launch_split(const SplitParams& p, int64_t blocks, hipStream_t st) {
    constexpr int TNF = sp_tnf(NB);
    hipLaunchKernelGGL((split_gemm_kernel<NA, NB, KSA, KSB, TNF, EPI, TR>), dim3(static_cast<unsigned>(blocks)),
                       dim3(SP_THREADS), 0, st, p);
}

// the head's products: logits (K_FAST, any pieces), hidden states' gradient
// (K_FAST gradient x K_SLOW weight) and weight's (both K_SLOW), A in 3 pieces
template <bool KSB>
void launch_split_pieces(const SplitParams& p, int na, int nb, int64_t blocks, hipStream_t st) {
    if (na == 3 && nb == 3) launch_split<3, 3, false, KSB>(p, blocks, st);
    else if (na == 3) launch_split<3, 1, false, KSB>(p, blocks, st);
    else if constexpr (!KSB) {
        if (nb == 3) launch_split<1, 3, false, KSB>(p, blocks, st);
        else launch_split<1, 1, false, KSB>(p, blocks, st);
    }
}

// Both operands K_SLOW, 3 x 1 pieces (the weight gradient of a bf16 hidden
// state): the operands swap places and the result is stored transposed, which
// is the 1 x 3 form with its smaller tiles and two work-groups per CU.  At 32000 x
// 768 over 4096 rows that is 750 tiles for 256 CUs (2.9 rounds) where the tiles of
// the 3 x 1 form, one work-group per CU, are 375 (1.5 rounds, run as 2): 552 -> 469
// us; over 1024 rows 184 -> 156, 256 rows 77 -> 56; 4000 x 256 over 1024 rows 30 ->
// 21; 16000 x 1024 over 4096 rows, where both fill their rounds, 305 in both.
bool swap_operands(int na, int nb, bool k_slow_a) { return k_slow_a && na == 3 && nb == 1; }

SplitPlan plan_launch(int64_t M, int64_t N, int64_t K, int na, int nb, bool k_slow_a, int64_t splits, int64_t cus) {
    return swap_operands(na, nb, k_slow_a) ? plan_split(N, M, K, nb, na, splits, cus) : plan_split(M, N, K, na, nb, splits, cus);
}

// Bytes of the slices' fp32 partials (M x N, N rounded up to 4): none where one
// slice writes fp32 straight to the output.
size_t partials_bytes(const SplitPlan& pl, int64_t M, int64_t N, int out_dtype) {
    if (pl.slices == 1 && out_dtype == MOGT_F32) return 0;
    return static_cast<size_t>(pl.slices) * M * ((N + 3) / 4 * 4) * sizeof(float);
}

template <int EPI>
void launch_split_ce(const SplitParams& p, int na, int nb, int64_t blocks, hipStream_t st) {
    if (na == 3 && nb == 3) launch_split<3, 3, false, false, EPI>(p, blocks, st);
    else if (na == 3) launch_split<3, 1, false, false, EPI>(p, blocks, st);
    else if (nb == 3) launch_split<1, 3, false, false, EPI>(p, blocks, st);
    else launch_split<1, 1, false, false, EPI>(p, blocks, st);
}

int check_split_shape(int64_t M, int64_t N, int64_t K, int na, int nb) {
    if (M < 0 || N < 0 || K < 0) return set_error(MOGT_E_INVALID, "split_gemm: negative size");
    if (M > 0x3fffffff || N > 0x3fffffff || K > 0x3fffffff) return set_error(MOGT_E_INVALID, "split_gemm: size");
    if ((na != 1 && na != 3) || (nb != 1 && nb != 3)) return set_error(MOGT_E_INVALID, "split_gemm: 1 or 3 pieces");
    return MOGT_OK;
}

}  // namespace
}  // namespace mogt

using namespace mogt;

extern "C" int mogt_split_pieces(const void* src, int64_t ld_src, void* dst, int64_t ld_dst, int64_t rows,
                                 int64_t cols, void* stream) {
    clear_error();
    if (rows < 0 || cols < 0 || ld_src < cols || ld_dst < cols || ld_dst % 8 != 0)
        return set_error(MOGT_E_INVALID, "split_pieces: bad shape or row stride");
    if (rows == 0 || ld_dst == 0) return MOGT_OK;
    if (!src || !dst) return set_error(MOGT_E_INVALID, "split_pieces: null pointer");
    if (reinterpret_cast<uintptr_t>(dst) & 15) return set_error(MOGT_E_INVALID, "split_pieces: dst needs 16-byte alignment");
    const int64_t groups = rows * (ld_dst / 4);
    const int64_t blocks = (groups + 255) / 256 < 8192 ? (groups + 255) / 256 : 8192;
    hipLaunchKernelGGL(split_pieces_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<const float*>(src), ld_src,
                       static_cast<bf16_t*>(dst), ld_dst, rows * ld_dst, rows, cols);
    return check_launch("split_pieces_kernel");
}

extern "C" size_t mogt_split_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int pieces_a, int pieces_b,
                                                  int k_slow_a, int out_dtype, int64_t splits, int64_t cus) {
    if (check_split_shape(M, N, K, pieces_a, pieces_b) != MOGT_OK || M == 0 || N == 0 || K == 0) return 0;
    if (cus <= 0) {
        int n = 0;
        if (device_cu_count(n) != MOGT_OK) return 0;
        cus = n;
    }
    return partials_bytes(plan_launch(M, N, K, pieces_a, pieces_b, k_slow_a, splits, cus), M, N, out_dtype);
}

extern "C" int mogt_split_gemm(const void* A, int64_t lda, int64_t plane_a, int pieces_a, int k_slow_a, const void* B,
                               int64_t ldb, int64_t plane_b, int pieces_b, int k_slow_b, void* C, int64_t ldc,
                               int64_t M, int64_t N, int64_t K, int accumulate, int out_dtype, int64_t splits,
                               void* workspace, size_t workspace_bytes, void* stream) {
    clear_error();
    if (int rc = check_split_shape(M, N, K, pieces_a, pieces_b)) return rc;
    if (out_dtype != MOGT_F32 && (out_dtype != MOGT_BF16 || accumulate))
        return set_error(MOGT_E_INVALID, "split_gemm: fp32 output, or bf16 without accumulation");
    if ((k_slow_a && !k_slow_b) || (k_slow_b && pieces_a != 3)) return set_error(MOGT_E_INVALID, "split_gemm: layout pair not built");
    const int64_t Kp = (K + SP_BK - 1) / SP_BK * SP_BK, Np = (N + 3) / 4 * 4;
    if (lda % 8 != 0 || ldb % 8 != 0 || plane_a % 8 != 0 || plane_b % 8 != 0 || ldc % 4 != 0 || ldc < Np ||
        lda < (k_slow_a ? M : Kp) || ldb < (k_slow_b ? N : Kp))
        return set_error(MOGT_E_INVALID, "split_gemm: row strides must cover the (padded) rows, multiples of 8 (C: 4)");
    if (M == 0 || N == 0) return MOGT_OK;
    if (K == 0) return set_error(MOGT_E_INVALID, "split_gemm: empty contraction");
    if (!A || !B || !C) return set_error(MOGT_E_INVALID, "split_gemm: null pointer");
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C)) & 15)
        return set_error(MOGT_E_INVALID, "split_gemm: A, B and C need 16-byte alignment");
    // byte offsets within a block's descriptor are 32-bit
    const int64_t spanA = (k_slow_a ? (Kp + SP_BK) : SP_BM) * lda * 2, spanB = (k_slow_b ? (Kp + SP_BK) : 256) * ldb * 2;
    if (spanA >= (int64_t(1) << 31) || spanB >= (int64_t(1) << 31))
        return set_error(MOGT_E_INVALID, "split_gemm: operand block exceeds 2 GiB");
    int cus = 0;
    if (int rc = device_cu_count(cus)) return rc;
    const bool swap = swap_operands(pieces_a, pieces_b, k_slow_a);
    const SplitPlan pl = plan_launch(M, N, K, pieces_a, pieces_b, k_slow_a, splits, cus);
    const int64_t blocks = pl.n_mb * pl.n_nb * pl.slices;
    if (blocks > 0x7fffffff) return set_error(MOGT_E_INVALID, "split_gemm: too many tiles");
    const size_t need = partials_bytes(pl, M, N, out_dtype);
    const bool parts = need > 0;
    if (parts) {
        if (!workspace || workspace_bytes < need)
            return set_error(MOGT_E_WORKSPACE, "split_gemm: workspace of %zu bytes needed, %zu given", need,
                             workspace_bytes);
        if (reinterpret_cast<uintptr_t>(workspace) & 15)
            return set_error(MOGT_E_INVALID, "split_gemm: workspace needs 16-byte alignment");
    }
    SplitParams p{};
    p.a = static_cast<const bf16_t*>(swap ? B : A);
    p.b = static_cast<const bf16_t*>(swap ? A : B);
    p.out = static_cast<float*>(parts ? workspace : C);
    p.lda = swap ? ldb : lda;
    p.ldb = swap ? lda : ldb;
    p.ldo = parts ? Np : ldc;
    p.pa = swap ? plane_b : plane_a;
    p.pb = swap ? plane_a : plane_b;
    p.po = M * Np;
    p.M = static_cast<int>(swap ? N : M);
    p.N = static_cast<int>(Np);
    p.K = static_cast<int>(K);
    p.nb_valid = static_cast<int>(swap ? M : N);
    p.n_mb = static_cast<int>(pl.n_mb);
    p.n_nb = static_cast<int>(pl.n_nb);
    p.stages = static_cast<int>(pl.stages);
    p.per_slice = static_cast<int>(pl.per_slice);
    p.accumulate = !parts && accumulate;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (swap) launch_split<1, 3, true, true, EPI_STORE, true>(p, blocks, st);
    else if (k_slow_a) launch_split<3, 3, true, true>(p, blocks, st);
    else if (k_slow_b) launch_split_pieces<true>(p, pieces_a, pieces_b, blocks, st);
    else launch_split_pieces<false>(p, pieces_a, pieces_b, blocks, st);
    int rc = check_launch("split_gemm_kernel");
    if (rc != MOGT_OK || !parts) return rc;
    const int64_t groups = M * (Np / 4);
    const dim3 rb(static_cast<unsigned>((groups + 255) / 256 < 8192 ? (groups + 255) / 256 : 8192));
    if (out_dtype == MOGT_BF16)
        hipLaunchKernelGGL(split_reduce_kernel<true>, rb, dim3(256), 0, st, static_cast<const float*>(workspace), C, ldc,
                           static_cast<int>(pl.slices), static_cast<int>(M), p.N, 0);
    else
        hipLaunchKernelGGL(split_reduce_kernel<false>, rb, dim3(256), 0, st, static_cast<const float*>(workspace), C,
                           ldc, static_cast<int>(pl.slices), static_cast<int>(M), p.N, accumulate);
    return check_launch("split_reduce_kernel");
}

namespace {

// Checks and fills the parameters the logits form's cross-entropy entries share;
// out: blocks of the launch.
int prepare_split_ce(SplitParams& p, const void* A, int64_t lda, int64_t plane_a, int na, const void* B, int64_t ldb,
                     int64_t plane_b, int nb, const int64_t* labels, int64_t M, int64_t N, int64_t K, int64_t ignore,
                     int64_t& blocks) {
    if (int rc = check_split_shape(M, N, K, na, nb)) return rc;
    const int64_t Kp = (K + SP_BK - 1) / SP_BK * SP_BK;
    if (N == 0 || K == 0) return set_error(MOGT_E_INVALID, "split_ce: empty vocabulary or contraction");
    if (lda % 8 != 0 || ldb % 8 != 0 || plane_a % 8 != 0 || plane_b % 8 != 0 || lda < Kp || ldb < Kp)
        return set_error(MOGT_E_INVALID, "split_ce: row strides must cover the padded rows, multiples of 8");
    if (M > 0 && (!A || !B || !labels)) return set_error(MOGT_E_INVALID, "split_ce: null pointer");
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15)
        return set_error(MOGT_E_INVALID, "split_ce: A and B need 16-byte alignment");
    if (SP_BM * lda * 2 >= (int64_t(1) << 31) || 256 * ldb * 2 >= (int64_t(1) << 31))
        return set_error(MOGT_E_INVALID, "split_ce: operand block exceeds 2 GiB");
    const SplitPlan pl = plan_split(M, N, K, na, nb, 1, 1);
    blocks = pl.n_mb * pl.n_nb;
    if (blocks > 0x7fffffff) return set_error(MOGT_E_INVALID, "split_ce: too many tiles");
    p.a = static_cast<const bf16_t*>(A);
    p.b = static_cast<const bf16_t*>(B);
    p.lda = lda;
    p.ldb = ldb;
    p.pa = plane_a;
    p.pb = plane_b;
    p.M = static_cast<int>(M);
    p.N = static_cast<int>(N);
    p.K = static_cast<int>(K);
    p.nb_valid = static_cast<int>(N);
    p.n_mb = static_cast<int>(pl.n_mb);
    p.n_nb = static_cast<int>(pl.n_nb);
    p.stages = p.per_slice = static_cast<int>(pl.stages);
    p.labels = labels;
    p.ignore = ignore;
    return MOGT_OK;
}

int64_t split_ce_pairs(int64_t N, int na, int nb) {
    const int64_t cols = 64 * sp_tnf(nb);
    return 2 * ((N + cols - 1) / cols);
}

}  // namespace

extern "C" int64_t mogt_split_gemm_slices(int64_t M, int64_t N, int64_t K, int pieces_a, int pieces_b, int64_t cus) {
    if (check_split_shape(M, N, K, pieces_a, pieces_b) != MOGT_OK || M == 0 || N == 0 || K == 0) return 0;
    if (cus <= 0) {
        int n = 0;
        if (device_cu_count(n) != MOGT_OK) return 0;
        cus = n;
    }
    return plan_split(M, N, K, pieces_a, pieces_b, 0, cus).slices;
}

extern "C" size_t mogt_split_ce_workspace_bytes(int64_t M, int64_t N, int pieces_a, int pieces_b) {
    if (M <= 0 || N <= 0) return 0;
    return static_cast<size_t>(M) * (split_ce_pairs(N, pieces_a, pieces_b) * 2 + 1) * sizeof(float);
}

extern "C" int mogt_split_ce_fwd(const void* A, int64_t lda, int64_t plane_a, int pieces_a, const void* B, int64_t ldb,
                                 int64_t plane_b, int pieces_b, const int64_t* labels, int64_t M, int64_t N, int64_t K,
                                 int64_t ignore_index, float* loss_rows, float* lse_rows, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    clear_error();
    SplitParams p{};
    int64_t blocks = 0;
    int rc = prepare_split_ce(p, A, lda, plane_a, pieces_a, B, ldb, plane_b, pieces_b, labels, M, N, K, ignore_index, blocks);
    if (rc) return rc;
    if (M == 0) return MOGT_OK;
    if (!loss_rows || !lse_rows) return set_error(MOGT_E_INVALID, "split_ce_fwd: null pointer");
    const size_t need = mogt_split_ce_workspace_bytes(M, N, pieces_a, pieces_b);
    if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15))
        return set_error(MOGT_E_WORKSPACE, "split_ce_fwd: 16-byte aligned workspace of %zu bytes needed, %zu given", need,
                         workspace_bytes);
    const int npair = static_cast<int>(split_ce_pairs(N, pieces_a, pieces_b));
    p.pairs = static_cast<float*>(workspace);
    p.xlab = p.pairs + M * npair * 2;
    hipStream_t st = static_cast<hipStream_t>(stream);
    launch_split_ce<EPI_CE_FWD>(p, pieces_a, pieces_b, blocks, st);
    rc = check_launch("split_gemm_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(ce_merge_kernel, dim3(static_cast<unsigned>((M + 3) / 4)), dim3(256), 0, st, p.pairs, p.xlab, labels,
                       ignore_index, p.M, npair, N, loss_rows, lse_rows);
    return check_launch("ce_merge_kernel");
}

extern "C" int mogt_split_ce_bwd(const void* A, int64_t lda, int64_t plane_a, int pieces_a, const void* B, int64_t ldb,
                                 int64_t plane_b, int pieces_b, const int64_t* labels, const float* lse_rows, int64_t M,
                                 int64_t N, int64_t K, int64_t ignore_index, const float* scale, void* grad,
                                 int64_t ld_grad, void* stream) {
    clear_error();
    SplitParams p{};
    int64_t blocks = 0;
    int rc = prepare_split_ce(p, A, lda, plane_a, pieces_a, B, ldb, plane_b, pieces_b, labels, M, N, K, ignore_index, blocks);
    if (rc) return rc;
    if (M == 0) return MOGT_OK;
    if (!lse_rows || !scale || !grad) return set_error(MOGT_E_INVALID, "split_ce_bwd: null pointer");
    // the zero padding is written by the tiles, which end at a multiple of 128
    if (ld_grad < N || ld_grad % 8 != 0 || ld_grad > (N + 127) / 128 * 128 || (reinterpret_cast<uintptr_t>(grad) & 15))
        return set_error(MOGT_E_INVALID, "split_ce_bwd: gradient row stride or alignment");
    p.lse = lse_rows;
    p.scale = scale;
    p.grad = static_cast<bf16_t*>(grad);
    p.ldo = ld_grad;
    p.N = static_cast<int>(ld_grad);
    launch_split_ce<EPI_CE_BWD>(p, pieces_a, pieces_b, blocks, static_cast<hipStream_t>(stream));
    return check_launch("split_gemm_kernel");
}
