// Parameters and element access of the generic affine scan's chunk passes
// (generic_scan.hip), and its matrix-core chunk kernel for ranks up to 64
// (instantiated per state type in generic_mfma_f32.hip / generic_mfma_f64.hip).
//
// generic_mfma_kernel: one wave per (sequence, chunk, group of CW 16-column
// state tiles), M_t = U_t M_{t-1} + [V_t | 0] on v_mfma_f32_16x16x4_f32 /
// v_mfma_f64_16x16x4_f64.  The state's R rows (RT 16-row tiles) stay in the
// wave's accumulators for the whole chunk.  Lane (g = lane / 16, n = lane % 16)
// holds rows 16 rt + 4 g + i, i = 0..3, of column n of a tile; K-step kk of
// contraction tile kt takes row 16 kt + 4 g + kk, i.e. accumulator register kk
// of the previous step in the same lane, so the state never moves between
// steps, and a lane's A operands are 4 consecutive values of one row of U_t.
// The f64 MFMA's result register i of group g is row g + 4 i (the f32 one's 4 g +
// i): the f64 form permutes the state's rows, rho(m) = 4 (m % 4) + m / 4, which
// only changes the row of U_t that a lane loads.
//
// Every step's block of U, V and the outputs is reached through a buffer
// descriptor: rows past R lie past its range, columns past a view's width get
// an offset past it, so padding loads zero and its stores are dropped.  PD steps
// of operands are in flight.
//
// What bounds it: a step's chain of MFMAs in a wave for R = 64 (128 MFMAs of 32
// cycles at CW = 2; counters over LOCAL of 24 x 2048 steps: matrix unit busy 69 % of
// the cycles, 4 % of the waves' spent waiting), memory for R = 16 in float64.  The
// scalar kernel it replaces at these ranks (one dot product per thread over LDS) spent
// about 2 us in every step on its barriers and LDS round trips; it stays for wide
// states of ranks up to 4 (generic_scan.hip, scalar_pays).  Measured: float64 R =
// 16, C = 48, L = 32768 1036 -> 198 us (LOCAL 52 us = 5.2 TB/s, OUTPUT 106, the
// carries in three passes 31 instead of 82 in one); fp32 R = C = 64, 24 x 2048
// steps 4360 -> 1178 us, and with the memory instructions spread between the
// MFMAs and a lane's two columns adjacent (P2: 8-byte loads and stores, whose
// counter then never limits the operands in flight) 1110 us; with the prefix
// written too 1795 -> 1548 us.  PD = 4 in place of 2: no gain, up to 8 % slower.
#pragma once

#include <math.h>

#include <type_traits>

#include "common.h"

namespace mogt {

// A [batch][sequence][rows][cols] view of a device buffer (strides in elements).
struct GView {
    void* p;
    int64_t bs, ss, rs;
    int code;
};

struct GParams {
    GView tr;        // transitions, state dtype; column offset tr_c0
    GView in;        // inputs, columns [0, cin)
    GView init;      // initial state per (batch, chunk), state dtype; p == nullptr: [0 | I]
    GView out_h;     // state columns [0, csplit)
    GView out_p;     // state columns [csplit, W), written at column c - csplit (p may be null)
    int64_t L;       // positions in the scanned sequence
    int64_t seg;     // positions per chunk (one work-group's run)
    int nseg, ntile;
    int R, W, Cb;    // rank, state width, column-tile width
    int tr_c0, cin, cid, csplit;  // cid: first identity column of the [0 | I] start
    int every;       // 1: write the state after every step; 0: the final state at the chunk index
    int shift;       // 1: step q is written at index q + 1 and the first chunk's initial state at index 0
    int rev;         // reverse, transposed transitions (generic_scan.hip's file comment)
    int stream;      // outputs are not read again by this scan
    int scalar;      // host: take the scalar kernel (generic_scan.hip)
};

__device__ __forceinline__ int64_t at(const GView& v, int64_t b, int64_t s, int64_t r, int64_t c) {
    return b * v.bs + s * v.ss + r * v.rs + c;
}

template <typename TS>
__device__ __forceinline__ TS ld_code(const void* p, int64_t i, int code) {
    if (code == MOGT_F64) return static_cast<TS>(static_cast<const double*>(p)[i]);
    if (code == MOGT_BF16) return static_cast<TS>(bf16_to_f32(static_cast<const bf16_t*>(p)[i]));
    if (code == MOGT_F16) return static_cast<TS>(static_cast<float>(static_cast<const _Float16*>(p)[i]));
    return static_cast<TS>(static_cast<const float*>(p)[i]);
}

// Narrow outputs round from the state through fp32 (round to nearest even at each step),
// as a torch float64 -> bfloat16 / float16 conversion does.
template <typename TS>
__device__ __forceinline__ void st_code(void* p, int64_t i, int code, TS x) {
    if (code == MOGT_F64) {
        static_cast<double*>(p)[i] = static_cast<double>(x);
        return;
    }
    const float f = static_cast<float>(x);
    if (code == MOGT_BF16) static_cast<bf16_t*>(p)[i] = f32_to_bf16(f);
    else if (code == MOGT_F16) static_cast<_Float16*>(p)[i] = static_cast<_Float16>(f);
    else static_cast<float*>(p)[i] = f;
}

template <typename TS>
__device__ __forceinline__ void put(const GParams& p, int64_t b, int64_t idx, int i, int c, TS x) {
    if (c < p.csplit) {
        st_code<TS>(p.out_h.p, at(p.out_h, b, idx, i, c), p.out_h.code, x);
    } else if (p.out_p.p) {
        st_code<TS>(p.out_p.p, at(p.out_p, b, idx, i, c - p.csplit), p.out_p.code, x);
    }
}

typedef uint32_t gm_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t gm_u32x4 __attribute__((ext_vector_type(4)));

template <typename TS> struct GMma;
template <> struct GMma<float> {
    typedef float vec __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ vec mma(float a, float b, vec c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int arow(int n) { return n; }
};
template <> struct GMma<double> {
    typedef double vec __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ vec mma(double a, double b, vec c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int arow(int n) { return 4 * (n & 3) + (n >> 2); }
};

constexpr int GM_MAX_R = 64;      // ranks of the matrix-core kernel
constexpr int GM_WAVES = 4;       // waves (independent) per work-group
constexpr uint32_t GM_OOB = 0x40000000u;   // past every range, also after a row offset
constexpr int64_t GM_MAX_BLOCK = 0x3fffffff;   // bytes of one step's block of a view, padded rows included

// Steps of operands in flight: what fits the registers beside the state.
template <typename TS, int RT> constexpr int gm_depth() { return RT == 1 ? 8 : RT == 2 ? 4 : 2; }

// How a lane loads its 4 values of a row of U: one by one, or as 16-byte loads
// (R a multiple of 4, rows 16-byte aligned, not reversed); FULL: those, and the
// rank fills its row tiles (no padded row to keep zero, 0.8 % of the R = 16,
// C = 48, L = 32768 float64 scan).
enum GmU { GM_U1 = 0, GM_U16 = 1, GM_U16_FULL = 2 };

// OUT of the native form (inputs and outputs in the state's dtype): what a pass
// writes.  The general form (any io dtype) decides at run time.
enum GmOut { GM_FINAL = 0, GM_EVERY_H = 1, GM_EVERY_HP = 2, GM_ANY = 3 };

// P2 (two tiles per wave, both columns of a pair inside or outside every view,
// 8-byte aligned): tile h of the wave holds columns 2 n + h of its 32.
// IS: bytes of an input element (2: bf16 or fp16); UA: GmU.  The native form
// issues the same loads and stores in every step (padding steps of a ragged
// chunk have empty ranges), so no wait has to assume that the operands in flight
// were never issued.
template <typename TS, int RT, int CW, int IS, int UA, int OUT, bool P2>
__global__ __launch_bounds__(64 * GM_WAVES) void generic_mfma_kernel(GParams p, int64_t waves) {
    static_assert(!P2 || (CW == 2 && sizeof(TS) == 4 && IS == 4 && OUT != GM_ANY), "paired columns: two fp32 tiles");
    typedef GMma<TS> M;
    typedef typename M::vec vec;
    constexpr bool ANY = OUT == GM_ANY;
    constexpr bool VA = UA != GM_U1;
    constexpr int PD = gm_depth<TS, RT>();
    constexpr int SS = static_cast<int>(sizeof(TS));
    constexpr bool SPREAD = !ANY && CW == 2;
    const int64_t wid = static_cast<int64_t>(blockIdx.x) * GM_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wid >= waves) return;   // whole waves: nothing below is shared between them
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int ct = static_cast<int>(wid % p.ntile);
    const int64_t rest = wid / p.ntile;
    const int j = static_cast<int>(rest % p.nseg);
    const int64_t b = rest / p.nseg;
    const int64_t q0 = static_cast<int64_t>(j) * p.seg;
    const int len = static_cast<int>(p.L - q0 < p.seg ? p.L - q0 : p.seg);
    const int R = p.R;

    auto rsrc = [](const void* base, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
    };
    auto code_bytes = [](int code) { return ANY ? (code == MOGT_F64 ? 8 : code == MOGT_F32 ? 4 : 2) : SS; };
    auto trow = [&](int rt, int i) { return 16 * rt + 4 * g + i; };
    int col[CW];
#pragma unroll
    for (int h = 0; h < CW; ++h) col[h] = P2 ? ct * 32 + 2 * n + h : (ct * CW + h) * 16 + n;

    // per-lane byte offsets inside a step's block
    uint32_t offA[RT][RT][VA ? 1 : 4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int kt = 0; kt < RT; ++kt)
#pragma unroll
            for (int kk = 0; kk < (VA ? 1 : 4); ++kk) {
                const int r = 16 * rt + M::arow(n), c = 16 * kt + 4 * g + kk;
                const int e = p.rev ? c * static_cast<int>(p.tr.rs) + r : r * static_cast<int>(p.tr.rs) + c;
                offA[rt][kt][kk] = (r < R && c < R) ? static_cast<uint32_t>((e + p.tr_c0) * SS) : GM_OOB;
            }
    const uint32_t vrow = static_cast<uint32_t>(p.in.rs) * IS;
    uint32_t offV[CW];
#pragma unroll
    for (int h = 0; h < CW; ++h)
        offV[h] = col[h] < p.cin ? 4 * g * vrow + static_cast<uint32_t>(col[h]) * IS : GM_OOB;
    const int ob_h = code_bytes(p.out_h.code), ob_p = code_bytes(p.out_p.code);
    const uint32_t hrow = static_cast<uint32_t>(p.out_h.rs) * ob_h, prow = static_cast<uint32_t>(p.out_p.rs) * ob_p;
    uint32_t offH[CW], offP[CW];
    bool anyH = false, anyP = false;   // uniform: whether the wave's tiles hold such columns
#pragma unroll
    for (int h = 0; h < CW; ++h) {
        const int c = col[h], c0 = (ct * CW + h) * 16;
        offH[h] = c < p.csplit ? 4 * g * hrow + static_cast<uint32_t>(c * ob_h) : GM_OOB;
        offP[h] = (c >= p.csplit && c < p.W && p.out_p.p) ? 4 * g * prow + static_cast<uint32_t>((c - p.csplit) * ob_p)
                                                         : GM_OOB;
        anyH |= c0 < p.csplit;
        anyP |= p.out_p.p && c0 + 16 > p.csplit && c0 < p.W;
    }
    const uint32_t trBytes = static_cast<uint32_t>((p.tr.rs * (R - 1) + p.tr_c0 + R) * SS);
    const uint32_t inBytes = p.in.p && p.cin > 0 ? static_cast<uint32_t>((p.in.rs * (R - 1) + p.cin) * IS) : 0u;
    const uint32_t hBytes = p.out_h.p && p.csplit > 0 ? static_cast<uint32_t>((p.out_h.rs * (R - 1) + p.csplit) * ob_h) : 0u;
    const uint32_t pBytes = p.out_p.p ? static_cast<uint32_t>((p.out_p.rs * (R - 1) + (p.W - p.csplit)) * ob_p) : 0u;

    // initial state; rows past R and columns past W stay zero
    vec X[RT][CW];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int h = 0; h < CW; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = trow(rt, i), c = col[h];
                TS x = TS(0);
                if (r < R && c < p.W) {
                    if (p.init.p) x = ld_code<TS>(p.init.p, at(p.init, b, j, r, c), p.init.code);
                    else if (c >= p.cid) x = r == c - p.cid ? TS(1) : TS(0);
                }
                X[rt][h][i] = x;
            }

    // Streamed outputs (not read again by this scan) are stored non-temporally
    // where a store instruction covers whole 128-byte lines (8-byte values).
    auto st_one = [](__amdgpu_buffer_rsrc_t r, uint32_t off, int code, TS x, bool stream) {
        if constexpr (!ANY && SS == 4) {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(static_cast<float>(x)), r, off, 0, 0);
        } else if (!ANY || code == MOGT_F64) {
            const gm_u32x2 w = __builtin_bit_cast(gm_u32x2, static_cast<double>(x));
            if (stream) __builtin_amdgcn_raw_buffer_store_b64(w, r, off, 0, 2);
            else __builtin_amdgcn_raw_buffer_store_b64(w, r, off, 0, 0);
        } else {
            const float f = static_cast<float>(x);
            if (code == MOGT_F32) {
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(f), r, off, 0, 0);
            } else {
                const uint16_t w = code == MOGT_BF16 ? f32_to_bf16(f)
                                                     : __builtin_bit_cast(uint16_t, static_cast<_Float16>(f));
                __builtin_amdgcn_raw_buffer_store_b16(w, r, off, 0, 0);
            }
        }
    };
    // element e = (rt, i, tile) of the lane's state, with P2 both tiles' values
    constexpr int HS = P2 ? 1 : CW;
    auto store_piece = [&](__amdgpu_buffer_rsrc_t r, const uint32_t (&off)[CW], uint32_t row, int code, int e, bool stream) {
        const int h = e % HS, i = e / HS % 4, rt = e / HS / 4;
        if constexpr (P2) {
            const gm_u32x2 w = {__float_as_uint(static_cast<float>(X[rt][0][i])), __float_as_uint(static_cast<float>(X[rt][1][i]))};
            __builtin_amdgcn_raw_buffer_store_b64(w, r, off[0] + (16 * rt + i) * row, 0, 0);
        } else {
            st_one(r, off[h] + (16 * rt + i) * row, code, X[rt][h][i], stream);
        }
    };
    auto store_state = [&](char* ph, char* pp, bool valid, bool stream, auto wantH, auto wantP) {
        if constexpr (decltype(wantH)::value) {
            const auto rh = rsrc(ph, valid ? hBytes : 0u);
#pragma unroll
            for (int e = 0; e < RT * 4 * HS; ++e) store_piece(rh, offH, hrow, p.out_h.code, e, stream);
        }
        if constexpr (decltype(wantP)::value) {
            const auto rp = rsrc(pp, valid ? pBytes : 0u);
#pragma unroll
            for (int e = 0; e < RT * 4 * HS; ++e) store_piece(rp, offP, prow, p.out_p.code, e, stream);
        }
    };
    constexpr std::true_type YES{};
    constexpr std::false_type NO{};
    auto store_any = [&](char* ph, char* pp, bool stream) {
        if (anyH) store_state(ph, pp, true, stream, YES, NO);
        if (anyP) store_state(ph, pp, true, stream, NO, YES);
    };
    auto out_at = [&](const GView& v, int64_t idx, int bytes) { return static_cast<char*>(v.p) + (b * v.bs + idx * v.ss) * bytes; };
    if (p.shift && j == 0) store_any(out_at(p.out_h, 0, ob_h), out_at(p.out_p, 0, ob_p), false);

    // running pointers of the next step to fetch and of the step in hand
    // (reversed: U at L - q, inputs and outputs at L - 1 - q)
    const int64_t dir = p.rev ? -1 : 1;
    const char* fu = static_cast<const char*>(p.tr.p) + (b * p.tr.bs + (p.rev ? p.L - q0 : q0) * p.tr.ss) * SS;
    const char* fv = static_cast<const char*>(p.in.p) + (b * p.in.bs + (p.rev ? p.L - 1 - q0 : q0) * p.in.ss) * IS;
    const int64_t du = dir * p.tr.ss * SS, dv = dir * p.in.ss * IS;
    char* oh = out_at(p.out_h, (p.rev ? p.L - 1 - q0 : q0) + p.shift, ob_h);
    char* op = out_at(p.out_p, (p.rev ? p.L - 1 - q0 : q0) + p.shift, ob_p);
    const int64_t dh = dir * p.out_h.ss * ob_h, dp = dir * p.out_p.ss * ob_p;

    struct Ops {
        vec A[RT][RT];
        uint32_t v[RT][CW][4][IS == 8 ? 2 : 1];
    };
    // operands of the chunk's step s, which must be fetched in order; an empty
    // range past the chunk, and for the transition of reversed position 0 (the
    // state before it is zero)
    auto rsrc_u = [&](int s) { return rsrc(fu, s < len && !(p.rev && q0 + s == 0) ? trBytes : 0u); };
    auto rsrc_v = [&](int s) { return rsrc(fv, s < len ? inBytes : 0u); };
    auto fetch_a = [&](__amdgpu_buffer_rsrc_t ru, Ops& o, int rt, int kt) {
        if constexpr (VA && SS == 4) {
            o.A[rt][kt] = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(ru, offA[rt][kt][0], 0, 0));
        } else if constexpr (VA) {
            struct Two { gm_u32x4 a, b; } w = {
                __builtin_bit_cast(gm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(ru, offA[rt][kt][0], 0, 0)),
                __builtin_bit_cast(gm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(ru, offA[rt][kt][0] + 16, 0, 0))};
            o.A[rt][kt] = __builtin_bit_cast(vec, w);
        } else {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                if constexpr (SS == 4)
                    o.A[rt][kt][kk] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ru, offA[rt][kt][kk], 0, 0));
                else
                    o.A[rt][kt][kk] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ru, offA[rt][kt][kk], 0, 0));
            }
        }
    };
    auto fetch_v = [&](__amdgpu_buffer_rsrc_t rv, Ops& o, int e) {
        const int h = e % HS, i = e / HS % 4, rt = e / HS / 4;
        const uint32_t off = offV[h] + (16 * rt + i) * vrow;
        if constexpr (P2) {
            const gm_u32x2 w = __builtin_bit_cast(gm_u32x2, __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0));
            o.v[rt][0][i][0] = w[0];
            o.v[rt][1][i][0] = w[1];
        } else if constexpr (IS == 8) {
            const gm_u32x2 w = __builtin_bit_cast(gm_u32x2, __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0));
            o.v[rt][h][i][0] = w[0];
            o.v[rt][h][i][1] = w[1];
        } else if constexpr (IS == 4) {
            o.v[rt][h][i][0] = __builtin_amdgcn_raw_buffer_load_b32(rv, off, 0, 0);
        } else {
            o.v[rt][h][i][0] = static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b16(rv, off, 0, 0));
        }
    };
    auto fetch = [&](int s, Ops& o) {
        const auto ru = rsrc_u(s), rv = rsrc_v(s);
        fu += du;
        fv += dv;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int kt = 0; kt < RT; ++kt) fetch_a(ru, o, rt, kt);
#pragma unroll
        for (int e = 0; e < RT * 4 * HS; ++e) fetch_v(rv, o, e);
    };
    auto input = [&](const uint32_t (&w)[IS == 8 ? 2 : 1]) -> TS {
        if constexpr (IS == 8) {
            const gm_u32x2 u = {w[0], w[1]};
            return static_cast<TS>(__builtin_bit_cast(double, u));
        } else if constexpr (IS == 4) {
            return static_cast<TS>(__uint_as_float(w[0]));
        } else {
            return static_cast<TS>(p.in.code == MOGT_BF16
                                       ? __uint_as_float(w[0] << 16)
                                       : static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w[0]))));
        }
    };

    // acc is the state after a step; the rows past R stay zero (an infinite state
    // times the zeros of U's padding would leave NaN there, which the next step
    // would multiply into every row)
    auto take = [&](const vec (&acc)[RT][CW]) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int h = 0; h < CW; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    X[rt][h][i] = UA == GM_U16_FULL || rt < RT - 1 || trow(rt, i) < R ? acc[rt][h][i] : TS(0);
    };

    Ops ring[PD];
#pragma unroll
    for (int pp = 0; pp < PD; ++pp) fetch(pp, ring[pp]);
    if constexpr (SPREAD) {
        // Two tiles per wave: memory instructions between the MFMAs, which a burst
        // of them after a step's last would leave idle.  While contraction tile kt
        // runs, the inputs of step s + PD (kt = 0) or its transition's tile kt - 1,
        // whose registers are free by then, and the stores of the state before this
        // step.  With one tile per wave the memory bounds the pass where it fills
        // the chip, and the order above it reads and writes in (R = C = 64, 64 x
        // 512 steps: OUTPUT 437 us) was better than this one (467 us).
        constexpr int NV = RT * 4 * HS, TM = 4 * RT * CW;              // input loads; MFMAs per contraction tile
        constexpr int NS = OUT == GM_EVERY_HP ? 2 * NV : OUT == GM_EVERY_H ? NV : 0, SM = (RT - 1) * TM;
        static_assert(NS <= SM && NV <= TM && RT <= TM, "one of each a slot");
        int s0 = 0;
        for (; s0 < len; s0 += PD) {
#pragma unroll
            for (int pp = 0; pp < PD; ++pp) {
                const int s = s0 + pp;
                Ops& o = ring[pp];
                vec acc[RT][CW];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int h = 0; h < CW; ++h)
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[rt][h][i] = input(o.v[rt][h][i]);
                const auto ru = rsrc_u(s + PD), rv = rsrc_v(s + PD);
                fu += du;
                fv += dv;
                const bool st = s > 0 && s <= len;
                const auto rh = rsrc(oh - dh, NS > 0 && st ? hBytes : 0u);
                const auto rp = rsrc(op - dp, NS > NV && st ? pBytes : 0u);
#pragma unroll
                for (int kt = 0; kt < RT; ++kt)
#pragma unroll
                    for (int m = 0; m < TM; ++m) {
                        const int kk = m / (RT * CW), rt = m / CW % RT, h = m % CW;
                        acc[rt][h] = M::mma(o.A[rt][kt][kk], X[kt][h][kk], acc[rt][h]);
                        if (kt == 0) {
                            if ((m + 1) * NV / TM > m * NV / TM) fetch_v(rv, o, m * NV / TM);
                        } else {
                            if ((m + 1) * RT / TM > m * RT / TM) fetch_a(ru, o, m * RT / TM, kt - 1);
                            const int q = (kt - 1) * TM + m, e = q * NS / SM;
                            if (NS > 0 && (q + 1) * NS / SM > e) {
                                if (e < NV) store_piece(rh, offH, hrow, MOGT_F32, e, true);
                                else store_piece(rp, offP, prow, MOGT_F32, e - NV, true);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) fetch_a(ru, o, rt, RT - 1);
                take(acc);
                oh += dh;
                op += dp;
            }
        }
        // the state after the last step (not a padding step's)
        if constexpr (OUT == GM_EVERY_H) store_state(oh - dh, op - dp, s0 == len, true, YES, NO);
        if constexpr (OUT == GM_EVERY_HP) store_state(oh - dh, op - dp, s0 == len, true, YES, YES);
        if constexpr (OUT == GM_FINAL) store_any(out_at(p.out_h, j, ob_h), out_at(p.out_p, j, ob_p), false);
        return;
    }
    for (int s0 = 0; s0 < len; s0 += PD) {
#pragma unroll
        for (int pp = 0; pp < PD; ++pp) {
            const int s = s0 + pp;
            Ops& o = ring[pp];
            vec acc[RT][CW];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int h = 0; h < CW; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[rt][h][i] = input(o.v[rt][h][i]);
            // K-step-major: consecutive MFMAs belong to different tiles
#pragma unroll
            for (int kt = 0; kt < RT; ++kt)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                        for (int h = 0; h < CW; ++h) acc[rt][h] = M::mma(o.A[rt][kt][kk], X[kt][h][kk], acc[rt][h]);
            // the chunk's final state is its last step's, not a padding step's
            if constexpr (ANY) {
                if (s >= len) break;   // uniform
            }
            take(acc);
            fetch(s + PD, o);
            if constexpr (ANY) {
                if (p.every) store_any(oh, op, p.stream);
            } else if constexpr (OUT == GM_EVERY_H) {
                store_state(oh, op, s < len, true, YES, NO);
            } else if constexpr (OUT == GM_EVERY_HP) {
                store_state(oh, op, s < len, true, YES, YES);
            }
            oh += dh;
            op += dp;
        }
    }
    if (OUT == GM_FINAL || (ANY && !p.every)) store_any(out_at(p.out_h, j, ob_h), out_at(p.out_p, j, ob_p), false);
}

// Steps of a chunk: the power of two (or the whole sequence, in one pass) that
// makes the three passes' serial time the least.  A wave's step is its MFMAs plus
// about 200 cycles of issue and waits, counted per single 16-column tile and SIMD;
// LOCAL carries C + R columns, CARRY and OUTPUT Wo.  In the general form (io types
// other than the state's) a step of an unloaded SIMD does not go below its memory
// latency, which that form exposes: 0.36 to 0.9 us for 1 to 4 row tiles.  Without
// that floor many narrow sequences ran as one chunk each: R = 64, C = 1, 16 x 512
// steps, bf16 io 723 us (scalar kernel 511), R = 1, C = 1000, 4 x 4000 steps, fp16
// io 1060 -> 413 us; over 636 shapes the mean distance from the best length of
// chunk fell from 4.8 to 1.0 %.
inline int64_t gm_segment(int64_t B, int64_t L, int64_t R, int64_t C, int64_t Wo, bool f64, bool native) {
    const int64_t rt = (R + 15) / 16, simds = 1024;
    const double step = static_cast<double>(rt * rt * 4) * (f64 ? 64 : 32) + 200.0;
    const double floors[4] = {750.0, 1160.0, 1640.0, 1920.0};   // cycles
    const double floor = native ? 0.0 : floors[rt - 1];
    const int64_t tl = (C + R + 15) / 16, to = (Wo + 15) / 16;
    auto rounds = [&](int64_t waves) { return static_cast<double>((waves + simds - 1) / simds); };
    auto pass = [&](int64_t waves, int64_t steps) {
        const double busy = rounds(waves) * step;
        return static_cast<double>(steps) * (busy > floor ? busy : floor);
    };
    int64_t best = L;
    double least = pass(B * to, L);
    for (int64_t seg = 16; seg < L && seg <= 1024; seg *= 2) {
        const int64_t nch = (L + seg - 1) / seg;
        // the carries (always native): one chain, or three of about sqrt(nch) steps
        const double one = rounds(B * to) * static_cast<double>(nch) * step;
        const double nested = 3.0 * rounds(B * to) * sqrt(static_cast<double>(nch)) * step + 2.0e4;
        const double t = pass(B * nch * tl, seg) + pass(B * nch * to, seg) + (one < nested ? one : nested) +
                         2.0e4;   // 2e4 cycles: two more launches
        if (t < least) {
            least = t;
            best = seg;
        }
    }
    return best;
}

// Whether every step's blocks fit the kernel's 32-bit offsets; row: the longest
// row of the views in elements.  A lane forms the offsets of all 16 RT padded
// rows (and GM_OOB plus them), so it is their extent that must not wrap: a
// wrapped offset of a padded row would lie inside the range again.
inline bool gm_fits(int64_t R, int64_t row) {
    return R <= GM_MAX_R && row <= GM_MAX_BLOCK && (R + 15) / 16 * 16 * row * 8 <= GM_MAX_BLOCK;
}

template <typename TS, int RT, int CW, int IS, int UA, int OUT, bool P2 = false>
int gm_launch_k(const GParams& p, int64_t waves, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((waves + GM_WAVES - 1) / GM_WAVES)), block(64 * GM_WAVES);
    hipLaunchKernelGGL((generic_mfma_kernel<TS, RT, CW, IS, UA, OUT, P2>), grid, block, 0, st, p, waves);
    return check_launch("generic_mfma_kernel");
}

// the native form
template <typename TS, int RT, int CW, int UA, bool P2>
int gm_launch_out(const GParams& p, int64_t waves, hipStream_t st) {
    constexpr int SS = static_cast<int>(sizeof(TS));
    if (!p.every) return gm_launch_k<TS, RT, CW, SS, UA, GM_FINAL, P2>(p, waves, st);
    if (!p.out_p.p) return gm_launch_k<TS, RT, CW, SS, UA, GM_EVERY_H, P2>(p, waves, st);
    return gm_launch_k<TS, RT, CW, SS, UA, GM_EVERY_HP, P2>(p, waves, st);
}

// the general form
template <typename TS, int RT, int UA>
int gm_launch_any(const GParams& p, int64_t waves, hipStream_t st) {
    switch (p.in.code) {
        case MOGT_F64: return gm_launch_k<TS, RT, 1, 8, UA, GM_ANY>(p, waves, st);
        case MOGT_F32: return gm_launch_k<TS, RT, 1, 4, UA, GM_ANY>(p, waves, st);
        default: return gm_launch_k<TS, RT, 1, 2, UA, GM_ANY>(p, waves, st);
    }
}

template <typename TS, int RT, int CW>
int gm_launch(const GParams& p, int64_t waves, hipStream_t st) {
    constexpr int SS = static_cast<int>(sizeof(TS)), code = SS == 8 ? MOGT_F64 : MOGT_F32;
    constexpr int PD = gm_depth<TS, RT>();
    const bool native = (p.in.code == code || p.cin == 0) && p.out_h.code == code && (!p.out_p.p || p.out_p.code == code);
    const int64_t align = 16 / SS;
    const bool va = !p.rev && p.R % 4 == 0 && p.tr.rs % align == 0 && p.tr.ss % align == 0 && p.tr.bs % align == 0 &&
                    p.tr_c0 % align == 0 && reinterpret_cast<uintptr_t>(p.tr.p) % 16 == 0;
    // the native form's final state is that of a whole chunk; the last chunk's,
    // which no other chunk takes, may be ragged
    if (!native || (!p.every && p.seg % PD != 0)) {
        if constexpr (CW > 1) {
            return set_error(MOGT_E_INVALID, "generic scan: form not built");   // not reached: generic_mfma_launch
        } else {
            // 16-byte loads of U where the number of loads bounds the step (R = 64, C = 1,
            // 16 x 512 steps, bf16 io: 723 us by element, 357 so; the scalar kernel 511)
            if constexpr (SS == 4 && RT >= 3) {
                if (va) return gm_launch_any<TS, RT, GM_U16>(p, waves, st);
            }
            return gm_launch_any<TS, RT, GM_U1>(p, waves, st);
        }
    }
    const bool full = va && p.R == 16 * RT;
    if constexpr (SS == 4 && CW == 2) {
        auto even = [](const GView& v) {
            return !v.p || ((v.rs | v.ss | v.bs) % 2 == 0 && reinterpret_cast<uintptr_t>(v.p) % 8 == 0);
        };
        if (va && (p.cin | p.csplit | p.W) % 2 == 0 && even(p.in) && even(p.out_h) && even(p.out_p))
            return full ? gm_launch_out<TS, RT, CW, GM_U16_FULL, true>(p, waves, st)
                        : gm_launch_out<TS, RT, CW, GM_U16, true>(p, waves, st);
    }
    if (full) return gm_launch_out<TS, RT, CW, GM_U16_FULL, false>(p, waves, st);
    if (va) return gm_launch_out<TS, RT, CW, GM_U16, false>(p, waves, st);
    return gm_launch_out<TS, RT, CW, GM_U1, false>(p, waves, st);
}

// Tiles per wave: every wave of a chunk reads the whole of U_t, so for fp32 ranks
// above 32 a wave takes two while that leaves each SIMD a wave (R = 64, C = 64, 24
// x 2048 steps, before the spread memory instructions: LOCAL 880 -> 520 us, OUTPUT
// 648 -> 540 us; four tiles spill and ran 550 and 900 us); else one (a shorter step, more waves).
inline int gm_tiles_per_wave(int64_t chunks, int tiles) {
    return tiles > 1 && chunks * ((tiles + 1) / 2) >= 1024 ? 2 : 1;
}

template <typename TS>
int generic_mfma_launch(GParams p, int64_t batch, hipStream_t st) {
    const int tiles = (p.W + 15) / 16;
    const bool native = sizeof(TS) == 4 && (p.in.code == MOGT_F32 || p.cin == 0) && p.out_h.code == MOGT_F32 &&
                        (!p.out_p.p || p.out_p.code == MOGT_F32) && (p.every || p.seg % 2 == 0);
    const int cw = native && p.R > 32 ? gm_tiles_per_wave(batch * p.nseg, tiles) : 1;
    p.ntile = (tiles + cw - 1) / cw;
    const int64_t waves = batch * p.nseg * p.ntile;
    if (waves <= 0) return MOGT_OK;
    if (waves > 0x7fffffffLL) return set_error(MOGT_E_INVALID, "generic scan: problem too large for one launch");
    if constexpr (sizeof(TS) == 4) {
        if (cw == 2) return p.R <= 48 ? gm_launch<TS, 3, 2>(p, waves, st) : gm_launch<TS, 4, 2>(p, waves, st);
    }
    if (p.R <= 16) return gm_launch<TS, 1, 1>(p, waves, st);
    if (p.R <= 32) return gm_launch<TS, 2, 1>(p, waves, st);
    if (p.R <= 48) return gm_launch<TS, 3, 1>(p, waves, st);
    return gm_launch<TS, 4, 1>(p, waves, st);
}

extern template int generic_mfma_launch<float>(GParams, int64_t, hipStream_t);
extern template int generic_mfma_launch<double>(GParams, int64_t, hipStream_t);

}  // namespace mogt
