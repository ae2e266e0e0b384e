// Generic dense affine scan  M_t = U_t M_{t-1} + [V_t | 0]  for any rank R <= 1024 and any
// number of channels, with the state carried in fp32 or fp64 (the reference scans'
// state_dtype argument, affine_scan.py:14-62, :127-172, :175-278).
//
// The MFMA pipeline of dense_scan.hip covers the model's shapes (R <= 32, fp32 state).
// This file covers everything else the reference's functions accept: a float64 state
// (the reference's own sanity check runs in float64, sanity_affine_scan.py:19-61), ranks
// above 32, fp16 / fp64 inputs and outputs.  Ranks up to 64 run on the matrix-core chunk
// kernel of generic_mfma.h; above, for wide states of ranks up to 4 (scalar_pays) and where
// a step's block exceeds its 32-bit offsets, on the scalar kernel below: every state element
// is one thread's running dot product over the R rows of the previous state, with the state
// in LDS.
//
// The prefix product U_prefix_t = U_t ... U_1 (return_prefix=True, affine_scan.py:43-55)
// is the same recurrence applied to R extra state columns that start at the identity and
// take no input, so one augmented state [H | U_prefix] of width C + R serves both.
//
// Three passes over chunks of `seg` steps (generic_geometry):
//   LOCAL   per chunk, from [0 | I]: the chunk's end state [E_j | P_j] (E_j: the
//           chunk's own contribution, P_j: the product of its transitions);
//   CARRY   M_in(j+1) = P_j M_in(j) + [E_j | 0], M_in(0) = [0 | I] (the carry recursion of
//           affine_scan.py:175-278): the same scan over the chunk summaries, in one pass or,
//           where that would be the longer chain, through these three passes once more;
//   OUTPUT  per chunk, from M_in(j): every step's state, written as H and U_prefix.
// One pass (OUTPUT from [0 | I]) when the whole sequence is one chunk.
//
// Reverse mode (the backward's total-gradient recursion, affine_scan.py:110-118):
// G_t = X_t + U_{t+1}^T G_{t+1}: position q of the scan is time L-1-q, its transition is
// U_{L-q}^T (the identity at q = 0, where the state is still zero).
#include "generic_mfma.h"

namespace mogt {
namespace {

constexpr int GS_THREADS = 256;
constexpr int GS_EPT = 4;                          // state elements per thread
constexpr int GS_MAX_ELEMS = GS_THREADS * GS_EPT;  // R * column-tile width
constexpr int GS_MAX_R = 1024;
constexpr int GS_STAGED_R = 16;                    // transitions staged in LDS up to this rank
constexpr int64_t GS_ONE_CHUNK = 16;               // steps up to which no workspace is asked for

// Row length in LDS of the staged transition and of a state column: R rounded
// up to 16 bytes, plus 16 bytes of skew between rows.
template <typename TS>
__host__ __device__ constexpr int gs_ld(int R) {
    return (R + static_cast<int>(16 / sizeof(TS)) - 1) / static_cast<int>(16 / sizeof(TS)) *
               static_cast<int>(16 / sizeof(TS)) + static_cast<int>(16 / sizeof(TS));
}

// PD: steps of operands in flight.  RM = 0: the threads read their rows of U_t from
// memory; else the rank is at most RM, U_t is staged through LDS (one value a
// thread) and the contraction is unrolled, its LDS reads issued together.
template <typename TS, int PD, int RM>
__global__ __launch_bounds__(GS_THREADS, sizeof(TS) == 4 ? 3 : 2) void generic_scan_kernel(GParams p) {
    extern __shared__ __align__(16) unsigned char gs_smem[];
    // LDS: the step's transition [R][ld] (staged form), then two state buffers
    // stored column-major, [Cb][ld]; ld = R rounded up to 16 bytes plus 16 bytes
    // of skew.  Padding columns / rows stay zero.
    static_assert(RM * RM <= GS_THREADS, "one value of U a thread");
    constexpr bool STAGED = RM > 0;
    constexpr int VE = 16 / static_cast<int>(sizeof(TS));
    const int R = p.R, Cb = p.Cb, RCb = R * Cb;
    const int ld = gs_ld<TS>(R);
    TS* sU = reinterpret_cast<TS*>(gs_smem);
    TS* sS = sU + (STAGED ? R * ld : 0);
    const int lds_elems = (STAGED ? R * ld : 0) + 2 * Cb * ld;
    for (int e = threadIdx.x; e < lds_elems; e += GS_THREADS) sU[e] = TS(0);
    __syncthreads();

    const int tid = threadIdx.x;
    int64_t blk = blockIdx.x;
    const int ct = static_cast<int>(blk % p.ntile);
    blk /= p.ntile;
    const int j = static_cast<int>(blk % p.nseg);
    const int64_t b = blk / p.nseg;
    const int64_t q0 = static_cast<int64_t>(j) * p.seg;
    const int64_t n = min(p.seg, p.L - q0);

    int oi[GS_EPT], ocl[GS_EPT], oc[GS_EPT];
    bool own[GS_EPT], ok[GS_EPT];
#pragma unroll
    for (int m = 0; m < GS_EPT; ++m) {
        const int e = tid + m * GS_THREADS;
        own[m] = e < RCb;
        oi[m] = own[m] ? e / Cb : 0;
        ocl[m] = own[m] ? e - oi[m] * Cb : 0;
        oc[m] = ct * Cb + ocl[m];
        ok[m] = own[m] && oc[m] < p.W;
    }

    // initial state (columns past W stay zero and are never written out)
    TS acc[GS_EPT];
#pragma unroll
    for (int m = 0; m < GS_EPT; ++m) {
        TS v0 = TS(0);
        if (ok[m]) {
            if (p.init.p) v0 = ld_code<TS>(p.init.p, at(p.init, b, j, oi[m], oc[m]), p.init.code);
            else if (oc[m] >= p.cid) v0 = (oi[m] == oc[m] - p.cid) ? TS(1) : TS(0);
            if (p.shift && j == 0) put<TS>(p, b, 0, oi[m], oc[m], v0);
        }
        acc[m] = v0;
        if (own[m]) sS[ocl[m] * ld + oi[m]] = v0;
    }

    // Operands of the next PD steps are in flight: slot pp of the ring holds
    // step s0 + pp of the current round and is refilled with step s0 + pp + PD
    // once its values have been consumed.
    TS ureg[PD];
    TS vreg[PD][GS_EPT];
    const int ur = tid / R, uc = tid - ur * R;   // the thread's value of U_t (staged form)
    auto fetch = [&](int64_t q, TS& u, TS (&v)[GS_EPT]) {
        // no transition enters the reversed position 0
        if (STAGED && ur < R)
            u = p.rev && q == 0 ? TS(0)
                                : static_cast<const TS*>(p.tr.p)[at(p.tr, b, p.rev ? p.L - q : q, ur, p.tr_c0 + uc)];
        const int64_t ti = p.rev ? p.L - 1 - q : q;
#pragma unroll
        for (int m = 0; m < GS_EPT; ++m)
            v[m] = (ok[m] && oc[m] < p.cin) ? ld_code<TS>(p.in.p, at(p.in, b, ti, oi[m], oc[m]), p.in.code)
                                            : TS(0);
    };

#pragma unroll
    for (int pp = 0; pp < PD; ++pp)
        if (pp < n) fetch(q0 + pp, ureg[pp], vreg[pp]);
    __syncthreads();
    int cur = 0;
    // one step: slot (u, v) holds step s; refilled with step s + PD
    auto step = [&](int64_t s, TS& u, TS (&v)[GS_EPT]) {
        const int64_t q = q0 + s;
        if (STAGED && ur < R) sU[p.rev ? uc * ld + ur : ur * ld + uc] = u;
        TS vin[GS_EPT];
#pragma unroll
        for (int m = 0; m < GS_EPT; ++m) vin[m] = v[m];
        if (s + PD < n) fetch(q + PD, u, v);   // later steps' loads overlap this step's arithmetic
        if constexpr (STAGED) __syncthreads();

        const TS* Sc = sS + cur * Cb * ld;
        TS* Sn = sS + (cur ^ 1) * Cb * ld;
        const bool ident = p.rev && q == 0;
        const int64_t tt = p.rev ? p.L - q : q;
        const int64_t tout = (p.rev ? p.L - 1 - q : q) + p.shift;
        // every element a thread owns sits in one column (the tile width
        // divides the thread count), so each state value read serves all
        const TS* scol = Sc + ocl[0] * ld;
        TS a[GS_EPT];
#pragma unroll
        for (int m = 0; m < GS_EPT; ++m) a[m] = vin[m];
        if (ident) {
#pragma unroll
            for (int m = 0; m < GS_EPT; ++m) a[m] += scol[oi[m]];
        } else if constexpr (STAGED) {
            typedef TS vec_t __attribute__((ext_vector_type(VE)));
#pragma unroll
            for (int k = 0; k < RM; k += VE) {
                if (k >= R) continue;
                const vec_t sv = *reinterpret_cast<const vec_t*>(scol + k);
#pragma unroll
                for (int m = 0; m < GS_EPT; ++m) {
                    const vec_t uv = *reinterpret_cast<const vec_t*>(sU + oi[m] * ld + k);
#pragma unroll
                    for (int e = 0; e < VE; ++e) a[m] += uv[e] * sv[e];
                }
            }
        } else {
            const TS* ut = static_cast<const TS*>(p.tr.p);
            for (int k = 0; k < R; ++k) {
                const TS sv = scol[k];
#pragma unroll
                for (int m = 0; m < GS_EPT; ++m) {
                    const int64_t ui = p.rev ? at(p.tr, b, tt, k, p.tr_c0 + oi[m]) : at(p.tr, b, tt, oi[m], p.tr_c0 + k);
                    a[m] += ut[ui] * sv;
                }
            }
        }
#pragma unroll
        for (int m = 0; m < GS_EPT; ++m) {
            if (!own[m]) continue;
            if (!ok[m]) a[m] = TS(0);
            else if (p.every) put<TS>(p, b, tout, oi[m], oc[m], a[m]);
            acc[m] = a[m];
            Sn[ocl[m] * ld + oi[m]] = a[m];
        }
        __syncthreads();
        cur ^= 1;
    };
    for (int64_t s0 = 0; s0 < n; s0 += PD) {
#pragma unroll
        for (int pp = 0; pp < PD; ++pp) {
            if (s0 + pp >= n) break;   // uniform over the work-group
            step(s0 + pp, ureg[pp], vreg[pp]);
        }
    }
    if (!p.every) {
#pragma unroll
        for (int m = 0; m < GS_EPT; ++m)
            if (ok[m]) put<TS>(p, b, j, oi[m], oc[m], acc[m]);
    }
}

// Level 0 is the sequence itself; a level above scans the chunk summaries of
// the one below (the carries).  Two levels above at most: the top one is one
// chunk per sequence.
constexpr int GS_LEVELS = 2;

// Whether the scalar kernel is the faster one at ranks of which the matrix tiles
// use few rows (a tile costs the same for 1 row as for 16): wide states over many
// steps, where throughput counts; with fewer columns or steps its barriers and LDS
// round trips do, and the matrix-core kernel is faster.  Matrix-core against
// scalar kernel: R = 1, C = 1000, 4 x 4000 steps: float64 611 against 277 us, fp16 io
// 414 against 197; R = 2, fp16 io, C = 500, 32 x 2000 955 against 442; R = 4, float64, C
// = 1000, 4 x 4000 696 against 646, 64 x 128 152 against 252; R = 1, float64, C = 64, 32
// x 2000 194 against 234; R = 2, fp16 io, C = 200, 4 x 4000 131 against 211.
bool scalar_pays(int64_t B, int64_t L, int64_t R, int64_t C, bool f64, bool native) {
    if (R < 1 || R > 4 || L <= GS_ONE_CHUNK) return false;
    const double columns = static_cast<double>(B) * static_cast<double>(C);
    const double values = columns * static_cast<double>(L);
    const bool large = values >= 1.6e7;
    if (f64 && native) {
        if (L < 48 && (R > 2 || values < 3.0e6)) return false;
        return values >= (R <= 2 ? 1.5e6 : 1.0e7) && (columns >= 2000.0 || large);
    }
    if (R == 1 && values >= 8.0e6 && L >= 48) return true;
    if (columns < 3000.0 || values < 1.5e6) return false;
    if (f64) return (R == 1 && L >= 48) || (R == 2 && L >= 100);
    if (R == 1) return L >= 48 || (L >= 24 && values >= 3.0e6);
    if (R == 2) return L >= 48 && (values >= 3.0e6 || (columns >= 6000.0 && L >= 100));
    return large && L >= 48 && (R == 3 || values >= 3.0e7);
}

struct GGeo {
    int64_t seg[GS_LEVELS], nch[GS_LEVELS];   // steps per chunk, chunks
    int levels;                               // levels cut into more than one chunk
    bool scalar;                              // every pass on the scalar kernel
    int Wl, Wo;          // LOCAL state width (C + R), OUTPUT / CARRY width (C + R if prefix)
    size_t s_off[GS_LEVELS], m_off[GS_LEVELS], bytes;
};

size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

// native: inputs and outputs in the state's dtype
GGeo geometry_of(int64_t B, int64_t L, int64_t R, int64_t C, int with_prefix, int state_code, bool native) {
    GGeo g{};
    g.Wl = static_cast<int>(C + R);
    g.Wo = static_cast<int>(C + (with_prefix ? R : 0));
    const size_t ts = state_code == MOGT_F64 ? 8 : 4;
    g.scalar = scalar_pays(B, L, R, C, state_code == MOGT_F64, native);
    const bool mfma = !g.scalar && gm_fits(R, C + R);
    size_t at = WS_HDR_BYTES;
    int64_t len = L;
    for (int l = 0; l < GS_LEVELS; ++l) {
        if (mfma) {
            g.seg[l] = gm_segment(B, len, R, C, g.Wo, state_code == MOGT_F64, native || l > 0);
        } else {
            if (l > 0) break;   // the scalar kernel's carries: one pass
            g.seg[l] = 16;
            while (g.seg[l] * g.seg[l] < len && g.seg[l] < 1024) g.seg[l] *= 2;
        }
        g.nch[l] = (len + g.seg[l] - 1) / g.seg[l];
        if (g.nch[l] <= 1) break;
        g.levels = l + 1;
        g.s_off[l] = at;
        g.m_off[l] = at + align256(static_cast<size_t>(B * g.nch[l] * R * g.Wl) * ts);
        at = g.m_off[l] + align256(static_cast<size_t>(B * g.nch[l] * R * g.Wo) * ts);
        len = g.nch[l] - 1;   // the last chunk's summary is not needed
    }
    return g;
}

// The geometry of a scan with these io types.  The workspace query knows the
// state's type only, so `bytes` has room for either form's chunks; and for those
// of a scan with and without the prefix, so that it grows with the prefix.
GGeo generic_geometry(int64_t B, int64_t L, int64_t R, int64_t C, int with_prefix, int state_code, bool native) {
    GGeo g = geometry_of(B, L, R, C, with_prefix, state_code, native);
    const size_t ts = state_code == MOGT_F64 ? 8 : 4;
    // callers bring room for two chunks' summaries beyond 16 steps, also where
    // one pass is the shorter chain
    int64_t most[GS_LEVELS] = {L > GS_ONE_CHUNK ? 2 : 0, 0};
    for (int form = 0; form < 4; ++form) {
        const GGeo f = geometry_of(B, L, R, C, form & 1, state_code, form & 2);
        for (int l = 0; l < f.levels; ++l) most[l] = f.nch[l] > most[l] ? f.nch[l] : most[l];
    }
    g.bytes = WS_HDR_BYTES;
    for (int l = 0; l < GS_LEVELS; ++l)
        g.bytes += align256(static_cast<size_t>(B * most[l] * R * g.Wl) * ts) +
                   align256(static_cast<size_t>(B * most[l] * R * g.Wo) * ts);
    return g;
}

int tile_width(int R, int W) {
    int cap = 1;   // a power of two dividing the thread count (one column per thread)
    while (cap * 2 * R <= GS_MAX_ELEMS && cap < GS_THREADS) cap *= 2;
    int cb = 1;
    while (cb < W && cb < cap) cb *= 2;
    return cb;
}

// Whether a pass takes the matrix-core kernel (rank <= 64).
bool takes_mfma(const GParams& p) {
    int64_t row = p.W;
    for (const GView* v : {&p.tr, &p.in, &p.out_h, &p.out_p}) row = v->rs > row ? v->rs : row;
    return !p.scalar && gm_fits(p.R, row);
}

template <typename TS>
int launch_generic(GParams p, int64_t batch, hipStream_t st, const char* what) {
    if (takes_mfma(p)) return generic_mfma_launch<TS>(p, batch, st);
    p.Cb = tile_width(p.R, p.W);
    p.ntile = (p.W + p.Cb - 1) / p.Cb;
    const int64_t blocks = batch * p.nseg * p.ntile;
    if (blocks <= 0) return MOGT_OK;
    if (blocks > 0x7fffffffLL) return set_error(MOGT_E_INVALID, "%s: problem too large for one launch", what);
    const bool staged = p.R <= GS_STAGED_R;
    const size_t lds = (2 * static_cast<size_t>(p.Cb) + (staged ? p.R : 0)) * gs_ld<TS>(p.R) * sizeof(TS);
    const dim3 grid(static_cast<unsigned>(blocks)), block(GS_THREADS);
    if (staged) hipLaunchKernelGGL((generic_scan_kernel<TS, 4, GS_STAGED_R>), grid, block, lds, st, p);
    else hipLaunchKernelGGL((generic_scan_kernel<TS, 2, 0>), grid, block, lds, st, p);
    return check_launch(what);
}

bool io_native(int64_t C, int v_code, int state_code, int out_code) {
    return (C == 0 || v_code == state_code) && out_code == state_code;
}

bool io_code(int c) { return c == MOGT_F32 || c == MOGT_BF16 || c == MOGT_F64 || c == MOGT_F16; }

// The scan `out` describes, at level l of the geometry: in one pass, or LOCAL
// over its chunks (state [H | P], the summaries), the carries as the exclusive
// scan of the summaries (one level up), then `out` from each chunk's carry.
// launch(pass, name): launches a pass, or checks it on the host.
template <typename Launch>
int scan_level(GParams out, const GGeo& g, int l, unsigned char* base, int state_code, const Launch& launch) {
    if (l >= g.levels) {
        out.seg = out.L; out.nseg = 1;
        return launch(out, "generic_scan output");
    }
    const int64_t R = out.R, nch = g.nch[l];
    const GView vS{base + g.s_off[l], nch * R * g.Wl, R * g.Wl, g.Wl, state_code};   // [B][nch][R][C+R]
    const GView vM{base + g.m_off[l], nch * R * g.Wo, R * g.Wo, g.Wo, state_code};   // [B][nch][R][Wo]
    const GView none{nullptr, 0, 0, 0, state_code};
    const int iC = out.cid;

    GParams loc = out;
    loc.seg = g.seg[l]; loc.nseg = static_cast<int>(nch);
    loc.init = none; loc.out_h = vS; loc.out_p = none;
    loc.W = g.Wl; loc.csplit = g.Wl; loc.every = 0; loc.shift = 0; loc.stream = 0;
    int rc = launch(loc, "generic_scan local");
    if (rc) return rc;

    GParams car{};
    car.tr = vS; car.in = vS; car.init = none; car.out_h = vM; car.out_p = none;
    car.L = nch - 1;
    car.R = out.R; car.W = g.Wo; car.tr_c0 = iC; car.cin = iC; car.cid = iC; car.csplit = g.Wo;
    car.every = 1; car.shift = 1; car.rev = 0; car.scalar = out.scalar;
    rc = scan_level(car, g, l + 1, base, state_code, launch);
    if (rc) return rc;

    out.seg = g.seg[l]; out.nseg = static_cast<int>(nch);
    out.init = vM;
    return launch(out, "generic_scan output");
}

template <typename Launch>
int run_passes(const void* U, const void* V, void* H, void* P, int64_t B, int64_t L, int64_t R, int64_t C,
               int v_code, int state_code, int out_code, int reverse, void* ws, const Launch& launch) {
    const GGeo g = generic_geometry(B, L, R, C, P != nullptr, state_code, io_native(C, v_code, state_code, out_code));
    const int iR = static_cast<int>(R), iC = static_cast<int>(C);
    // U / V / H / U_prefix views: [B][L][R][*]
    const GView vU{const_cast<void*>(U), L * R * R, R * R, R, state_code};
    const GView vV{const_cast<void*>(V), L * R * C, R * C, C, v_code};
    const GView vH{H, L * R * C, R * C, C, out_code};
    const GView vP{P, L * R * R, R * R, R, out_code};
    const GView none{nullptr, 0, 0, 0, state_code};
    unsigned char* base = static_cast<unsigned char*>(ws);

    GParams out{};   // the sequence's OUTPUT pass
    out.tr = vU; out.in = vV; out.init = none; out.out_h = vH; out.out_p = vP;
    out.L = L; out.R = iR; out.W = g.Wo; out.tr_c0 = 0; out.cin = iC; out.cid = iC; out.csplit = iC;
    out.every = 1; out.shift = 0; out.rev = reverse; out.stream = 1; out.scalar = g.scalar;
    return scan_level(out, g, 0, base, state_code, launch);
}

template <typename TS>
int run_generic(const void* U, const void* V, void* H, void* P, int64_t B, int64_t L, int64_t R, int64_t C,
                int v_code, int state_code, int out_code, int reverse, void* ws, hipStream_t st) {
    return run_passes(U, V, H, P, B, L, R, C, v_code, state_code, out_code, reverse, ws,
                      [&](const GParams& p, const char* what) { return launch_generic<TS>(p, B, st, what); });
}

int64_t code_size(int code) { return code == MOGT_F64 ? 8 : code == MOGT_F32 ? 4 : 2; }

// The matrix-core kernel's offsets of one view's step block, as the kernel
// forms them in 32 bits: rows below R and columns below `width` inside the
// range, every other (padded row, or GM_OOB for a column) past it.  The offsets
// rise with the column, so the ends of a row stand for it.
bool offsets_ok(const GView& v, int R, int64_t c0, int64_t width) {
    if (!v.p || width <= 0) return true;
    const int64_t es = code_size(v.code), range = (v.rs * (R - 1) + c0 + width) * es;
    if (range > GM_MAX_BLOCK) return false;
    const uint32_t row = static_cast<uint32_t>(v.rs) * static_cast<uint32_t>(es);
    for (int r = 0; r < (R + 15) / 16 * 16; ++r)
        for (int k = 0; k < 3; ++k) {
            const int64_t c = k == 0 ? c0 : c0 + width - 1;
            const uint32_t off = k == 2 ? GM_OOB : static_cast<uint32_t>(c * es);
            const uint32_t got = off + static_cast<uint32_t>(r) * row;
            const bool inside = got < static_cast<uint32_t>(range);
            if (inside != (k < 2 && r < R) || (inside && got != (r * v.rs + c) * es)) return false;
        }
    return true;
}

int check_generic(int64_t B, int64_t L, int64_t R, int64_t C, int v_code, int state_code, int out_code,
                  int reverse, const void* P) {
    if (B < 0 || L < 0 || R < 0 || C < 0) return set_error(MOGT_E_INVALID, "negative size");
    if (R == 0 && B > 0 && L > 0) return set_error(MOGT_E_INVALID, "rank must be positive");
    if (R > GS_MAX_R) return set_error(MOGT_E_INVALID, "rank %lld above the generic scan's limit %d",
                                       static_cast<long long>(R), GS_MAX_R);
    if (C + R > 0x3fffffffLL) return set_error(MOGT_E_INVALID, "too many channels");
    if (state_code != MOGT_F32 && state_code != MOGT_F64)
        return set_error(MOGT_E_INVALID, "state dtype must be MOGT_F32 or MOGT_F64");
    if (!io_code(v_code) || !io_code(out_code)) return set_error(MOGT_E_INVALID, "unsupported V or output dtype");
    if (reverse && P) return set_error(MOGT_E_INVALID, "the reverse scan has no prefix output");
    return MOGT_OK;
}

}  // namespace
}  // namespace mogt

using namespace mogt;

extern "C" size_t mogt_affine_scan_generic_workspace_bytes(int64_t batch, int64_t length, int64_t rank,
                                                          int64_t channels, int with_prefix, int state_dtype) {
    if (batch <= 0 || length <= 0 || rank <= 0 || rank > GS_MAX_R || channels < 0) return WS_HDR_BYTES;
    return generic_geometry(batch, length, rank, channels, with_prefix != 0, state_dtype, true).bytes;
}

extern "C" int mogt_affine_scan_generic_fwd(const void* U, const void* V, void* H, void* U_prefix, int64_t batch,
                                            int64_t length, int64_t rank, int64_t channels, int v_dtype,
                                            int state_dtype, int out_dtype, int reverse, void* workspace,
                                            size_t workspace_bytes, void* stream) {
    clear_error();
    int rc = check_generic(batch, length, rank, channels, v_dtype, state_dtype, out_dtype, reverse, U_prefix);
    if (rc) return rc;
    if (batch == 0 || length == 0 || (channels == 0 && !U_prefix)) return MOGT_OK;
    if (!U || (channels > 0 && (!V || !H))) return set_error(MOGT_E_INVALID, "null tensor pointer");
    const GGeo g = generic_geometry(batch, length, rank, channels, U_prefix != nullptr, state_dtype, true);
    if (length > GS_ONE_CHUNK && (!workspace || workspace_bytes < g.bytes))
        return set_error(MOGT_E_WORKSPACE, "workspace of %zu bytes needed", g.bytes);
    hipStream_t st = static_cast<hipStream_t>(stream);
    return state_dtype == MOGT_F64
               ? run_generic<double>(U, V, H, U_prefix, batch, length, rank, channels, v_dtype, state_dtype,
                                     out_dtype, reverse, workspace, st)
               : run_generic<float>(U, V, H, U_prefix, batch, length, rank, channels, v_dtype, state_dtype,
                                    out_dtype, reverse, workspace, st);
}

extern "C" int mogt_affine_scan_generic_check_offsets(int64_t batch, int64_t length, int64_t rank, int64_t channels,
                                                      int with_prefix, int v_dtype, int state_dtype, int out_dtype,
                                                      int reverse) {
    clear_error();
    void* some = reinterpret_cast<void*>(uintptr_t(256));   // views are told from absent ones; nothing is read
    void* P = with_prefix ? some : nullptr;
    if (int rc = check_generic(batch, length, rank, channels, v_dtype, state_dtype, out_dtype, reverse, P)) return rc;
    if (batch == 0 || length == 0 || (channels == 0 && !P)) return MOGT_OK;
    return run_passes(some, some, some, P, batch, length, rank, channels, v_dtype, state_dtype, out_dtype, reverse,
                      some, [](const GParams& p, const char* what) -> int {
                          if (!takes_mfma(p)) return MOGT_OK;
                          const bool ok = offsets_ok(p.tr, p.R, p.tr_c0, p.R) && offsets_ok(p.in, p.R, 0, p.cin) &&
                                          offsets_ok(p.out_h, p.R, 0, p.csplit) &&
                                          offsets_ok(p.out_p, p.R, 0, p.W - p.csplit);
                          return ok ? MOGT_OK : set_error(MOGT_E_INVALID, "%s: a 32-bit offset wraps", what);
                      });
}

extern "C" int mogt_affine_local_scan_generic(const void* U, const void* V, void* U_prefix, void* H_prefix,
                                              int64_t batch, int64_t length, int64_t rank, int64_t channels,
                                              int64_t block_size, int v_dtype, int state_dtype, int out_dtype,
                                              void* stream) {
    clear_error();
    int rc = check_generic(batch, length, rank, channels, v_dtype, state_dtype, out_dtype, 0, nullptr);
    if (rc) return rc;
    if (block_size <= 0) return set_error(MOGT_E_INVALID, "block_size must be positive");
    if (batch == 0 || length == 0) return MOGT_OK;
    if (!U || !U_prefix || (channels > 0 && (!V || !H_prefix))) return set_error(MOGT_E_INVALID, "null tensor pointer");
    const int64_t nb = (length + block_size - 1) / block_size;
    if (nb > 0x7fffffffLL) return set_error(MOGT_E_INVALID, "too many blocks");
    const int iR = static_cast<int>(rank), iC = static_cast<int>(channels);
    const GView none{nullptr, 0, 0, 0, state_dtype};
    GParams loc{};
    // one pass: every block from [0 | I], every step written (the OUTPUT pass
    // with no carries)
    loc.tr = GView{const_cast<void*>(U), length * rank * rank, rank * rank, rank, state_dtype};
    loc.in = GView{const_cast<void*>(V), length * rank * channels, rank * channels, channels, v_dtype};
    loc.init = none;
    loc.out_h = GView{H_prefix, length * rank * channels, rank * channels, channels, out_dtype};
    loc.out_p = GView{U_prefix, length * rank * rank, rank * rank, rank, out_dtype};
    loc.L = length; loc.seg = block_size; loc.nseg = static_cast<int>(nb);
    loc.R = iR; loc.W = iC + iR; loc.tr_c0 = 0; loc.cin = iC; loc.cid = iC; loc.csplit = iC;
    loc.every = 1; loc.shift = 0; loc.rev = 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return state_dtype == MOGT_F64 ? launch_generic<double>(loc, batch, st, "generic local scan")
                                   : launch_generic<float>(loc, batch, st, "generic local scan");
}
