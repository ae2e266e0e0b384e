// Instantiations of the decay-gradient scan (MODE_DIAG_GRAD, diag_kernel.h): the
// tiles of the default lists, outputs in the inputs' dtype; bf16 also writes G
// rounded to bf16 (the gradient of b).
//
// Bound by HBM: a, b and G in, da out (fp32).  At B = 1, L = 32768, D = 768 the
// pass takes 76 us (403 MB, 5.3 TB/s, the rate of a large copy); before, the
// gradient wrote the recomputed h (57 us), shifted it by a copy (14 + 37 us)
// and multiplied (43 us): forward and backward 266 -> 189 us.  The tiles are the
// forward's: at (2, 32, 32, 8) the stash of a and b frees the registers that h
// and the batches of G take (177 of 256 VGPRs).
#include "diag_kernel.h"

namespace mogt {

#define MOGT_GRAD_F32_TILES(X) X(2, 32, 32, 8) X(2, 32, 32, 4) X(2, 32, 16, 8) X(2, 32, 8, 16) X(1, 64, 32, 16) X(1, 64, 16, 16) X(1, 64, 8, 16)
#define MOGT_GRAD_BF16_TILES(X) X(4, 16, 16, 8) X(2, 32, 16, 8) X(2, 32, 8, 16) X(1, 64, 32, 16) X(1, 64, 16, 16) X(1, 64, 8, 16)

int diag_run_grad(const DiagParams& prm, const DiagTile& t, int in_dtype, hipStream_t st) {
    if (in_dtype == MOGT_BF16) {
#define MOGT_CASE(V_, F_, S_, W_)                                       \
    if (t.vec == V_ && t.lanes == F_ && t.steps == S_ && t.waves == W_) \
        return diag_launch<MODE_DIAG_GRAD, bf16_t, float, bf16_t, V_, F_, S_, W_, true>(prm, st);
        MOGT_GRAD_BF16_TILES(MOGT_CASE)
#undef MOGT_CASE
    } else {
#define MOGT_CASE(V_, F_, S_, W_)                                       \
    if (t.vec == V_ && t.lanes == F_ && t.steps == S_ && t.waves == W_) \
        return diag_launch<MODE_DIAG_GRAD, float, float, float, V_, F_, S_, W_, false>(prm, st);
        MOGT_GRAD_F32_TILES(MOGT_CASE)
#undef MOGT_CASE
    }
    return set_error(MOGT_E_INVALID, "diag scan gradient: tile (vec=%d, lanes=%d, steps=%d, waves=%d) not compiled",
                     t.vec, t.lanes, t.steps, t.waves);
}

}  // namespace mogt
