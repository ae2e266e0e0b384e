// Matrix-core chunk kernel of the generic affine scan, double state.
#include "generic_mfma.h"

namespace mogt {
template int generic_mfma_launch<double>(GParams, int64_t, hipStream_t);
}  // namespace mogt
