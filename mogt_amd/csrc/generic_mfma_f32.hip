// Matrix-core chunk kernel of the generic affine scan, float state.
#include "generic_mfma.h"

namespace mogt {
template int generic_mfma_launch<float>(GParams, int64_t, hipStream_t);
}  // namespace mogt
