// Decode kernels of 8-token pages for GQA group sizes 1-4
// (decode_kernels.h): the launchers' explicit instantiations.
#include "decode_kernels.h"

namespace cvsa {
CVSA_PAGES8_INSTANTIATE(1)
CVSA_PAGES8_INSTANTIATE(2)
CVSA_PAGES8_INSTANTIATE(3)
CVSA_PAGES8_INSTANTIATE(4)
}  // namespace cvsa
