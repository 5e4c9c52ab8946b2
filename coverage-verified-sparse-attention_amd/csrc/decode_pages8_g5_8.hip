// Decode kernels of 8-token pages for GQA group sizes 5-8
// (decode_kernels.h): the launchers' explicit instantiations.
#include "decode_kernels.h"

namespace cvsa {
CVSA_PAGES8_INSTANTIATE(5)
CVSA_PAGES8_INSTANTIATE(6)
CVSA_PAGES8_INSTANTIATE(7)
CVSA_PAGES8_INSTANTIATE(8)
}  // namespace cvsa
