// Decode kernels of 8-token pages for GQA group sizes 9-12
// (decode_kernels.h): the launchers' explicit instantiations.
#include "decode_kernels.h"

namespace cvsa {
CVSA_PAGES8_INSTANTIATE(9)
CVSA_PAGES8_INSTANTIATE(10)
CVSA_PAGES8_INSTANTIATE(11)
CVSA_PAGES8_INSTANTIATE(12)
}  // namespace cvsa
