// Decode kernels of 8-token pages for GQA group sizes 13-16
// (decode_kernels.h): the launchers' explicit instantiations.
#include "decode_kernels.h"

namespace cvsa {
CVSA_PAGES8_INSTANTIATE(13)
CVSA_PAGES8_INSTANTIATE(14)
CVSA_PAGES8_INSTANTIATE(15)
CVSA_PAGES8_INSTANTIATE(16)
}  // namespace cvsa
