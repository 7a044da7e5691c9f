// FP32 Toeplitz passes of the lengths of set 1 (toeplitz_ct.h).
#include "toeplitz_ct.h"

namespace tc {

TC_FOR_TOEPLITZ_PLAIN_1(TC_TOEPLITZ_PLAIN_DEF)

}  // namespace tc
