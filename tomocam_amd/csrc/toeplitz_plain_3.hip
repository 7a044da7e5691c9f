// FP32 Toeplitz passes of the lengths of set 3 (toeplitz_ct.h).
#include "toeplitz_ct.h"

namespace tc {

TC_FOR_TOEPLITZ_PLAIN_3(TC_TOEPLITZ_PLAIN_DEF)

}  // namespace tc
