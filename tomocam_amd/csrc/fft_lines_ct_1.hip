// Line transforms of the lengths of set 1 (fft_lines_ct.h).
#include "fft_lines_ct.h"

namespace tc {

TC_FOR_LINE_LENGTHS_1(TC_LINE_OPS_DEF)

}  // namespace tc
