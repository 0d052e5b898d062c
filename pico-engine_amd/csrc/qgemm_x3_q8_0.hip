// Short-prompt products of Q8_0 weights (qgemm_x3.h).
#include "qgemm_x3_launch.h"

namespace pe {
PE_X3_DEFINE(q8_0, PE_TYPE_Q8_0, PE_TYPE_Q5_0)
}  // namespace pe
