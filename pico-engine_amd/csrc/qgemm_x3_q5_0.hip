// Short-prompt products of Q5_0 weights (qgemm_x3.h).
#include "qgemm_x3_launch.h"

namespace pe {
PE_X3_DEFINE(q5_0, PE_TYPE_Q5_0, PE_TYPE_Q8_0)
}  // namespace pe
