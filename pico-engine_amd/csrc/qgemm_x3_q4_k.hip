// Short-prompt products of Q4_K weights (qgemm_x3.h).
#include "qgemm_x3_launch.h"

namespace pe {
PE_X3_DEFINE(q4_k, PE_TYPE_Q4_K, PE_TYPE_Q6_K)
}  // namespace pe
