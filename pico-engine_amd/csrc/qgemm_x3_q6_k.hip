// Short-prompt products of Q6_K weights (qgemm_x3.h).
#include "qgemm_x3_launch.h"

namespace pe {
PE_X3_DEFINE(q6_k, PE_TYPE_Q6_K, PE_TYPE_Q4_K)
}  // namespace pe
