// fast64.hip -- the specialised line kernels (fast.hip) for complex128, a
// translation unit of its own so that both precisions compile in parallel.
#define RFH_FAST_F64
#include "fast.hip"
