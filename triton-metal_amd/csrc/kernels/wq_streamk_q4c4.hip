// W-only streaming kernels (wq_streamk.h) for short K: int4, 4 chunks per wave
// (K <= 4096).
#include "wq_streamk.h"

TM_STREAMK_S(4, 1, 4)
TM_STREAMK_S(4, 2, 4)
TM_STREAMK_MN(4, 1, 4)
TM_STREAMK_MN(4, 2, 4)
