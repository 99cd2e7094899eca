// W-only streaming kernels (wq_streamk.h) for short K: int8, 8 chunks per wave
// (K <= 4096).
#include "wq_streamk.h"

TM_STREAMK_S(8, 1, 8)
TM_STREAMK_S(8, 2, 8)
TM_STREAMK_MN(8, 1, 8)
TM_STREAMK_MN(8, 2, 8)
