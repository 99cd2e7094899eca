// The pipelined matrix products for bf16 operands: mm_bf16_<a><b>_<tile>, each
// operand k- (k) or row-contiguous (r), the tile 64 RT x 64 CT.
#include "gemm_pipe.h"

// NS stages; W: waves per SIMD that the tile's LDS and accumulators leave room for
#define TM_MM(AN, BN, ARC, BRC, T, RT, CT, NS, W)                                           \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(W, W)))   \
      void mm_bf16_##AN##BN##_##T(MmParams p) {                                               \
    mm_body<mm::BF16, ARC, BRC, RT, CT, NS>(p);                                             \
  }
#define TM_MM_TILES(AN, BN, ARC, BRC)       \
  TM_MM(AN, BN, ARC, BRC, 44, 4, 4, 2, 1)   \
  TM_MM(AN, BN, ARC, BRC, 42, 4, 2, 3, 1)   \
  TM_MM(AN, BN, ARC, BRC, 22, 2, 2, 2, 2)   \
  TM_MM(AN, BN, ARC, BRC, 22d, 2, 2, 4, 1)  \
  TM_MM(AN, BN, ARC, BRC, 21, 2, 1, 3, 2)   \
  TM_MM(AN, BN, ARC, BRC, 11, 1, 1, 4, 2)
TM_MM_TILES(k, k, false, false)
TM_MM_TILES(k, r, false, true)
TM_MM_TILES(r, k, true, false)
TM_MM_TILES(r, r, true, true)
