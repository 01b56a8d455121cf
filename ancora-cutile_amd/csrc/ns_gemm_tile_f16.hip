// The kernels of ns_gemm_tile.hip on fp16 (FMT_TO_F16, FMT_F16), as a unit of their own: the two compile side by side.
#define ANC_NS_F16_UNIT
#include "ns_gemm_tile.hip"
