// The grouped GEMM for 8-bit codes with IEEE-half storage; the source is ggemm.hip.
#define TFM_GG_F16 1
#define TFM_GG_BITS 8
#include "ggemm.hip"
