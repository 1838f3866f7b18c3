// The grouped GEMM for 4-bit codes with IEEE-half storage; the source is ggemm.hip.
#define TFM_GG_F16 1
#include "ggemm.hip"
