// The grouped GEMM for 8-bit codes with bf16 storage; the source is ggemm.hip.
#define TFM_GG_BITS 8
#include "ggemm.hip"
