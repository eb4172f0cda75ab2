// The fitted tiles for FP8 operands: a translation unit of its own, so that the two halves of the kernels compile side by side.
#define DAXQ_FIT_FP8 1
#include "gemm_tile_fit.hip"
