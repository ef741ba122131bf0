// hh_gemm_mlx.hip — the MLX decode kernels (up_small, down_small), compiled apart from hh_gemm.hip's
// MXFP4 ones. See hh_gemm.hip.
#define HH_GEMM_MLX
#include "hh_gemm.hip"
