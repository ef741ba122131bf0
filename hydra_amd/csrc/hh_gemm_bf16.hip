// hh_gemm_bf16.hip — the BF16 decode kernels (up_small, down_small), compiled apart from hh_gemm.hip's
// MXFP4 ones. See hh_gemm.hip.
#define HH_GEMM_BF16
#include "hh_gemm.hip"
