// The dgrad GEMMs for K (dim of dgrad_down, dim_ffn of dgrad_in) that is a
// multiple of 8 but not of the 64-K step: the kernels of moe_gemm_bwd.hip with
// the last step's activation chunks and weight rows past K staged from zeros,
// in a code object of its own as moe_gemm_mfma_ragged.hip.
#define ASTRAI_MOE_RAGGED_K 1
#include "moe_gemm_bwd.hip"
