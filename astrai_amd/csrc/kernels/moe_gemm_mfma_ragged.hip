// The bf16 grouped GEMMs for K (dim of the gate/up GEMM, dim_ffn of the down
// GEMM) that is a multiple of 8 but not of the 64-K step: the kernels of
// moe_gemm_mfma.hip, whose DMA then stages the last step's chunks past the end
// of a row from zeros (dma_16_or_zero). Built as a code object of its own,
// under namespace ragged: in one code object with the whole-step kernels, or
// with the select in them, those measured 0.4-0.8 % slower (16384 tokens at D
// 4096, F 14336; 333 at D 2048, F 1408) with the same K loops.
//
// Before, these shapes ran on the general FMA kernel: 1500 tokens at D 1000,
// F 2664, 8 experts, top-2 and a shared expert took 2350 us a layer, and 149 with
// their rows gathered (245 copied, before narrower tiles).
#define ASTRAI_MOE_RAGGED_K 1
#include "moe_gemm_mfma.hip"
