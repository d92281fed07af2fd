// The smaller dense fp16 Gemm tilings of the LDS-DMA ring (gemm_ring.h): 4 waves, several workgroups per CU.
#include "gemm_ring.h"

SOX_GEMM(sox_gemm_f16_128x128_k64s2, half_t, 128, 128, 64, 64, 64, 2, 4, 2, 4)
SOX_GEMM(sox_gemm_f16_128x128_k32s4, half_t, 128, 128, 32, 64, 64, 4, 4, 2, 4)
// 128x64 with its epilogue through LDS: wide outputs over a short K are bound by their stores (16000 x 128 ->
// 256: 6.1 us against 6.9 from registers); 64x64, the tile of few workgroups and long K, is not
// (786 x 768 -> 760: 8.1 us with it, 6.8 without)
SOX_GEMM_E(sox_gemm_f16_128x64_k64s2e, half_t, 128, 64, 64, 64, 32, 2, 4, 3, 4)
SOX_GEMM(sox_gemm_f16_128x64_k64s2, half_t, 128, 64, 64, 64, 32, 2, 4, 3, 4)
SOX_GEMM(sox_gemm_f16_64x64_k64s2, half_t, 64, 64, 64, 32, 32, 2, 4, 4, 4)
// at most 32 columns (57600 x 128 -> 32: 5.9 -> 4.8 us)
SOX_GEMM(sox_gemm_f16_128x32_k64s2, half_t, 128, 32, 64, 32, 32, 2, 4, 3, 4)
SOX_GEMM_E(sox_gemm_f16_64x64_k64s4, half_t, 64, 64, 64, 32, 32, 4, 4, 2, 4)
SOX_GEMM(sox_gemm_f16_128x64_k64s4, half_t, 128, 64, 64, 64, 32, 4, 4, 1, 4)
// A rows through a LayerNorm folded into the Gemm (the default tilings)
SOX_GEMM_LN(sox_gemm_ln_f16_256x128_w8k64s2, half_t, 256, 128, 64, 64, 64, 2, 8, 1, 4, true)
SOX_GEMM_LN(sox_gemm_ln_f16_128x128_k64s2, half_t, 128, 128, 64, 64, 64, 2, 4, 2, 4, false)
SOX_GEMM_LN(sox_gemm_ln_f16_128x64_k64s2, half_t, 128, 64, 64, 64, 32, 2, 4, 3, 4, false)
SOX_GEMM_LN(sox_gemm_ln_f16_64x64_k64s2, half_t, 64, 64, 64, 32, 32, 2, 4, 4, 4, false)
