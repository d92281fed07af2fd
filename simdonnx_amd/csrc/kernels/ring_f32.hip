// fp32 instances of the LDS-DMA ring (gemm_ring.h), 32 floats (128 bytes) of K per slice, on
// v_mfma_f32_32x32x2_f32: dense Gemm (K a multiple of 4) and implicit-GEMM conv (ic % 4 == 0). They run at
// three quarters of the fp32 matrix rate once every CU has a tile; below that the 32 x 32 tiles of
// conv_f32.hip spread the work over more CUs. Against the register-staged implicit GEMM they replace:
// 2000 x 1000 -> 1000 63.4 -> 45.9 us, 8192 x 512 -> 512 55 -> 45.5 us, conv 4x64x64 128 -> 128 3x3
// 72.5 -> 50.7 us.
#include "gemm_ring.h"

SOX_GEMM_KT(sox_gemm_f32_128x64_k32s2, float, 128, 64, 32, 64, 32, 2, 4, 3, 4, false)
SOX_GEMM_KT(sox_gemm_f32_64x64_k32s2, float, 64, 64, 32, 32, 32, 2, 4, 4, 4, false)
SOX_GEMM_KT(sox_gemm_f32_128x32_k32s2, float, 128, 32, 32, 32, 32, 2, 4, 4, 4, false)
SOX_CONV(sox_conv_f32_128x64_k32s2, float, 128, 64, 32, 64, 32, 2, 4, 3, 4)
SOX_CONV(sox_conv_f32_64x64_k32s4, float, 64, 64, 32, 32, 32, 4, 4, 2, 4)
SOX_CONV(sox_conv_f32_128x32_k32s2, float, 128, 32, 32, 32, 32, 2, 4, 4, 4)
