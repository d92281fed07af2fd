// bf16 instances of the implicit-GEMM Conv2d / ConvTranspose ring (gemm_ring.h) for bf16 graphs: the
// tilings of the fp16 table (conv_ring.hip), v_mfma_f32_32x32x16_bf16, bf16 storage.
#include "gemm_ring.h"

SOX_CONV(sox_conv_bf16_64x64_k32s4, bf16_t, 64, 64, 32, 32, 32, 4, 4, 2, 4)
SOX_CONV(sox_conv_bf16_64x64_k64s4, bf16_t, 64, 64, 64, 32, 32, 4, 4, 2, 4)
SOX_CONV(sox_conv_bf16_128x32_k32s2, bf16_t, 128, 32, 32, 32, 32, 2, 4, 4, 4)
SOX_CONV(sox_conv_bf16_128x64_k64s2, bf16_t, 128, 64, 64, 64, 32, 2, 4, 3, 4)
SOX_CONV(sox_conv_bf16_128x96_k32s2, bf16_t, 128, 96, 32, 32, 96, 2, 4, 3, 4)
SOX_CONV(sox_conv_bf16_128x96_k64s2, bf16_t, 128, 96, 64, 32, 96, 2, 4, 2, 4)
SOX_CONV(sox_conv_bf16_128x128_k64s2, bf16_t, 128, 128, 64, 64, 64, 2, 4, 2, 4)
SOX_CONV(sox_conv_bf16_128x128_k32s4, bf16_t, 128, 128, 32, 64, 64, 4, 4, 2, 4)
SOX_CONV_E(sox_conv_bf16_256x128_w8k64s2, bf16_t, 256, 128, 64, 64, 64, 2, 8, 1, 4)
SOX_CONV_L(sox_conv_bf16_256x256_w8k64s2, bf16_t, 256, 256, 64, 128, 64, 2, 8, 1, 4, 2)
