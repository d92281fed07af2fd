// bf16 twins of gemm_kt.hip.
#include "gemm_ring.h"

SOX_GEMM_KT(sox_gemm_kt_bf16_256x128_w8k64s2, bf16_t, 256, 128, 64, 64, 64, 2, 8, 1, 4, true)
SOX_GEMM_KT(sox_gemm_kt_bf16_128x128_k64s2, bf16_t, 128, 128, 64, 64, 64, 2, 4, 2, 4, false)
SOX_GEMM_KT(sox_gemm_kt_bf16_128x64_k64s2, bf16_t, 128, 64, 64, 64, 32, 2, 4, 3, 4, false)
SOX_GEMM_KT(sox_gemm_kt_bf16_64x64_k64s2, bf16_t, 64, 64, 64, 32, 32, 2, 4, 4, 4, false)
SOX_GEMM_KT(sox_gemm_kt_bf16_128x96_k32s2, bf16_t, 128, 96, 32, 32, 96, 2, 4, 3, 4, false)
SOX_GEMM_KT(sox_gemm_kt_bf16_64x64_k32s2, bf16_t, 64, 64, 32, 32, 32, 2, 4, 4, 4, false)
SOX_GEMM_KT(sox_gemm_kt_bf16_128x32_k32s2, bf16_t, 128, 32, 32, 32, 32, 2, 4, 4, 4, true)
