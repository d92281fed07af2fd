// Dense fp16 Gemm instances of the LDS-DMA ring (gemm_ring.h) for a K that is a multiple of 8 but not of 64,
// the 1x1 convs over 16, 24, 40, 72 ... channels among them. Without them such products ran on the
// register-staged implicit GEMM: 4096 x 1000 -> 2000 66.2 -> 28.9 us, 786 x 760 -> 760 12.6 -> 7.8 us,
// 720 x 432 -> 360 10.4 -> 5.6 us. (A 256x192 tile would spill, and 256x128 is faster on 8192 x 760 -> 3000:
// 63 against 67 us.) 32-deep slices where a 64-deep one would be half zeros.
#include "gemm_ring.h"

SOX_GEMM_KT(sox_gemm_kt_f16_256x128_w8k64s2, half_t, 256, 128, 64, 64, 64, 2, 8, 1, 4, true)
SOX_GEMM_KT(sox_gemm_kt_f16_128x128_k64s2, half_t, 128, 128, 64, 64, 64, 2, 4, 2, 4, false)
SOX_GEMM_KT(sox_gemm_kt_f16_128x64_k64s2, half_t, 128, 64, 64, 64, 32, 2, 4, 3, 4, false)
SOX_GEMM_KT(sox_gemm_kt_f16_64x64_k64s2, half_t, 64, 64, 64, 32, 32, 2, 4, 4, 4, false)
SOX_GEMM_KT(sox_gemm_kt_f16_128x96_k32s2, half_t, 128, 96, 32, 32, 96, 2, 4, 3, 4, false)
SOX_GEMM_KT(sox_gemm_kt_f16_64x64_k32s2, half_t, 64, 64, 32, 32, 32, 2, 4, 4, 4, false)
// at most 32 columns, the projections to 16 .. 32 channels of large maps: 57600 x 96 -> 24 5.9 -> 4.5 us,
// 230400 x 16 -> 16 14.0 -> 7.7; stored through LDS (8.5 from registers)
SOX_GEMM_KT(sox_gemm_kt_f16_128x32_k32s2, half_t, 128, 32, 32, 32, 32, 2, 4, 4, 4, true)
