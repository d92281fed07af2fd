// Implicit-GEMM Conv2d / ConvTranspose instances of the LDS-DMA persistent ring (gemm_ring.h): fp16 NHWC,
// ic % 8 == 0, constant-0 or reflect padding.
#include "gemm_ring.h"

// few tiles: four stages of 64 or 32 input channels (32 where a 64-channel block would be half zeros)
SOX_CONV(sox_conv_f16_64x64_k32s4, half_t, 64, 64, 32, 32, 32, 4, 4, 2, 4)
SOX_CONV(sox_conv_f16_64x64_k64s4, half_t, 64, 64, 64, 32, 32, 4, 4, 2, 4)
// at most 32 output channels: a 64-wide tile multiplies at least half padding (1x1088x1920 16 -> 32 3x3 s2:
// 85.8 -> 42.3 us; 8x200x200 32 -> 16 3x3 s2: 18.0 -> 10.7; 4x128x128 24 -> 32 5x5: 25.4 -> 16.8)
SOX_CONV(sox_conv_f16_128x32_k32s2, half_t, 128, 32, 32, 32, 32, 2, 4, 4, 4)
// many tiles: two stages, two or three workgroups per CU; 96-wide tiles for 72..96, 168..192 .. channels
SOX_CONV(sox_conv_f16_128x64_k64s2, half_t, 128, 64, 64, 64, 32, 2, 4, 3, 4)
SOX_CONV(sox_conv_f16_128x96_k32s2, half_t, 128, 96, 32, 32, 96, 2, 4, 3, 4)
SOX_CONV(sox_conv_f16_128x96_k64s2, half_t, 128, 96, 64, 32, 96, 2, 4, 2, 4)
SOX_CONV(sox_conv_f16_128x128_k64s2, half_t, 128, 128, 64, 64, 64, 2, 4, 2, 4)
// ... many taps of few channels, where a 64-deep slice is half zeros (8x93x91 24 -> 112 5x5: 41 us, 56 on the 64x64
// tile that the estimate took without it)
SOX_CONV(sox_conv_f16_128x128_k32s4, half_t, 128, 128, 32, 64, 64, 4, 4, 2, 4)
// large convs (many output pixels, K >= 1024): the headline Gemm's 8-wave tilings, LDS-staged epilogue
SOX_CONV_E(sox_conv_f16_256x128_w8k64s2, half_t, 256, 128, 64, 64, 64, 2, 8, 1, 4)
// 256 output channels: the whole N in one tile (fewer DMA and LDS bytes per MFMA than 256 x 128); its
// LDS-staged epilogue would not fit beside the two 64 KiB stages, so it stores from registers. Each
// slice's DMA goes out in two parts (after the barrier and after the first k-step's MFMAs); its DMA
// rows hold 32-bit input offsets (the launcher routes inputs of fewer than 2^31 elements only)
SOX_CONV_L(sox_conv_f16_256x256_w8k64s2, half_t, 256, 256, 64, 128, 64, 2, 8, 1, 4, 2)
