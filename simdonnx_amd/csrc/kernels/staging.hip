// Host staging on gfx950: the fp32 input / output windows of a session (pinned, mapped host memory) read
// and written by the kernels themselves, converted to and from the storage type on the way (the uploads
// around f32to16.comp / f16to32.comp, VkSession.cs:200-240, without the device copy between them).
//
// Bound by PCIe (57 GB/s each way on this host). A copy-engine transfer plus a conversion kernel pays the
// engine's start and two hand-overs between the engine and the compute queue, ~8 us each, and an fp32 pass
// over device memory. Host-timed from launch to wait on one MI355X, copy + conversion against these kernels:
//   in  (fp32 -> fp16):  1.0 MB 36.7 / 31.5 us,  5.9 MB 123 / 118 us,  11.1 MB 215 / 209 us,  30 MB 551 / 540 us
//   out (fp16 -> fp32):  1.0 MB 38.7 / 29.0 us,  5.9 MB 132 / 117 us,  11.1 MB 223 / 210 us,  30 MB 557 / 556 us
// Reading host memory wants few requests in flight over few distinct pages: 64 workgroups with two 16-byte
// loads per thread in flight (512 KiB) keep up with the copy engine at every size (a whole call with 64 / 256 /
// 512 MB going up: engine + conversion 1234 / 4847 / 9660 us, here 1207 / 4762 / 9505; fp32 1234 / 4829 / 9627 and 1214 /
// 4783 / 9597), 256 workgroups with eight take 245 us for the 11.1 MB. Writes are posted: 256 workgroups with four stores each.
#include "sox_device.h"

namespace {

template <typename A, typename B, int U>
__device__ __forceinline__ void stage_body(const sox_cvt_args& p) {
    typedef vec_t<A, 4> A4;
    typedef vec_t<B, 4> B4;
    const A* x = (const A*)p.x;
    B* y = (B*)p.y;
    const long tid = (long)blockIdx.x * 256 + threadIdx.x, threads = (long)gridDim.x * 256;
    // an arena plan may place a value anywhere: whole vectors only where both sides are aligned to them
    if (((uintptr_t)x % sizeof(A4)) | ((uintptr_t)y % sizeof(B4))) {
        for (long i = tid; i < p.count; i += threads) y[i] = (B)x[i];
        return;
    }
    const long n4 = p.count / 4;
    for (long b = (long)blockIdx.x * 256 * U + threadIdx.x; b < n4; b += threads * U) {
        A4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (b + u * 256 < n4) v[u] = ((const A4*)x)[b + u * 256];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (b + u * 256 < n4) ((B4*)y)[b + u * 256] = __builtin_convertvector(v[u], B4);  // to nearest even
    }
    if (tid < p.count % 4) y[n4 * 4 + tid] = (B)x[n4 * 4 + tid];
}

}  // namespace

// grid: min(64, ceil(count / 2048)) workgroups of 256
extern "C" __global__ void __launch_bounds__(256) sox_stage_in_f32(sox_cvt_args p) { stage_body<float, float, 2>(p); }
extern "C" __global__ void __launch_bounds__(256) sox_stage_in_f16(sox_cvt_args p) { stage_body<float, half_t, 2>(p); }
extern "C" __global__ void __launch_bounds__(256) sox_stage_in_bf16(sox_cvt_args p) { stage_body<float, bf16_t, 2>(p); }
// grid: min(256, ceil(count / 4096)) workgroups of 256
extern "C" __global__ void __launch_bounds__(256) sox_stage_out_f32(sox_cvt_args p) { stage_body<float, float, 4>(p); }
extern "C" __global__ void __launch_bounds__(256) sox_stage_out_f16(sox_cvt_args p) { stage_body<half_t, float, 4>(p); }
extern "C" __global__ void __launch_bounds__(256) sox_stage_out_bf16(sox_cvt_args p) { stage_body<bf16_t, float, 4>(p); }
