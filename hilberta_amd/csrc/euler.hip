// Flow-matching Euler update of the FLUX latents, the step between two transformer evaluations
// (diffusers 0.36.0 FlowMatchEulerDiscreteScheduler.step inside the loop that reference
// hilberta/sampling_layout.py:20-148 wraps).
#include "common.h"
#include "../../include/hilberta_hip.h"

namespace hb {
namespace {

// Flow-matching Euler update: out = 16-bit(x + step * y) in fp32, the product rounded first as the
// torch sequence rounds it.  Eight values per thread; bound by its launch at FLUX latent sizes
// (2 MB at 2048 px, where the five torch passes took 5 us each).
template <bool F16>
__global__ __launch_bounds__(256) void euler_kernel(const uint16_t* x, const uint16_t* y, float step,
                                                    uint16_t* out, int64_t n) {
#pragma clang fp contract(off)
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i + 8 <= n) {
    float xv[8], yv[8];
    unpack8<F16>(*(const u32x4*)(x + i), xv);
    unpack8<F16>(*(const u32x4*)(y + i), yv);
#pragma unroll
    for (int k = 0; k < 8; ++k) xv[k] = xv[k] + step * yv[k];
    *(u32x4*)(out + i) = pack8<F16>(xv);
  } else {
    for (int64_t k = i; k < n; ++k)
      out[k] = from_f<F16>(to_f<F16>(x[k]) + step * to_f<F16>(y[k]));
  }
}

}  // namespace
}  // namespace hb

using namespace hb;

extern "C" int hb_euler_step(const void* x, const void* y, float step, void* out, int64_t n,
                             int32_t dtype, hb_stream_t stream) {
  HB_REQUIRE(n >= 0 && n < (1ll << 40), "n must be in [0, 2^40)");
  if (n == 0) return HB_OK;
  HB_REQUIRE(x && y && out, "null pointer argument");
  HB_REQUIRE(dtype == HB_DTYPE_BF16 || dtype == HB_DTYPE_F16, "dtype must be bf16 or fp16");
  HB_REQUIRE((((uintptr_t)x | (uintptr_t)y | (uintptr_t)out) & 15) == 0,
             "every pointer must be 16-byte aligned");
  const dim3 grid((unsigned)((n + 2047) / 2048)), block(256);
  if (dtype == HB_DTYPE_F16)
    hipLaunchKernelGGL(euler_kernel<true>, grid, block, 0, stream, (const uint16_t*)x, (const uint16_t*)y,
                       step, (uint16_t*)out, n);
  else
    hipLaunchKernelGGL(euler_kernel<false>, grid, block, 0, stream, (const uint16_t*)x, (const uint16_t*)y,
                       step, (uint16_t*)out, n);
  HB_HIP(hipGetLastError());
  return HB_OK;
}
