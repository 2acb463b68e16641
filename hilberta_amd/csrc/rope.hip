// FLUX rotary tables: cos and sin of every token's position angles, one launch.
//
// FluxPosEmbed (diffusers 0.36.0, called through the transformer that hilberta/flux_adapter.py
// wraps, whose image ids it permutes at :210-212) takes per axis the float64 angles
// pos * theta^(-2j/d), repeats each for its pair and rounds cos and sin to float32.  As torch
// passes that is about 45 launches of 2-7 us over tables that fit the caches: bound by launches,
// not by bytes.  Here a thread owns one pair column: it computes its frequency once (float64 pow)
// and walks ROWS consecutive tokens, so a token costs one float64 sincos and two 8-byte stores (a
// wave writes whole 512-byte rows of both tables).  With 16896 tokens (17.3 MB written) a 2048 px
// evaluation of a two-block transformer went from 7444 to 7263 us, and a 1024 px sampling step,
// where the launches also hold up the host, from 3079 to 2867 us.
#include "common.h"
#include "../../include/hilberta_hip.h"

namespace hb {
namespace {

constexpr int PAIRS = 64;  // columns 2j, 2j + 1 of a 128-wide row
// Tokens per thread: the pow is amortised over eight rows, and 16896 tokens still make 528
// workgroups of four waves (two per CU).
constexpr int ROWS = 8;

struct RopeArgs {
  const float* ids;  // [tokens, 3]
  float* cos;        // [tokens, 128]
  float* sin;
  int64_t tokens;
  int32_t pairs0, pairs01;  // pairs of axis 0, and of axes 0 and 1
  int32_t dim[3];
  double theta;
};

__global__ __launch_bounds__(256) void rope_kernel(RopeArgs a) {
#pragma clang fp contract(off)
  const int col = threadIdx.x & (PAIRS - 1);
  const int axis = col < a.pairs0 ? 0 : col < a.pairs01 ? 1 : 2;
  const int j = col - (axis == 0 ? 0 : axis == 1 ? a.pairs0 : a.pairs01);
  const int dim = axis == 0 ? a.dim[0] : axis == 1 ? a.dim[1] : a.dim[2];
  const double freq = 1.0 / pow(a.theta, (double)(2 * j) / (double)dim);
  const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * ROWS;
  float pos[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int64_t t = first + r < a.tokens ? first + r : a.tokens - 1;
    pos[r] = a.ids[t * 3 + axis];
  }
  for (int r = 0; r < ROWS; ++r) {
    if (first + r >= a.tokens) return;
    double s, c;
    sincos((double)pos[r] * freq, &s, &c);
    const float2 cc = make_float2((float)c, (float)c), ss = make_float2((float)s, (float)s);
    *(float2*)(a.cos + (first + r) * 2 * PAIRS + 2 * col) = cc;
    *(float2*)(a.sin + (first + r) * 2 * PAIRS + 2 * col) = ss;
  }
}

}  // namespace
}  // namespace hb

using namespace hb;

extern "C" int hb_rotary_tables(const float* ids, int64_t tokens, double theta,
                                const int32_t* axes_dim, float* cos, float* sin,
                                hb_stream_t stream) {
  HB_REQUIRE(tokens >= 0 && tokens < (1ll << 31), "tokens must be in [0, 2^31)");
  if (tokens == 0) return HB_OK;
  HB_REQUIRE(ids && axes_dim && cos && sin, "null pointer argument");
  int total = 0;
  for (int i = 0; i < 3; ++i) {
    HB_REQUIRE(axes_dim[i] >= 0 && axes_dim[i] <= 2 * PAIRS && axes_dim[i] % 2 == 0,
               "axis sizes must be even and non-negative");
    total += axes_dim[i];
  }
  HB_REQUIRE(total == 2 * PAIRS, "axis sizes must add up to 128 (got %d)", total);
  HB_REQUIRE(((uintptr_t)ids & 3) == 0 && ((uintptr_t)cos & 7) == 0 && ((uintptr_t)sin & 7) == 0,
             "ids must be 4-byte, cos and sin 8-byte aligned");
  RopeArgs a;
  a.ids = ids;
  a.cos = cos;
  a.sin = sin;
  a.tokens = tokens;
  a.pairs0 = axes_dim[0] / 2;
  a.pairs01 = (axes_dim[0] + axes_dim[1]) / 2;
  for (int i = 0; i < 3; ++i) a.dim[i] = axes_dim[i];
  a.theta = theta;
  const int64_t groups = (tokens + 4 * ROWS - 1) / (4 * ROWS);
  hipLaunchKernelGGL(rope_kernel, dim3((unsigned)groups), dim3(256), 0, stream, a);
  HB_HIP(hipGetLastError());
  return HB_OK;
}
