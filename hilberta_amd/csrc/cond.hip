// Conditioning of the FLUX transformer: the linear layers whose input is a row or a few per call.
//
// The timestep, guidance and pooled-text embedders (diffusers 0.36.0 CombinedTimestepGuidanceText-
// ProjEmbeddings) and every block's AdaLN modulation (AdaLayerNormZero and its kin), inside the
// transformer hilberta/flux_adapter.py wraps, multiply 1..8 rows by [N, K] matrices: 0.11 GB per
// double-block stream, 6.4 GB over the 57 blocks.  Bound by the read of the weights.  The library
// GEMM takes 65 us per 113 MB matrix (1.75 TB/s: a 16 x 16 tile leaves most of the chip idle) and
// the passes around it about 40 launches of 2-5 us.  Here all modulations of a two-block model,
// 321 MB, take 52 us (6.2 TB/s) in one launch, of 57 blocks (6.49 GB, two launches) 0.95 ms (6.8 TB/s),
// and the embedders three launches.  With three to eight rows the products bound it instead.
//
//  * linear_rows_kernel: a wave owns ROWS (1 or 4) output columns and reads their weight rows
//    whole, 16 bytes per lane, with all ROWS loads of a step in flight; the input rows come from L1/L2 and
//    are unpacked once per step for all ROWS columns.  No LDS, no barrier: a wave's only tail is
//    the final cross-lane sum.  One launch takes up to MAX_LAYERS layers of any N and K, so all
//    modulations of a model stream back to back.
//  * Sums of layers (the three embedders) are rounded as the separate torch calls round: each
//    layer's output, then each addition.
#include "common.h"
#include "../../include/hilberta_hip.h"

namespace hb {
namespace {

constexpr int MAX_LAYERS = 64;  // layer descriptors per launch (48 bytes each: 3 KB of kernel arguments)

struct Layer {
  const uint16_t* x;     // [batch, k], rows x_stride apart
  const uint16_t* w;     // [n, k] contiguous
  const uint16_t* bias;  // [n] or null
  uint16_t* out;         // [batch, n] contiguous (of the last layer of a sum)
  int32_t x_stride, n, k, pad;
};

struct LinearArgs {
  Layer layer[MAX_LAYERS];
  int32_t outputs, batch, silu;
};

template <bool F16>
__device__ __forceinline__ float silu(float v) {
  return round_f<F16>(v / (1.f + expf(-v)));
}

// B input rows (the last ones repeat row batch - 1 and are not stored), SUM consecutive layers
// added into one output.
template <bool F16, int B, int SUM, int ROWS>
__global__ __launch_bounds__(256) void linear_rows_kernel(LinearArgs a) {
  const int lane = threadIdx.x & 63;
  int group = uniform(blockIdx.x * 4 + (threadIdx.x >> 6));
  int o = 0;
  for (; o < a.outputs; ++o) {
    const int groups = (a.layer[o * SUM].n + ROWS - 1) / ROWS;
    if (group < groups) break;
    group -= groups;
  }
  if (o == a.outputs) return;
  const int n = a.layer[o * SUM].n;
  float total[ROWS][B];
#pragma unroll
  for (int s = 0; s < SUM; ++s) {
    const Layer& l = a.layer[o * SUM + s];
    const uint16_t* w[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) w[r] = l.w + (int64_t)min(group * ROWS + r, n - 1) * l.k;
    float acc[ROWS][B];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int b = 0; b < B; ++b) acc[r][b] = 0.f;
#pragma unroll 2
    for (int k = lane * 8; k < l.k; k += 512) {
      u32x4 raw[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) raw[r] = __builtin_nontemporal_load((const u32x4*)(w[r] + k));
      float x[B][8];
#pragma unroll
      for (int b = 0; b < B; ++b)
        unpack8<F16>(*(const u32x4*)(l.x + (int64_t)min(b, a.batch - 1) * l.x_stride + k), x[b]);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        float wv[8];
        unpack8<F16>(raw[r], wv);
#pragma unroll
        for (int b = 0; b < B; ++b)
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[r][b] = __builtin_fmaf(wv[i], x[b][i], acc[r][b]);
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const float bias = l.bias ? to_f<F16>(l.bias[min(group * ROWS + r, n - 1)]) : 0.f;
#pragma unroll
      for (int b = 0; b < B; ++b) {
        float v = acc[r][b];
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
        v = round_f<F16>(v + bias);
        total[r][b] = s == 0 ? v : round_f<F16>(total[r][b] + v);
      }
    }
  }
  // every lane holds every sum: lane b * ROWS + r stores column r of row b
  uint16_t* out = a.layer[o * SUM + SUM - 1].out;
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const float v = a.silu ? silu<F16>(total[r][b]) : total[r][b];
      if (lane == b * ROWS + r && b < a.batch && group * ROWS + r < n)
        out[(int64_t)b * n + group * ROWS + r] = from_f<F16>(v);
    }
}

// Sinusoidal embeddings of up to two sets of scalars (diffusers get_timestep_embedding with
// flip_sin_to_cos and no frequency shift): row b of set s is [cos | sin] of
// (1000 t_b) * 10000^(-j / half), the product 1000 t_b in the 16-bit type as the model scales it.
template <bool F16>
__global__ __launch_bounds__(256) void sinusoid_kernel(const uint16_t* t0, const uint16_t* t1, int batch,
                                                       int half, uint16_t* out) {
#pragma clang fp contract(off)
  const int row = blockIdx.x, b = row % batch;
  const float t = round_f<F16>(to_f<F16>((row < batch ? t0 : t1)[b]) * 1000.f);
  for (int j = threadIdx.x; j < half; j += 256) {
    const float angle = t * expf(-9.210340371976184f * (float)j / (float)half);
    out[(int64_t)row * 2 * half + j] = from_f<F16>(cosf(angle));
    out[(int64_t)row * 2 * half + half + j] = from_f<F16>(sinf(angle));
  }
}

template <bool F16, int SUM, int ROWS>
void launch_linear(const LinearArgs& a, hipStream_t st) {
  int64_t waves = 0;
  for (int o = 0; o < a.outputs; ++o) waves += (a.layer[o * SUM].n + ROWS - 1) / ROWS;
  const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
  if (a.batch == 1) hipLaunchKernelGGL((linear_rows_kernel<F16, 1, SUM, ROWS>), grid, block, 0, st, a);
  else if (a.batch == 2) hipLaunchKernelGGL((linear_rows_kernel<F16, 2, SUM, ROWS>), grid, block, 0, st, a);
  else if (a.batch <= 4) hipLaunchKernelGGL((linear_rows_kernel<F16, 4, SUM, ROWS>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((linear_rows_kernel<F16, 8, SUM, ROWS>), grid, block, 0, st, a);
}

// Four columns per wave keep 64 bytes per lane in flight and share each unpacked input value; below
// NARROW columns that leaves CUs without a wave, and one column per wave is taken (the embedders'
// 3072-column sum of three layers: 21 us with four, 13 with one).
constexpr int64_t NARROW = 16384;

template <bool F16, int SUM>
void launch_rows(const LinearArgs& a, int64_t columns, hipStream_t st) {
  if (columns < NARROW) launch_linear<F16, SUM, 1>(a, st);
  else launch_linear<F16, SUM, 4>(a, st);
}

template <bool F16>
void launch_sum(const LinearArgs& a, int sum, int64_t columns, hipStream_t st) {
  if (sum == 1) launch_rows<F16, 1>(a, columns, st);
  else if (sum == 2) launch_rows<F16, 2>(a, columns, st);
  else launch_rows<F16, 3>(a, columns, st);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace
}  // namespace hb

using namespace hb;

extern "C" int hb_linear_rows(int32_t outputs, int32_t sum, int32_t batch, int32_t dtype,
                              int32_t silu, const void* const* x, const int64_t* x_strides,
                              const void* const* weights, const void* const* biases,
                              void* const* out, const int32_t* n, const int32_t* k,
                              hb_stream_t stream) {
  HB_REQUIRE(outputs >= 1 && sum >= 1 && sum <= 3 && (int64_t)outputs * sum <= MAX_LAYERS,
             "outputs and sum must be positive, sum at most 3, with at most %d layers", MAX_LAYERS);
  HB_REQUIRE(batch >= 1 && batch <= 8, "batch must be in [1, 8] (got %d)", batch);
  HB_REQUIRE(dtype == HB_DTYPE_BF16 || dtype == HB_DTYPE_F16, "dtype must be bf16 or fp16");
  HB_REQUIRE(x && x_strides && weights && biases && out && n && k, "null pointer argument");
  LinearArgs a = {};
  int64_t columns = 0;
  for (int o = 0; o < outputs; ++o) {
    HB_REQUIRE(n[o] >= 1 && out[o], "each output needs a column count and a pointer");
    HB_REQUIRE(((uintptr_t)out[o] & 1) == 0, "outputs must be 2-byte aligned");
    columns += n[o];
    for (int s = 0; s < sum; ++s) {
      const int i = o * sum + s;
      HB_REQUIRE(x[i] && weights[i], "null pointer argument");
      HB_REQUIRE(k[i] >= 8 && k[i] % 8 == 0, "k must be a positive multiple of 8 (got %d)", k[i]);
      HB_REQUIRE(x_strides[i] >= 0 && x_strides[i] % 8 == 0 && x_strides[i] < (1ll << 31),
                 "input row strides must be non-negative multiples of 8 below 2^31");
      HB_REQUIRE(aligned16(x[i]) && aligned16(weights[i]) && ((uintptr_t)biases[i] & 1) == 0,
                 "inputs and weights must be 16-byte aligned");
      a.layer[i].x = (const uint16_t*)x[i];
      a.layer[i].w = (const uint16_t*)weights[i];
      a.layer[i].bias = (const uint16_t*)biases[i];
      a.layer[i].out = (uint16_t*)out[o];
      a.layer[i].x_stride = (int32_t)x_strides[i];
      a.layer[i].n = n[o];
      a.layer[i].k = k[i];
    }
  }
  HB_REQUIRE(columns < (1ll << 31), "too many output columns for one launch");
  a.outputs = outputs;
  a.batch = batch;
  a.silu = silu;
  if (dtype == HB_DTYPE_F16) launch_sum<true>(a, sum, columns, stream);
  else launch_sum<false>(a, sum, columns, stream);
  HB_HIP(hipGetLastError());
  return HB_OK;
}

extern "C" int hb_sinusoid_rows(const void* t0, const void* t1, int32_t batch, int32_t dim,
                                int32_t dtype, void* out, hb_stream_t stream) {
  HB_REQUIRE(t0 && out, "null pointer argument");
  HB_REQUIRE(batch >= 1 && batch < (1 << 30) && dim >= 2 && dim % 2 == 0,
             "batch must be positive and dim even");
  HB_REQUIRE(dtype == HB_DTYPE_BF16 || dtype == HB_DTYPE_F16, "dtype must be bf16 or fp16");
  const dim3 grid(batch * (t1 ? 2 : 1)), block(256);
  const uint16_t *a = (const uint16_t*)t0, *b = (const uint16_t*)t1;
  if (dtype == HB_DTYPE_F16)
    hipLaunchKernelGGL(sinusoid_kernel<true>, grid, block, 0, stream, a, b, batch, dim / 2, (uint16_t*)out);
  else
    hipLaunchKernelGGL(sinusoid_kernel<false>, grid, block, 0, stream, a, b, batch, dim / 2, (uint16_t*)out);
  HB_HIP(hipGetLastError());
  return HB_OK;
}
