// Gated residual update + AdaLN modulation of the FLUX transformer blocks, one pass per row.
//
// The FLUX blocks the reference runs (diffusers 0.36.0 FluxTransformerBlock /
// FluxSingleTransformerBlock / AdaLayerNormContinuous, called through the transformer that
// hilberta/flux_adapter.py wraps) repeat, per token row of `hidden` values:
//   r   = x + gate * y                      (gated residual; torch.addcmul, one rounding)
//   n   = LayerNorm(r)                      (no affine, eps; fp32 statistics, rounded)
//   out = shift + n * (1 + scale)           (1 + scale rounded first, as torch adds in 16 bit)
// as three to five separate passes over the row.  This kernel does it in one: it reads x (and
// y), writes the new residual (optional, may be in place) and the modulated row.  One wave per
// row: 64 lanes x NV 16-byte vectors cover hidden = 512 * NV values, the statistics are two
// wave reductions (mean, then the centred sum of squares) with no LDS.  HBM-bound: 2 bytes per
// value for each of x, y, the residual and the output.  Past the cache size (CACHE_BYTES) the inputs
// and the residual, which is not read again before the next projections, bypass the caches, and the
// output, which the next projection reads at once, stays: 16384 rows of 3072 (403 MB) take 69.0 us, 5.8
// TB/s (77.8 us with all of them cached, 72.1 with none).
#include "common.h"
#include "../../include/hilberta_hip.h"

namespace hb {
namespace {

struct AdaArgs {
  const uint16_t* x;
  int64_t x_b, x_n;
  const uint16_t* y;  // null: no residual update
  int64_t y_b, y_n;
  const uint16_t* gate;
  int64_t gate_b;
  uint16_t* x_out;    // null: residual not stored
  int64_t xo_b, xo_n;
  const uint16_t* shift;
  const uint16_t* scale;
  int64_t mod_b;
  uint16_t* out;
  int64_t out_b, out_n;
  uint32_t rows;
  float inv_hidden, eps;
};

// Two row sets of one shape (the image and text rows of a double-stream block) share a launch: 512
// text rows alone are 6-9 us of a mostly idle chip (a two-block transformer at 1024 px 0.5-0.8 % faster).
// The first `rows0` of `total` rows are a[0]'s.
struct AdaPair {
  AdaArgs a[2];
  uint32_t rows0, total;
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

template <bool F16, int NV, bool STREAM, bool PAIR>
__global__ __launch_bounds__(256) void adaln_kernel(AdaPair p) {
#pragma clang fp contract(off)
  uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (row >= p.total) return;  // the whole wave leaves together
  // (a wave lives for one row, so a single set's operands are not made to wait for the choice: 2 % of
  // a 403 MB call)
  const bool second = PAIR && (uint32_t)uniform(row) >= p.rows0;
  const AdaArgs& a = p.a[second];
  if (second) row -= p.rows0;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t b = row / a.rows;
  const uint32_t i = row - b * a.rows;
  const uint16_t* xp = a.x + b * a.x_b + (int64_t)i * a.x_n + lane * 8;
  float r[NV][8];
  u32x4 raw[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) raw[v] = load_once<STREAM>((const u32x4*)(xp + v * 512));
  if (a.y) {
    const uint16_t* yp = a.y + b * a.y_b + (int64_t)i * a.y_n + lane * 8;
    const uint16_t* gp = a.gate + b * a.gate_b + lane * 8;
    u32x4 yr[NV], gr[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      yr[v] = load_once<STREAM>((const u32x4*)(yp + v * 512));
      gr[v] = *(const u32x4*)(gp + v * 512);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      float xv[8], yv[8], gv[8];
      unpack8<F16>(raw[v], xv);
      unpack8<F16>(yr[v], yv);
      unpack8<F16>(gr[v], gv);
#pragma unroll
      for (int k = 0; k < 8; ++k) r[v][k] = round_f<F16>(xv[k] + gv[k] * yv[k]);
    }
    if (a.x_out) {
      uint16_t* op = a.x_out + b * a.xo_b + (int64_t)i * a.xo_n + lane * 8;
#pragma unroll
      for (int v = 0; v < NV; ++v) store_once<STREAM>((u32x4*)(op + v * 512), pack8<F16>(r[v]));
    }
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v) unpack8<F16>(raw[v], r[v]);
  }
  float s = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int k = 0; k < 8; ++k) s += r[v][k];
  const float mean = wave_sum(s) * a.inv_hidden;
  float q = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float d = r[v][k] - mean;
      q += d * d;
    }
  const float rstd = __builtin_amdgcn_rsqf(wave_sum(q) * a.inv_hidden + a.eps);
  const uint16_t* sp = a.shift + b * a.mod_b + lane * 8;
  const uint16_t* cp = a.scale + b * a.mod_b + lane * 8;
  uint16_t* op = a.out + b * a.out_b + (int64_t)i * a.out_n + lane * 8;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    float sh[8], sc[8], o[8];
    unpack8<F16>(*(const u32x4*)(sp + v * 512), sh);
    unpack8<F16>(*(const u32x4*)(cp + v * 512), sc);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float n = round_f<F16>((r[v][k] - mean) * rstd);
      o[k] = sh[k] + n * round_f<F16>(1.f + sc[k]);
    }
    *(u32x4*)(op + v * 512) = pack8<F16>(o);
  }
}

template <bool F16, bool STREAM, bool PAIR>
int launch(const AdaPair& a, int nv, hipStream_t st) {
  const dim3 grid((a.total + 3) / 4), block(256);
  switch (nv) {
    case 1: hipLaunchKernelGGL((adaln_kernel<F16, 1, STREAM, PAIR>), grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL((adaln_kernel<F16, 2, STREAM, PAIR>), grid, block, 0, st, a); break;
    case 3: hipLaunchKernelGGL((adaln_kernel<F16, 3, STREAM, PAIR>), grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL((adaln_kernel<F16, 4, STREAM, PAIR>), grid, block, 0, st, a); break;
    case 6: hipLaunchKernelGGL((adaln_kernel<F16, 6, STREAM, PAIR>), grid, block, 0, st, a); break;
    case 8: hipLaunchKernelGGL((adaln_kernel<F16, 8, STREAM, PAIR>), grid, block, 0, st, a); break;
    default: set_error("hidden must be 512, 1024, 1536, 2048, 3072 or 4096"); return HB_EINVAL;
  }
  HB_HIP(hipGetLastError());
  return HB_OK;
}

template <bool F16, bool STREAM>
int launch_sets(const AdaPair& p, int nv, int count, hipStream_t st) {
  return count == 2 ? launch<F16, STREAM, true>(p, nv, st) : launch<F16, STREAM, false>(p, nv, st);
}

}  // namespace
}  // namespace hb

using namespace hb;

namespace {

// Operands of one row set, as the entry points take them.
struct Operands {
  const void *x, *y, *gate;
  void* x_out;
  const void *shift, *scale;
  void* out;
  int64_t x_b, x_n, y_b, y_n, gate_b, xo_b, xo_n, mod_b, out_b, out_n;
};

int modulate(int count, int32_t batch, const int32_t* rows, int32_t hidden, int32_t dtype, float eps,
             const Operands* sets, hipStream_t stream) {
  AdaPair p = {};
  int64_t total = 0, bytes = 0;
  bool repeats = false;
  for (int i = 0; i < count; ++i) {
    const Operands& o = sets[i];
    HB_REQUIRE(batch > 0 && rows[i] > 0, "batch and rows must be positive");
    total += (int64_t)batch * rows[i];
    HB_REQUIRE(total < (1ll << 31), "too many rows for one launch");
    HB_REQUIRE(hidden > 0 && hidden % 512 == 0, "hidden must be a multiple of 512 (got %d)", hidden);
    HB_REQUIRE(dtype == HB_DTYPE_BF16 || dtype == HB_DTYPE_F16, "dtype must be bf16 or fp16");
    HB_REQUIRE(eps > 0.f, "eps must be positive");
    HB_REQUIRE(o.x && o.shift && o.scale && o.out, "null pointer argument");
    HB_REQUIRE(!o.y || o.gate, "a residual update needs its gate");
    HB_REQUIRE(!o.x_out || o.y, "x_out is written only with a residual update");
    const void* ptrs[7] = {o.x, o.y, o.gate, o.x_out, o.shift, o.scale, o.out};
    for (int k = 0; k < 7; ++k)
      HB_REQUIRE(((uintptr_t)ptrs[k] & 15) == 0, "every pointer must be 16-byte aligned");
    const int64_t strides[10] = {o.x_b, o.x_n, o.y_b, o.y_n, o.gate_b, o.xo_b, o.xo_n, o.mod_b, o.out_b, o.out_n};
    for (int k = 0; k < 10; ++k)
      HB_REQUIRE(strides[k] >= 0 && strides[k] % 8 == 0, "strides must be non-negative multiples of 8");
    // x (and y) in, the residual (when stored) and the rows out
    bytes += (int64_t)batch * rows[i] * hidden * 2 * (2 + (o.y != nullptr) + (o.x_out != nullptr));
    // one image for a batch, or one row for an image (x_n, y_n of 0), is read from the caches
    repeats |= (batch > 1 && (o.x_b == 0 || (o.y && o.y_b == 0))) || (rows[i] > 1 && (o.x_n == 0 || (o.y && o.y_n == 0)));
    AdaArgs& a = p.a[i];
    a.x = (const uint16_t*)o.x;
    a.x_b = o.x_b;
    a.x_n = o.x_n;
    a.y = (const uint16_t*)o.y;
    a.y_b = o.y_b;
    a.y_n = o.y_n;
    a.gate = (const uint16_t*)o.gate;
    a.gate_b = o.gate_b;
    a.x_out = (uint16_t*)o.x_out;
    a.xo_b = o.xo_b;
    a.xo_n = o.xo_n;
    a.shift = (const uint16_t*)o.shift;
    a.scale = (const uint16_t*)o.scale;
    a.mod_b = o.mod_b;
    a.out = (uint16_t*)o.out;
    a.out_b = o.out_b;
    a.out_n = o.out_n;
    a.rows = (uint32_t)rows[i];
    a.inv_hidden = 1.f / (float)hidden;
    a.eps = eps;
    if (i == 0) p.rows0 = (uint32_t)total;
  }
  p.total = (uint32_t)total;
  const int nv = hidden / 512;
  // (3072 wide, cached / past the caches: 12 x 4096 rows of one image 88 / 109 us, 6 x 4096 47 / 54;
  // 12288 rows and one row of y 38 / 48)
  const bool stream_in = bytes > CACHE_BYTES && !repeats;
  if (dtype == HB_DTYPE_F16)
    return stream_in ? launch_sets<true, true>(p, nv, count, stream) : launch_sets<true, false>(p, nv, count, stream);
  return stream_in ? launch_sets<false, true>(p, nv, count, stream) : launch_sets<false, false>(p, nv, count, stream);
}

}  // namespace

extern "C" int hb_adaln_modulate(int32_t batch, int32_t rows, int32_t hidden, int32_t dtype,
                                 float eps, const void* x, int64_t x_batch_stride,
                                 int64_t x_row_stride, const void* y, int64_t y_batch_stride,
                                 int64_t y_row_stride, const void* gate,
                                 int64_t gate_batch_stride, void* x_out,
                                 int64_t x_out_batch_stride, int64_t x_out_row_stride,
                                 const void* shift, const void* scale, int64_t mod_batch_stride,
                                 void* out, int64_t out_batch_stride, int64_t out_row_stride,
                                 hb_stream_t stream) {
  const Operands o = {x, y, gate, x_out, shift, scale, out, x_batch_stride, x_row_stride,
                      y_batch_stride, y_row_stride, gate_batch_stride, x_out_batch_stride,
                      x_out_row_stride, mod_batch_stride, out_batch_stride, out_row_stride};
  return modulate(1, batch, &rows, hidden, dtype, eps, &o, stream);
}

extern "C" int hb_adaln_modulate_pair(int32_t batch, const int32_t* rows, int32_t hidden,
                                      int32_t dtype, float eps, void* const* pointers,
                                      const int64_t* strides, hb_stream_t stream) {
  HB_REQUIRE(rows && pointers && strides, "null pointer argument");
  Operands o[2];
  for (int i = 0; i < 2; ++i) {
    void* const* q = pointers + 7 * i;
    const int64_t* s = strides + 10 * i;
    o[i] = {q[0], q[1], q[2], q[3], q[4], q[5], q[6], s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], s[9]};
  }
  return modulate(2, batch, rows, hidden, dtype, eps, o, stream);
}
