// Token-dimension gather for the persistent Hilbert layout (permute / unpermute).
//
// Replaces the torch index_select calls of the reference at transformer entry and exit
// (hilberta/flux_adapter.py:209-212, :243) and around sampling (sampling_layout.py:96-97, :110):
//   dst[o, i, :] = src[o, index[i], :]   for o < outer, i < rows
// Each row is `row_bytes` contiguous bytes.  The copy moves 16-byte vectors, aligned where every
// pointer, stride and the row size allow it, and narrower ones only for rows shorter than that;
// consecutive threads walk consecutive vectors
// of one destination row, so both the gathered reads and the writes are coalesced.  This is an
// HBM-bound byte move: 2 * outer * rows * row_bytes plus the index reads per call.
#include "common.h"
#include "../../include/hilberta_hip.h"

namespace hb {
namespace {

template <int V>
struct Vec;
// 0: 16 bytes at any address, for rows of at least 16 bytes that no wider vector divides
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
template <> struct Vec<0> { typedef u32x4_any T; };
template <> struct Vec<16> { typedef u32x4 T; };
template <> struct Vec<8> { typedef u32x2 T; };
template <> struct Vec<4> { typedef uint32_t T; };
template <> struct Vec<2> { typedef uint16_t T; };
template <> struct Vec<1> { typedef uint8_t T; };

// I is the index type of the flat thread walk: 32-bit when the walk fits (cheap division).
template <int V, typename I, bool STREAM>
__global__ __launch_bounds__(256) void gather_rows_kernel(const char* __restrict__ src, char* __restrict__ dst,
                                   const int64_t* __restrict__ index, I rows, I outer,
                                   int64_t src_outer, int64_t dst_outer, int64_t src_row,
                                   int64_t dst_row, I vec_per_row, int64_t row_bytes,
                                   int64_t src_rows, int32_t* error) {
  typedef typename Vec<V>::T T;
  const I total = outer * rows * vec_per_row;
  for (I t = blockIdx.x * (I)blockDim.x + threadIdx.x; t < total; t += (I)gridDim.x * blockDim.x) {
    const I row = t / vec_per_row;
    const I v = t - row * vec_per_row;
    const I o = row / rows;
    const I r = row - o * rows;
    const int64_t s = index[r];
    if (s < 0 || s >= src_rows) {  // never read out of bounds; report instead
      if (error) atomicOr(error, 1);
      continue;
    }
    // (a ragged row's last vector ends with the row and repeats bytes of the one before it)
    const int64_t at = V ? (int64_t)v * V : (int64_t)v * 16 < row_bytes - 16 ? (int64_t)v * 16 : row_bytes - 16;
    const T* from = (const T*)(src + o * src_outer + s * src_row + at);
    T val;
    if constexpr (STREAM) val = __builtin_nontemporal_load(from);
    else val = *from;
    *(T*)(dst + o * dst_outer + r * dst_row + at) = val;
  }
}

template <int V, bool STREAM>
void launch_walk(unsigned blocks, const void* src, void* dst, const int64_t* index, int64_t rows,
                 int64_t outer, int64_t so, int64_t dso, int64_t sr, int64_t dr, int64_t vpr,
                 int64_t row_bytes, int64_t src_rows, int32_t* error, hipStream_t stream) {
  if (outer * rows * vpr + (int64_t)blocks * 256 < (int64_t)0xffffffffu) {
    hipLaunchKernelGGL((gather_rows_kernel<V, uint32_t, STREAM>), dim3(blocks), dim3(256), 0, stream,
                       (const char*)src, (char*)dst, index, (uint32_t)rows, (uint32_t)outer, so, dso,
                       sr, dr, (uint32_t)vpr, row_bytes, src_rows, error);
  } else {
    hipLaunchKernelGGL((gather_rows_kernel<V, uint64_t, STREAM>), dim3(blocks), dim3(256), 0, stream,
                       (const char*)src, (char*)dst, index, (uint64_t)rows, (uint64_t)outer, so, dso,
                       sr, dr, (uint64_t)vpr, row_bytes, src_rows, error);
  }
}

template <int V>
void launch_gather(const void* src, void* dst, const int64_t* index, int64_t rows, int64_t outer,
                   int64_t so, int64_t dso, int64_t sr, int64_t dr, int64_t row_bytes,
                   int64_t src_rows, int32_t* error, hipStream_t stream) {
  const int64_t vpr = V ? row_bytes / (V ? V : 1) : (row_bytes + 15) / 16;
  const int64_t total = outer * rows * vpr;
  // One vector per thread and one pass for every size up to 2^28 vectors: a grid capped at a few
  // workgroups per CU with a grid-stride loop measured 9-11 % slower on 100-400 MB gathers (the
  // last pass leaves most CUs idle); beyond 2^20 workgroups the loop strides.
  int64_t blocks = (total + 255) / 256;
  const int64_t cap = (int64_t)1 << 20;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  // (402 MB of 6144-byte rows 75.9 -> 61.3 us; 134 MB 21.5 -> 22.8 us, so below the line they stay)
  // Not where source rows repeat, more rows than the source has or one image for a whole batch: those
  // are read from the caches (65536 such rows out of 16: 101 us cached, 171 past them; 2^21 rows of 128
  // bytes out of 512: 63, 112; 16384 x 6144 bytes four times over: 112, 137).
  const bool once = rows <= src_rows && (outer == 1 || so != 0) && (rows == 1 || sr != 0);
  if (once && 2 * outer * rows * row_bytes > CACHE_BYTES)
    launch_walk<V, true>((unsigned)blocks, src, dst, index, rows, outer, so, dso, sr, dr, vpr, row_bytes, src_rows, error, stream);
  else
    launch_walk<V, false>((unsigned)blocks, src, dst, index, rows, outer, so, dso, sr, dr, vpr, row_bytes, src_rows, error, stream);
}

}  // namespace
}  // namespace hb

extern "C" int hb_gather_rows(const void* src, void* dst, const int64_t* index, int64_t rows, int64_t outer, int64_t src_outer_stride,
                              int64_t dst_outer_stride, int64_t src_row_stride,
                              int64_t dst_row_stride, int64_t row_bytes, int64_t src_rows,
                              int32_t* error, hb_stream_t stream) {
  HB_REQUIRE(src && dst && index, "null pointer argument");
  HB_REQUIRE(rows >= 0 && outer >= 0 && row_bytes > 0 && src_rows >= 0, "negative sizes");
  if (rows == 0 || outer == 0) return HB_OK;
  const int64_t vals[7] = {(int64_t)(uintptr_t)src, (int64_t)(uintptr_t)dst, src_outer_stride,
                           dst_outer_stride, src_row_stride, dst_row_stride, row_bytes};
  int width = 16;
  for (int i = 0; i < 7; ++i)
    while (width > 1 && vals[i] % width) width >>= 1;
  // rows of 16 bytes or more that nothing wider than 1-8 bytes divides (odd channel counts): 16-byte
  // vectors at any address, the last one of a row shifted back (16384 rows of 2052 bytes 21.6 -> 12.2
  // us, eight times as many 225 -> 106, of 4094 bytes, three times, 276 -> 79, of 2056 bytes, twice 65536,
  // 143 -> 111; launch-bound sizes as before)
  if (width < 16 && row_bytes >= 16) width = 0;
  switch (width) {
    case 0: hb::launch_gather<0>(src, dst, index, rows, outer, src_outer_stride, dst_outer_stride, src_row_stride, dst_row_stride, row_bytes, src_rows, error, stream); break;
    case 16: hb::launch_gather<16>(src, dst, index, rows, outer, src_outer_stride, dst_outer_stride, src_row_stride, dst_row_stride, row_bytes, src_rows, error, stream); break;
    case 8: hb::launch_gather<8>(src, dst, index, rows, outer, src_outer_stride, dst_outer_stride, src_row_stride, dst_row_stride, row_bytes, src_rows, error, stream); break;
    case 4: hb::launch_gather<4>(src, dst, index, rows, outer, src_outer_stride, dst_outer_stride, src_row_stride, dst_row_stride, row_bytes, src_rows, error, stream); break;
    case 2: hb::launch_gather<2>(src, dst, index, rows, outer, src_outer_stride, dst_outer_stride, src_row_stride, dst_row_stride, row_bytes, src_rows, error, stream); break;
    default: hb::launch_gather<1>(src, dst, index, rows, outer, src_outer_stride, dst_outer_stride, src_row_stride, dst_row_stride, row_bytes, src_rows, error, stream); break;
  }
  HB_HIP(hipGetLastError());
  return HB_OK;
}
