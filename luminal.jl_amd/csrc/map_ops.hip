// The data movement of a model graph around its attention nodes: permutes, reshapes, repeats, sums with broadcasting and
// element type conversions (reference src/Execution.jl:207-250), and the copy of a call's inputs into a compiled graph's
// buffers (reference src/Compiler.jl:80-96). All of it is bound by HBM and, at the sizes of a decode step, by the launch.
//
// map: out[i0, i1, ...] = a[i . a_stride] (+ b[i . b_stride]), out contiguous, any element types. Two forms:
//   * rows: consecutive threads take consecutive elements of out, four at a time; the operands are contiguous along out's
//     innermost dimension or constant along it, so every access is coalesced;
//   * tiles: where an operand's contiguous dimension is another one than out's (a transpose), 64 x 64 tiles of those two
//     dimensions pass through LDS, so that both sides move whole lines.
#include "common.hpp"
#include "copy.hpp"
#include "dtypes.hpp"

namespace lmh {
namespace {

// F32: the operand is known to be fp32 when the kernel is compiled. A switch in front of every load keeps the compiler from
// issuing a thread's loads together (the heads of 700 x 2048 fp32 merged, [32, 700, 64] -> [700, 64, 32]: 8.4 us with the
// switch and a branch per load, 5.6 us without; 4096 x 4096: 42 -> 25.7 us = 5.2 TB/s).
template <bool F32>
__device__ inline float map_load(const void *p, int64_t i, int dtype) {
  if constexpr (F32) return reinterpret_cast<const float *>(p)[i];
  switch (dtype) {
    case LMH_F16: return (float)reinterpret_cast<const _Float16 *>(p)[i];
    case LMH_BF16: return bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p)[i]);
    case LMH_I32: return (float)reinterpret_cast<const int32_t *>(p)[i];
    default: return reinterpret_cast<const float *>(p)[i];
  }
}
template <bool F32>
__device__ inline void map_store(void *p, int64_t i, int dtype, float x) {
  if constexpr (F32) dtype = LMH_F32;
  switch (dtype) {
    case LMH_F16: reinterpret_cast<_Float16 *>(p)[i] = (_Float16)x; break;
    case LMH_BF16: reinterpret_cast<uint16_t *>(p)[i] = f32_to_bf16_bits(x); break;
    default: reinterpret_cast<float *>(p)[i] = x;
  }
}

constexpr int kRowElems = 4;  // consecutive elements of out's innermost dimension per thread

// (indices are 32-bit: 64-bit divisions are a hundred instructions each here, and there is one per dimension)
template <bool F32>
__global__ __launch_bounds__(256) void map_rows_kernel(MapArgs a, uint32_t n_groups, uint32_t groups_per_row) {
  const int inner = a.n_dims - 1;
  for (uint32_t t = blockIdx.x * 256 + threadIdx.x; t < n_groups; t += gridDim.x * 256) {
    uint32_t row = t / groups_per_row;
    const int i0 = (int)(t - row * groups_per_row) * kRowElems;
    const int64_t out0 = (int64_t)row * a.dims[inner] + i0;
    int64_t off_a = 0, off_b = 0;
    for (int d = inner - 1; d >= 0; d--) {
      const uint32_t q = row / (uint32_t)a.dims[d];
      const int64_t i = row - q * (uint32_t)a.dims[d];
      off_a += i * a.as[d];
      off_b += i * a.bs[d];
      row = q;
    }
    float x[kRowElems];
#pragma unroll
    for (int e = 0; e < kRowElems; e++) {
      const int i = i0 + e;
      if (i >= a.dims[inner]) break;
      x[e] = map_load<F32>(a.a, off_a + i * a.as[inner], a.a_dtype);
      if (a.b) x[e] += map_load<F32>(a.b, off_b + i * a.bs[inner], a.b_dtype);
    }
#pragma unroll
    for (int e = 0; e < kRowElems; e++)
      if (i0 + e < a.dims[inner]) map_store<F32>(a.out, out0 + e, a.out_dtype, x[e]);
  }
}

constexpr int kTile = 64;

// a.tile_dim is the dimension along which operand a is contiguous; the tile spans it and out's innermost dimension.
template <bool F32>
__global__ __launch_bounds__(256) void map_tiles_kernel(MapArgs a, int tiles_in, int tiles_out) {
  __shared__ float tile[kTile][kTile + 1];
  const int inner = a.n_dims - 1;
  uint32_t rest = blockIdx.x;
  const int t_out = (int)(rest % (uint32_t)tiles_out);
  rest /= (uint32_t)tiles_out;
  const int t_in = (int)(rest % (uint32_t)tiles_in);
  rest /= (uint32_t)tiles_in;
  int64_t off_a = 0, off_b = 0, off_o = 0, out_stride_in = 0, out_stride = 1;
  for (int d = inner; d >= 0; d--) {  // offsets of the remaining dimensions, and out's stride along the tiled one
    if (d == a.tile_dim) out_stride_in = out_stride;
    if (d != a.tile_dim && d != inner) {
      const uint32_t q = rest / (uint32_t)a.dims[d];
      const int64_t i = rest - q * (uint32_t)a.dims[d];
      off_a += i * a.as[d];
      off_b += i * a.bs[d];
      off_o += i * out_stride;
      rest = q;
    }
    out_stride *= a.dims[d];
  }
  const int n_in = a.dims[a.tile_dim], n_out = a.dims[inner];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  {  // all of a thread's loads first, without branches: elements past the tile's edge repeat the last valid one
    const int i = min(t_in * kTile + lane, n_in - 1);
    float x[kTile / 4];
#pragma unroll
    for (int r = 0; r < kTile / 4; r++) {
      const int o = min(t_out * kTile + 4 * r + wave, n_out - 1);
      x[r] = map_load<F32>(a.a, off_a + i * a.as[a.tile_dim] + o * a.as[inner], a.a_dtype);
    }
#pragma unroll
    for (int r = 0; r < kTile / 4; r++) tile[4 * r + wave][lane] = x[r];
  }
  __syncthreads();
  const int o = t_out * kTile + lane;
#pragma unroll
  for (int r = wave; r < kTile; r += 4) {
    const int i = t_in * kTile + r;
    if (i >= n_in || o >= n_out) continue;
    float x = tile[lane][r];
    if (a.b) x += map_load<F32>(a.b, off_b + i * a.bs[a.tile_dim] + o * a.bs[inner], a.b_dtype);
    map_store<F32>(a.out, off_o + i * out_stride_in + o, a.out_dtype, x);
  }
}

// Up to kCopyMany byte ranges in one launch: the inputs of a compiled graph's call are a handful of small tensors, and a
// runtime copy of each costs the host 3.4 us (a decode step's five: 17.8 us of its 26 us). A workgroup moves 16 KB.
__global__ __launch_bounds__(256) void copy_many_kernel(CopyManyArgs a) { copy_block<256>(a, blockIdx.x); }

}  // namespace

int launch_map(MapArgs &a, hipStream_t stream) {
  // a dimension other than out's innermost along which operand a is contiguous, long enough to be worth a tile
  a.tile_dim = -1;
  const int inner = a.n_dims - 1;
  if (a.as[inner] != 1 && a.as[inner] != 0 && a.dims[inner] >= 8)
    for (int d = 0; d < inner; d++)
      if (a.as[d] == 1 && a.dims[d] >= 8) a.tile_dim = d;
  const bool f32 = a.a_dtype == LMH_F32 && a.out_dtype == LMH_F32 && (!a.b || a.b_dtype == LMH_F32);
  int64_t total = 1;
  for (int d = 0; d < a.n_dims; d++) total *= a.dims[d];
  if (a.tile_dim >= 0) {
    const int64_t tiles_in = (a.dims[a.tile_dim] + kTile - 1) / kTile, tiles_out = (a.dims[inner] + kTile - 1) / kTile;
    const int64_t blocks = total / ((int64_t)a.dims[a.tile_dim] * a.dims[inner]) * tiles_in * tiles_out;
    if (blocks < (int64_t(1) << 31)) {
      if (f32) hipLaunchKernelGGL(map_tiles_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, stream, a, (int)tiles_in, (int)tiles_out);
      else hipLaunchKernelGGL(map_tiles_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, stream, a, (int)tiles_in, (int)tiles_out);
      LMH_HIP_TRY(hipGetLastError());
      return LMH_OK;
    }
  }
  const int groups_per_row = (a.dims[inner] + kRowElems - 1) / kRowElems;
  const int64_t n_groups = total / a.dims[inner] * groups_per_row;
  if (n_groups >= (int64_t(1) << 31)) return fail(LMH_E_UNSUPPORTED, "lmh_map: %lld elements are too many", (long long)total);
  const int64_t blocks = (n_groups + 255) / 256;
  const dim3 grid((unsigned)(blocks > 65536 ? 65536 : blocks));
  if (f32) hipLaunchKernelGGL(map_rows_kernel<true>, grid, dim3(256), 0, stream, a, (uint32_t)n_groups, (uint32_t)groups_per_row);
  else hipLaunchKernelGGL(map_rows_kernel<false>, grid, dim3(256), 0, stream, a, (uint32_t)n_groups, (uint32_t)groups_per_row);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

int launch_copy_many(CopyManyArgs &a, int n, hipStream_t stream) {
  const int64_t blocks = number_copy_blocks(a, n);
  if (blocks < 0) return fail(LMH_E_UNSUPPORTED, "copy: too many bytes in one call");
  if (blocks == 0) return LMH_OK;
  hipLaunchKernelGGL(copy_many_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

}  // namespace lmh
