// Host arrays to the device and back (to_device / from_device, reference src/Device.jl:82-105): element type conversion on
// the GPU, pinned staging instead of the runtime's pageable copies.
//
// Bound: PCIe (57 GB/s). A runtime copy from pageable memory reaches 25 to 30 GB/s up and 17 down, waits for itself, and
// costs 13 to 35 us however small it is; converting to fp16 or bf16 on the host took ten times as long as the transfer.
// Upload: the host copies a piece of the caller's arrays into a pinned slot (a memcpy at 30 to 80 GB/s) while the GPU reads
// the piece before it straight from its slot, converting on the way (47 to 54 GB/s); the pieces of small arrays share a slot
// and a launch. Download: the GPU writes fp32 into pinned memory that becomes the caller's array.
#include <immintrin.h>
#include <string.h>

#include <mutex>

#include "common.hpp"
#include "dtypes.hpp"

namespace lmh {
namespace {

constexpr int kSegments = 8;           // pieces of arrays per launch
constexpr int kBlockBytes = 16384;     // source bytes per workgroup
constexpr size_t kSlotBytes = 1 << 20;
constexpr size_t kFirstBytes = 1 << 18;  // the first piece of a call is smaller, so that the GPU starts early
constexpr int kSlots = 16;
constexpr int kHalf = kSlots / 2;
constexpr int kMaxDevices = 64;

struct UploadArgs {
  void *dst[kSegments];
  const void *src[kSegments];
  int32_t bytes[kSegments];        // of the source
  int32_t first_block[kSegments];
  int32_t dtype[kSegments];        // what fp32 source values become; -1: bytes as they are
};

// Sources are 16-byte aligned (pieces are laid out so); destinations are aligned to their element, pieces start at multiples
// of 16 source bytes.
__global__ __launch_bounds__(256) void upload_kernel(UploadArgs a) {
  int s = 0;
#pragma unroll
  for (int i = 1; i < kSegments; i++)
    if (blockIdx.x >= (unsigned)a.first_block[i]) s = i;
  const int begin = (int)(blockIdx.x - a.first_block[s]) * kBlockBytes;
  const int end = min(begin + kBlockBytes, a.bytes[s]);
  const char *src = reinterpret_cast<const char *>(a.src[s]);
  const int dtype = a.dtype[s];
  uint4 x[kBlockBytes / 4096];
#pragma unroll
  for (int r = 0; r < kBlockBytes / 4096; r++) {
    const int i = begin + (r * 256 + threadIdx.x) * 16;
    x[r] = i < end ? *reinterpret_cast<const uint4 *>(src + i) : make_uint4(0, 0, 0, 0);  // (slots are padded to 16 bytes)
  }
#pragma unroll
  for (int r = 0; r < kBlockBytes / 4096; r++) {
    const int i = begin + (r * 256 + threadIdx.x) * 16;
    if (i >= end) continue;
    const uint32_t w[4] = {x[r].x, x[r].y, x[r].z, x[r].w};
    if (dtype == LMH_F16 || dtype == LMH_BF16) {
      uint16_t *dst = reinterpret_cast<uint16_t *>(a.dst[s]) + i / 4;
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float f = __uint_as_float(w[e]);
        h[e] = dtype == LMH_F16 ? __builtin_bit_cast(uint16_t, (_Float16)f) : f32_to_bf16_bits(f);
      }
      if (i + 16 <= end && ((uintptr_t)dst & 7) == 0) {
        *reinterpret_cast<uint2 *>(dst) = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (i + 4 * e < end) dst[e] = h[e];
      }
    } else {
      char *dst = reinterpret_cast<char *>(a.dst[s]) + i;
      if (i + 16 <= end && ((uintptr_t)dst & 15) == 0) {
        *reinterpret_cast<uint4 *>(dst) = x[r];
      } else {
        for (int e = 0; e < 16 && i + e < end; e++) dst[e] = (char)(w[e >> 2] >> (8 * (e & 3)));
      }
    }
  }
}

// n values of any type -> fp32 in pinned host memory, four per thread and step. (32-bit ones too: a copy of the runtime's begins 10 us
// after the kernel in front of it. execute() of 2 MB of results 292 -> 280 us, of 256 KB 76.9 -> 72.9.)
__global__ __launch_bounds__(256) void download_kernel(float *dst, const void *src, int64_t n, int dtype) {
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += (int64_t)gridDim.x * 1024) {
    float f[4];
    const bool words = dtype == LMH_F32;
    if (words && i + 4 <= n && ((uintptr_t)src & 15) == 0) {
      *reinterpret_cast<uint4 *>(dst + i) = *reinterpret_cast<const uint4 *>(reinterpret_cast<const float *>(src) + i);
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (i + e >= n) break;
      if (words) {
        f[e] = reinterpret_cast<const float *>(src)[i + e];
        continue;
      }
      const uint16_t h = reinterpret_cast<const uint16_t *>(src)[i + e];
      f[e] = dtype == LMH_F16 ? (float)__builtin_bit_cast(_Float16, h) : bf16_bits_to_f32(h);
    }
    if (i + 4 <= n) {
      *reinterpret_cast<float4 *>(dst + i) = make_float4(f[0], f[1], f[2], f[3]);
    } else {
      for (int e = 0; i + e < n; e++) dst[i + e] = f[e];
    }
  }
}

// memcpy into a slot without reading its old lines into the cache first: the GPU reads them next, not this core (72 MB of
// host arrays up: 26 -> 38 GB/s). Slots and pieces are 16-byte aligned; the stores want 32.
__attribute__((target("avx2"))) void copy_streaming(char *dst, const char *src, size_t n) {
  size_t i = 0;
  if (((uintptr_t)dst & 31) && n >= 16) {
    _mm_stream_si128((__m128i *)dst, _mm_loadu_si128((const __m128i *)src));
    i = 16;
  }
  for (; i + 128 <= n; i += 128) {
    const __m256i a = _mm256_loadu_si256((const __m256i *)(src + i)), b = _mm256_loadu_si256((const __m256i *)(src + i + 32));
    const __m256i c = _mm256_loadu_si256((const __m256i *)(src + i + 64)), d = _mm256_loadu_si256((const __m256i *)(src + i + 96));
    _mm256_stream_si256((__m256i *)(dst + i), a);
    _mm256_stream_si256((__m256i *)(dst + i + 32), b);
    _mm256_stream_si256((__m256i *)(dst + i + 64), c);
    _mm256_stream_si256((__m256i *)(dst + i + 96), d);
  }
  memcpy(dst + i, src + i, n - i);
  _mm_sfence();
}
void copy_to_slot(char *dst, const char *src, size_t n) {
  static const bool avx2 = __builtin_cpu_supports("avx2");
  if (avx2 && n >= 4096) copy_streaming(dst, src, n);
  else memcpy(dst, src, n);
}

// The pinned slots of one GPU, used in turn. An event behind the launches that read a half of them says when that half is
// free again; it covers one stream's launches: calls on the null stream fill a half together, a call on any other stream
// closes its half when it is done (the stream may be gone later). (An event behind every launch leaves the GPU idle for some microseconds each time: 6 MB of arrays 223 -> 168 us.)
// One upload at a time fills slots (any thread, any stream); they are held until the process ends.
struct Stage {
  char *slot[kSlots] = {};
  hipEvent_t read[2] = {};
  bool pending[2] = {};
  hipStream_t stream = nullptr;  // of the launches since the last event
  bool open = false;             // there are such launches
  int next = 0;
};
Stage g_stage[kMaxDevices];
std::mutex g_stage_mutex;

int stage_setup(Stage &st) {
  if (st.slot[kSlots - 1]) return LMH_OK;
  for (int i = 0; i < 2; i++)
    if (!st.read[i]) LMH_HIP_TRY(hipEventCreateWithFlags(&st.read[i], hipEventDisableTiming));
  for (int i = 0; i < kSlots; i++)
    if (!st.slot[i]) LMH_HIP_TRY(hipHostMalloc((void **)&st.slot[i], kSlotBytes, hipHostMallocDefault));
  return LMH_OK;
}

// Close the half that `next` lies in (or just left): its event goes behind the launches that read it.
int stage_close(Stage &st) {
  if (!st.open) return LMH_OK;
  const int half = (st.next + kSlots - 1) % kSlots / kHalf;
  LMH_HIP_TRY(hipEventRecord(st.read[half], st.stream));
  st.pending[half] = true;
  st.open = false;
  return LMH_OK;
}

}  // namespace

int launch_upload(const UploadItem *items, int n, hipStream_t stream) {
  int dev = 0;
  LMH_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(LMH_E_NODEVICE, "upload: device index %d is too large", dev);
  std::lock_guard<std::mutex> lock(g_stage_mutex);
  Stage &st = g_stage[dev];
  const int rc = stage_setup(st);
  if (rc != LMH_OK) return rc;
  auto close_half = [&st]() {  // even if it is not full
    const int closed = stage_close(st);
    st.next = (st.next + kHalf - 1) / kHalf * kHalf % kSlots;
    return closed;
  };
  if (st.open && stream) {
    const int closed = close_half();
    if (closed != LMH_OK) return closed;
  }
  size_t limit = kFirstBytes, done = 0;  // bytes of item `i` already on their way
  for (int i = 0; i < n;) {
    const int k = st.next, half = k / kHalf;
    if (k % kHalf == 0 && st.pending[half]) {
      LMH_HIP_TRY(hipEventSynchronize(st.read[half]));
      st.pending[half] = false;
    }
    UploadArgs a = {};
    size_t used = 0;
    int segments = 0, blocks = 0;
    for (; i < n && segments < kSegments && used < limit;) {
      const size_t left = items[i].bytes - done, take = left < limit - used ? left : limit - used;
      if (take) {
        copy_to_slot(st.slot[k] + used, reinterpret_cast<const char *>(items[i].src) + done, take);
        const size_t elem = items[i].dtype < 0 || items[i].dtype == LMH_F32 ? 1 : 2;  // destination bytes: done / elem
        a.dst[segments] = reinterpret_cast<char *>(items[i].dst) + done / elem;
        a.src[segments] = st.slot[k] + used;
        a.bytes[segments] = (int32_t)take;
        a.dtype[segments] = items[i].dtype;
        a.first_block[segments] = blocks;
        blocks += (int)((take + kBlockBytes - 1) / kBlockBytes);
        segments++;
        used += (take + 15) & ~(size_t)15;
        done += take;
      }
      if (done == items[i].bytes) i++, done = 0;
    }
    if (blocks == 0) continue;
    for (int j = segments; j < kSegments; j++) a.first_block[j] = blocks;
    hipLaunchKernelGGL(upload_kernel, dim3(blocks), dim3(256), 0, stream, a);
    LMH_HIP_TRY(hipGetLastError());
    st.stream = stream;
    st.open = true;
    st.next = (k + 1) % kSlots;
    if (st.next % kHalf == 0) {
      const int closed = stage_close(st);
      if (closed != LMH_OK) return closed;
    }
    limit = kSlotBytes;
  }
  return stream ? close_half() : LMH_OK;
}

int launch_download(float *dst, const void *src, int64_t n, int dtype, hipStream_t stream) {
  if (dtype == LMH_F32) {  // the runtime's copy takes memory that a kernel does not reach: of the host's but not pinned, of another GPU
    hipPointerAttribute_t to, from;
    int dev = 0;
    const bool reached = ((uintptr_t)dst & 15) == 0 && ((uintptr_t)src & 3) == 0 && hipGetDevice(&dev) == hipSuccess &&
                         hipPointerGetAttributes(&to, dst) == hipSuccess && to.type == hipMemoryTypeHost &&
                         hipPointerGetAttributes(&from, src) == hipSuccess && from.type == hipMemoryTypeDevice && from.device == dev;
    if (!reached) {
      (void)hipGetLastError();
      LMH_HIP_TRY(hipMemcpyAsync(dst, src, (size_t)n * 4, hipMemcpyDeviceToHost, stream));
      return LMH_OK;
    }
  }
  const int64_t blocks = (n + 1023) / 1024;
  hipLaunchKernelGGL(download_kernel, dim3((unsigned)(blocks > 1024 ? 1024 : blocks)), dim3(256), 0, stream, dst, src, n, dtype);
  LMH_HIP_TRY(hipGetLastError());
  return LMH_OK;
}

}  // namespace lmh
