// C-ABI layer of libluminal_hip.so: argument validation, dispatch to the kernel launchers, and
// the small device-runtime surface (allocation, copies, sync, events) that stands in for the
// CuArray()/Array() calls of the reference's device layer (reference src/Device.jl:82-105).
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>

#include "common.hpp"
#include "copy.hpp"

// Split-KV partial storage of lmh_decode_attn_static, for callers that cannot allocate device memory.
// One copy per GPU, held from the moment the code object is loaded on that GPU until the process ends.
static __device__ __align__(256) unsigned char scratch[LMH_STATIC_SCRATCH_BYTES];

namespace lmh {

static thread_local char g_last_error[512] = "";

int device_cu_count() {
  static const int n = [] {  // one device kind per process (gfx950); initialised once, thread-safely
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess || prop.multiProcessorCount < 1) {
      (void)hipGetLastError();
      return 256;
    }
    return prop.multiProcessorCount;
  }();
  return n;
}

int check_grid(int64_t workgroups, int threads) {
  if (workgroups * threads <= 0xffffffffll) return LMH_OK;
  return fail(LMH_E_UNSUPPORTED, "%lld workgroups of %d threads are more than a launch can number", (long long)workgroups, threads);
}

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return code;
}

static thread_local char *g_plan_buf = nullptr;
static thread_local size_t g_plan_bytes = 0;

bool plan_only(const char *fmt, ...) {
  if (!g_plan_buf) return false;
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_plan_buf, g_plan_bytes, fmt, ap);
  va_end(ap);
  return true;
}

int hip_fail(hipError_t e, const char *what) {
  return fail(LMH_E_HIP, "HIP error %d (%s) in %s", (int)e, hipGetErrorString(e), what);
}

namespace {

bool all_zero(const int64_t *s, int n) {
  for (int i = 0; i < n; i++)
    if (s[i] != 0) return false;
  return true;
}

size_t elem_bytes(int dtype) { return dtype == LMH_F32 ? 4 : 2; }

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

constexpr int kMaxDevices = 64;
// Device address of `scratch` on each GPU. In host code the array's name is only a handle for
// hipGetSymbolAddress, never an address a kernel can use.
void *g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mutex;
// Who used the scratch last on each GPU: an event recorded behind that call's kernels and the stream it ran on. The next
// call on another stream asks the event whether the earlier call has finished, and refuses to race with it.
struct ScratchUse {
  hipEvent_t done = nullptr;
  hipStream_t stream = nullptr;
  bool pending = false;
};
ScratchUse g_scratch_use[kMaxDevices];

// Looks the address up once per device, with that device current, and returns it in *out.
int static_scratch_for_current_device(void **out) {
  *out = nullptr;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return fail(LMH_E_NODEVICE, "static scratch: no current HIP device (or its index is >= %d)", kMaxDevices);
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!ptr) return fail(LMH_E_HIP, "static scratch: hipGetSymbolAddress returned a null address");
    hipEvent_t ev = nullptr;  // part of the same one-time set-up: the entry point itself creates nothing
    const hipError_t ee = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (ee != hipSuccess) return hip_fail(ee, "hipEventCreateWithFlags(static scratch)");
    g_scratch_use[dev].done = ev;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return LMH_OK;
}

// True while `stream` is recording a HIP graph (then nothing may be queried or recorded on its behalf).
bool stream_is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &st) != hipSuccess) {
    (void)hipGetLastError();
    return true;  // cannot tell: behave as under capture (no event calls)
  }
  return st != hipStreamCaptureStatusNone;
}

// Before a call that uses the scratch: refuse when the previous user, on another stream, is still running. Two calls on
// one stream are ordered by the stream; the null stream and the streams of lmh_stream_create order themselves against
// each other, so only two different non-null streams can overlap. Calls recorded into a graph are not seen here.
int static_scratch_claim(hipStream_t stream, const char *fn) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return LMH_OK;
  }
  if (stream_is_capturing(stream)) return LMH_OK;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  ScratchUse &u = g_scratch_use[dev];
  if (u.pending && u.stream != stream && u.stream != nullptr && stream != nullptr) {
    const hipError_t q = hipEventQuery(u.done);
    if (q == hipErrorNotReady)
      return fail(LMH_E_BUSY, "%s: the previous call that uses this GPU's static scratch is still running on another stream; "
                              "calls that share the scratch must not overlap (order them, or use lmh_decode_attn with a workspace)", fn);
    if (q != hipSuccess) (void)hipGetLastError();
  }
  return LMH_OK;
}

// After the kernels of such a call were enqueued.
void static_scratch_mark(hipStream_t stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return;
  }
  if (stream_is_capturing(stream)) return;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  ScratchUse &u = g_scratch_use[dev];
  if (!u.done) return;
  if (hipEventRecord(u.done, stream) != hipSuccess) {
    (void)hipGetLastError();
    u.pending = false;
    return;
  }
  u.stream = stream;
  u.pending = true;
}

}  // namespace
}  // namespace lmh

using namespace lmh;

extern "C" {

int lmh_version(void) { return LMH_VERSION; }

int lmh_measurement_build(void) {
#ifdef LMH_MEASUREMENT_BUILD
  return 1;
#else
  return 0;
#endif
}

const char *lmh_last_error(void) { return g_last_error; }

int lmh_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  int usable = 0;
  for (int i = 0; i < n; i++) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, i) == hipSuccess && strncmp(prop.gcnArchName, "gfx950", 6) == 0) usable++;
  }
  return usable;
}

int lmh_init(int device) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return fail(LMH_E_NODEVICE, "no HIP device visible");
  }
  if (device < 0 || device >= n) return fail(LMH_E_NODEVICE, "device %d out of range (have %d)", device, n);
  hipDeviceProp_t prop;
  LMH_HIP_TRY(hipGetDeviceProperties(&prop, device));
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(LMH_E_NODEVICE, "device %d is %s; this library carries gfx950 code only", device, prop.gcnArchName);
  LMH_HIP_TRY(hipSetDevice(device));
  void *probe = nullptr;  // same health check as get_device(): a tiny allocation
  LMH_HIP_TRY(hipMalloc(&probe, 4));
  LMH_HIP_TRY(hipFree(probe));
  // set-up for lmh_decode_attn_static: resolve this device's copy of the static scratch now, so that the
  // entry point itself never has to (a failure here is reported by that entry point, not by init)
  void *unused = nullptr;
  if (static_scratch_for_current_device(&unused) != LMH_OK) g_last_error[0] = 0;  // init succeeded: leave no stale message
  return LMH_OK;
}

int lmh_device_name(char *buf, size_t buf_bytes) {
  if (!buf || buf_bytes == 0) return fail(LMH_E_NULL, "lmh_device_name: null buffer");
  int dev = 0;
  LMH_HIP_TRY(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  LMH_HIP_TRY(hipGetDeviceProperties(&prop, dev));
  snprintf(buf, buf_bytes, "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
  return LMH_OK;
}

int lmh_malloc(void **dev_ptr, size_t bytes) {
  if (!dev_ptr) return fail(LMH_E_NULL, "lmh_malloc: null result pointer");
  *dev_ptr = nullptr;
  if (bytes == 0) return LMH_OK;
  LMH_HIP_TRY(hipMalloc(dev_ptr, bytes));
  return LMH_OK;
}

int lmh_free(void *dev_ptr) {
  if (!dev_ptr) return LMH_OK;
  LMH_HIP_TRY(hipFree(dev_ptr));
  return LMH_OK;
}

int lmh_memset(void *dev_ptr, int byte_value, size_t bytes, void *stream) {
  if (bytes == 0) return LMH_OK;
  if (!dev_ptr) return fail(LMH_E_NULL, "lmh_memset: null pointer");
  LMH_HIP_TRY(hipMemsetAsync(dev_ptr, byte_value, bytes, (hipStream_t)stream));
  return LMH_OK;
}

int lmh_memcpy_h2d(void *dst_dev, const void *src_host, size_t bytes, void *stream) {
  if (bytes == 0) return LMH_OK;
  if (!dst_dev || !src_host) return fail(LMH_E_NULL, "lmh_memcpy_h2d: null pointer");
  LMH_HIP_TRY(hipMemcpyAsync(dst_dev, src_host, bytes, hipMemcpyHostToDevice, (hipStream_t)stream));
  LMH_HIP_TRY(hipStreamSynchronize((hipStream_t)stream));  // the host buffer may be reused at once
  return LMH_OK;
}

int lmh_memcpy_d2h(void *dst_host, const void *src_dev, size_t bytes, void *stream) {
  if (bytes == 0) return LMH_OK;
  if (!dst_host || !src_dev) return fail(LMH_E_NULL, "lmh_memcpy_d2h: null pointer");
  LMH_HIP_TRY(hipMemcpyAsync(dst_host, src_dev, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream));
  LMH_HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
  return LMH_OK;
}

int lmh_memcpy_d2d(void *dst_dev, const void *src_dev, size_t bytes, void *stream) {
  if (bytes == 0) return LMH_OK;
  if (!dst_dev || !src_dev) return fail(LMH_E_NULL, "lmh_memcpy_d2d: null pointer");
  LMH_HIP_TRY(hipMemcpyAsync(dst_dev, src_dev, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream));
  return LMH_OK;
}

int lmh_sync(void *stream) {
  LMH_HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
  return LMH_OK;
}

int lmh_host_alloc(void **ptr, size_t bytes) {
  if (!ptr) return fail(LMH_E_NULL, "lmh_host_alloc: null result pointer");
  *ptr = nullptr;
  if (bytes == 0) return LMH_OK;
  LMH_HIP_TRY(hipHostMalloc(ptr, bytes, hipHostMallocDefault));
  return LMH_OK;
}

int lmh_host_free(void *ptr) {
  if (!ptr) return LMH_OK;
  LMH_HIP_TRY(hipHostFree(ptr));
  return LMH_OK;
}

int lmh_upload(const lmh_upload_item *items, int32_t n, void *stream) {
  if (n < 0 || n > LMH_UPLOAD_ITEMS) return fail(LMH_E_SHAPE, "lmh_upload: %d arrays, up to %d fit a call", n, LMH_UPLOAD_ITEMS);
  if (n > 0 && !items) return fail(LMH_E_NULL, "lmh_upload: null list");
  UploadItem out[LMH_UPLOAD_ITEMS];
  for (int i = 0; i < n; i++) {
    if (items[i].n < 0) return fail(LMH_E_SHAPE, "lmh_upload: negative length");
    if (items[i].n > 0 && (!items[i].dst || !items[i].src)) return fail(LMH_E_NULL, "lmh_upload: null pointer");
    if (items[i].convert && items[i].dtype != LMH_F32 && items[i].dtype != LMH_F16 && items[i].dtype != LMH_BF16)
      return fail(LMH_E_UNSUPPORTED, "lmh_upload: unknown element type %d", items[i].dtype);
    out[i].dst = items[i].dst;
    out[i].src = items[i].src;
    out[i].bytes = (size_t)items[i].n * (items[i].convert ? 4 : 1);
    out[i].dtype = items[i].convert && items[i].dtype != LMH_F32 ? items[i].dtype : -1;
  }
  return launch_upload(out, n, (hipStream_t)stream);
}

int lmh_download(void *dst_pinned, const void *src_dev, int64_t n, int32_t dtype, void *stream) {
  if (n < 0) return fail(LMH_E_SHAPE, "lmh_download: negative length");
  if (n == 0) return LMH_OK;
  if (!dst_pinned || !src_dev) return fail(LMH_E_NULL, "lmh_download: null pointer");
  if (dtype != LMH_F32 && dtype != LMH_F16 && dtype != LMH_BF16) return fail(LMH_E_UNSUPPORTED, "lmh_download: unknown element type %d", dtype);
  return launch_download(reinterpret_cast<float *>(dst_pinned), src_dev, n, dtype, (hipStream_t)stream);
}

int lmh_stream_create(void **stream) {
  if (!stream) return fail(LMH_E_NULL, "lmh_stream_create: null result pointer");
  hipStream_t s;
  LMH_HIP_TRY(hipStreamCreate(&s));  // default flags and priority
  *stream = s;
  return LMH_OK;
}

int lmh_stream_destroy(void *stream) {
  if (!stream) return LMH_OK;
  LMH_HIP_TRY(hipStreamDestroy((hipStream_t)stream));
  return LMH_OK;
}

int lmh_graph_capture_begin(void *stream) {
  if (!stream) return fail(LMH_E_NULL, "lmh_graph_capture_begin: the null stream cannot be captured");
  // thread-local: API calls of other host threads (a finalizer freeing memory) do not break the capture
  LMH_HIP_TRY(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeThreadLocal));
  return LMH_OK;
}

int lmh_graph_capture_end(void *stream, void **graph_exec) {
  if (!stream || !graph_exec) return fail(LMH_E_NULL, "lmh_graph_capture_end: null stream or result pointer");
  *graph_exec = nullptr;
  hipGraph_t graph = nullptr;
  LMH_HIP_TRY(hipStreamEndCapture((hipStream_t)stream, &graph));
  if (!graph) return fail(LMH_E_HIP, "lmh_graph_capture_end: the capture was invalidated");
  hipGraphExec_t exec = nullptr;
  const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  LMH_HIP_TRY(e);
  *graph_exec = exec;
  return LMH_OK;
}

int lmh_graph_launch(void *graph_exec, void *stream) {
  if (!graph_exec) return fail(LMH_E_NULL, "lmh_graph_launch: null graph");
  LMH_HIP_TRY(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
  return LMH_OK;
}

int lmh_graph_destroy(void *graph_exec) {
  if (!graph_exec) return LMH_OK;
  LMH_HIP_TRY(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
  return LMH_OK;
}

int lmh_event_create(void **event) {
  if (!event) return fail(LMH_E_NULL, "lmh_event_create: null result pointer");
  hipEvent_t e;
  LMH_HIP_TRY(hipEventCreate(&e));
  *event = e;
  return LMH_OK;
}

int lmh_event_destroy(void *event) {
  if (!event) return LMH_OK;
  LMH_HIP_TRY(hipEventDestroy((hipEvent_t)event));
  return LMH_OK;
}

int lmh_event_record(void *event, void *stream) {
  if (!event) return fail(LMH_E_NULL, "lmh_event_record: null event");
  LMH_HIP_TRY(hipEventRecord((hipEvent_t)event, (hipStream_t)stream));
  return LMH_OK;
}

int lmh_event_elapsed_ms(float *ms, void *start, void *stop) {
  if (!ms || !start || !stop) return fail(LMH_E_NULL, "lmh_event_elapsed_ms: null argument");
  LMH_HIP_TRY(hipEventSynchronize((hipEvent_t)stop));
  LMH_HIP_TRY(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
  return LMH_OK;
}

// --------------------------------------------------------------------------------------------
// flash attention forward
// --------------------------------------------------------------------------------------------
static int attn_args(const lmh_attn_params *p, PrefillArgs &a, bool &mfma_ok) {
  if (!p) return fail(LMH_E_NULL, "lmh_flash_attn_fwd: null params");
  if (!p->out || !p->q || !p->k || !p->v) return fail(LMH_E_NULL, "lmh_flash_attn_fwd: null tensor pointer");
  if (p->B <= 0 || p->Hq <= 0 || p->Hkv <= 0 || p->Sq <= 0 || p->Sk <= 0 || p->D <= 0)
    return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: non-positive dimension (B=%d Hq=%d Hkv=%d Sq=%d Sk=%d D=%d)", p->B,
                p->Hq, p->Hkv, p->Sq, p->Sk, p->D);
  if (p->Hq % p->Hkv != 0)
    return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: Hq=%d is not a multiple of Hkv=%d", p->Hq, p->Hkv);
  if (p->dtype != LMH_F32 && p->dtype != LMH_F16 && p->dtype != LMH_BF16)
    return fail(LMH_E_UNSUPPORTED, "lmh_flash_attn_fwd: unknown dtype %d", p->dtype);
  if (p->head_map != LMH_HEADMAP_INTERLEAVED && p->head_map != LMH_HEADMAP_BLOCKED)
    return fail(LMH_E_UNSUPPORTED, "lmh_flash_attn_fwd: unknown head_map %d", p->head_map);
  if (p->D > 256) return fail(LMH_E_UNSUPPORTED, "lmh_flash_attn_fwd: head dim %d > 256 is not supported", p->D);
  if (!(p->scale == p->scale)) return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: scale is NaN");
  if (p->q_rope) {
    if (p->D % 2 != 0) return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: head dim %d must be even for the rotary embedding", p->D);
    if (p->q_rope_pairing != LMH_ROPE_HALF_SPLIT && p->q_rope_pairing != LMH_ROPE_INTERLEAVED)
      return fail(LMH_E_UNSUPPORTED, "lmh_flash_attn_fwd: unknown q_rope_pairing %d", p->q_rope_pairing);
    if (!(p->q_rope_base > 0.f)) return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: q_rope_base must be positive");
  }

  a.out = p->out; a.q = p->q; a.k = p->k; a.v = p->v; a.kv_len = p->kv_len;
  a.B = p->B; a.Hq = p->Hq; a.Hkv = p->Hkv; a.Sq = p->Sq; a.Sk = p->Sk; a.D = p->D;
  a.scale = p->scale; a.causal = p->causal ? 1 : 0; a.head_map = p->head_map;
  a.out_f32 = (p->out_f32 != 0 || p->dtype == LMH_F32) ? 1 : 0;
  a.q_rope = p->q_rope ? 1 : 0;
  a.q_interleaved = p->q_rope_pairing == LMH_ROPE_INTERLEAVED;
  a.q_pos0 = p->q_rope ? p->q_pos0 : nullptr;
  a.q_prev_seq = p->q_prev_seq;
  a.q_log2_base = p->q_rope ? log2f(p->q_rope_base) : 0.f;
  auto fill = [&](int64_t *dst, const int64_t *src, int64_t H, int64_t S) {
    if (all_zero(src, 3)) {
      dst[0] = H * S * p->D; dst[1] = S * p->D; dst[2] = p->D;
    } else {
      dst[0] = src[0]; dst[1] = src[1]; dst[2] = src[2];
    }
  };
  fill(a.qs, p->q_stride, p->Hq, p->Sq);
  fill(a.os, p->o_stride, p->Hq, p->Sq);
  fill(a.ks, p->k_stride, p->Hkv, p->Sk);
  fill(a.vs, p->v_stride, p->Hkv, p->Sk);
  for (int i = 0; i < 3; i++)
    if (a.qs[i] < 0 || a.os[i] < 0 || a.ks[i] < 0 || a.vs[i] < 0)
      return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: negative stride");
  if (a.qs[2] < p->D || a.os[2] < p->D || a.ks[2] < p->D || a.vs[2] < p->D)
    return fail(LMH_E_SHAPE, "lmh_flash_attn_fwd: row stride smaller than head dim (rows overlap)");

  // The matrix-core kernels do 128-bit accesses, track the max on raw scores (needs scale > 0) and fetch
  // K/V tiles with 32-bit buffer offsets inside one (b, kv head) slice.
  const int64_t esz = (int64_t)elem_bytes(p->dtype), vec = 16 / esz;
  mfma_ok = (prefill_mfma_supported(p->dtype, p->D) || prefill_f32_mfma_supported(p->dtype, p->D)) && p->scale > 0.f &&
                 aligned16(p->q) && aligned16(p->k) && aligned16(p->v) && aligned16(p->out);
  // (offsets from 0x7ffffff0 up are what the half-precision kernel uses as "out of range")
  constexpr int64_t kMaxSliceBytes = 0x7ffffff0;
  mfma_ok = mfma_ok && (int64_t)p->Sk * a.ks[2] * esz < kMaxSliceBytes && (int64_t)p->Sk * a.vs[2] * esz < kMaxSliceBytes;
  mfma_ok = mfma_ok && (!p->q_rope || prefill_mfma_rope_ok(p->D));  // the rotation in registers needs a head dim that fills its tiling
  for (int i = 0; i < 3 && mfma_ok; i++)
    mfma_ok = (a.qs[i] % vec == 0) && (a.ks[i] % vec == 0) && (a.vs[i] % vec == 0) && (a.os[i] % vec == 0);
  return LMH_OK;
}

static int launch_attn(const PrefillArgs &a, int dtype, bool mfma_ok, hipStream_t stream) {
  if (mfma_ok && dtype == LMH_F32) return launch_prefill_f32_mfma(a, stream);
  if (mfma_ok) return launch_prefill_mfma(a, dtype, stream);
  return launch_prefill_valu(a, dtype, stream);
}

int lmh_flash_attn_fwd(const lmh_attn_params *p) {
  PrefillArgs a;
  bool mfma_ok;
  const int rc = attn_args(p, a, mfma_ok);
  return rc != LMH_OK ? rc : launch_attn(a, p->dtype, mfma_ok, (hipStream_t)p->stream);
}

int lmh_flash_attn_plan(const lmh_attn_params *p, char *plan, size_t plan_bytes) {
  if (!plan || plan_bytes < 2) return fail(LMH_E_NULL, "lmh_flash_attn_plan: no room for the description");
  plan[0] = 0;
  g_plan_buf = plan;
  g_plan_bytes = plan_bytes;
  const int rc = lmh_flash_attn_fwd(p);
  g_plan_buf = nullptr;
  return rc;
}

// --------------------------------------------------------------------------------------------
// decode attention
// --------------------------------------------------------------------------------------------
int32_t lmh_decode_auto_splits(int32_t B, int32_t Hkv, int32_t Lmax) {
  if (B <= 0 || Hkv <= 0 || Lmax <= 0) return 0;
  // The chunk (keys per split) is the unit the persistent decode kernel balances its workgroups
  // with: aim for >= 2048 units (4 per resident workgroup) with 128..512 keys each. Shorter chunks
  // only add partial-result slots; longer ones leave the last workgroups of a ragged batch idle.
  const int64_t pairs = (int64_t)B * Hkv;
  int64_t want = (2048 + pairs - 1) / pairs;
  int64_t chunk = (Lmax + want - 1) / want;
  if (chunk < 128) chunk = 128;
  if (chunk > 512) chunk = 512;
  chunk = (chunk + 63) / 64 * 64;
  int64_t splits = (Lmax + chunk - 1) / chunk;
  return (int32_t)(splits < 1 ? 1 : splits);
}

size_t lmh_decode_workspace_bytes(int32_t B, int32_t Hq, int32_t Hkv, int32_t Lmax, int32_t D, int32_t num_splits) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || Lmax <= 0 || D <= 0 || num_splits < 0) return 0;
  if (num_splits == 0) num_splits = lmh_decode_auto_splits(B, Hkv, Lmax);
  if (num_splits == 1) return 0;
  return (size_t)B * Hq * num_splits * (size_t)(D + 2) * sizeof(float);
}

// Where the caller leaves the split count to the library, the matrix-core kernel takes fewer than lmh_decode_auto_splits where
// that is faster (us with that count and with this one, D = 128 bf16 unless named; 190 sizes timed):
//   * one, so that the merge launch and the partials drop out, where a workgroup of a kernel of its own walks a whole pair
//     (decode_by_pairs, steps as well), or where the pairs fill the CUs and the walk is short beside the whole launch: B=16 L=1024 20.8
//     -> 18.7 (L=2100 33.5 -> 32.3, ragged 26.0 -> 28.8), B=64 L=512 ragged 35.1 -> 24.0, L=2100 92 -> 90 (L=4096 169.6 -> 167.6,
//     ragged 121.0 -> 120.6: within what cards differ by); the longer walks only where the last round of pairs is nearly full
//     (B=81 Hkv=4 L=3522 D=64 54.5 -> 58.6);
//   * one unit per CU for few pairs, in chunks long enough for the merge: B=4 Hkv=8 L=2100 19.3 -> 16.0, L=8192 ragged
//     28.4 -> 24.0, B=1 L=8192 19.0 -> 16.4, L=32768 41.4 -> 29.9. From 128 pairs on more units balance ragged batches better
//     (B=16 L=4096 ragged 38.5 with 16, 39.9 with 2).
// Other steps keep their two launches and with them two splits at least; there, few are no better than more.
// The sums are the same fp32 sums in another order, and no less exact for it (the kernel adds a block's share once and holds the
// weights in full): against 64 bits (2-norm, fp32 results) B=4 Hkv=8 L=512 D=128 bf16 1.57e-7 with four splits and 1.55e-7 with
// one, D=64 fp16 1.56e-7 and 1.51e-7, B=1 L=32768 D=64 fp16 2.31e-7 with 256 and 2.13e-7 with 32.
static int32_t decode_splits(const DecodeArgs &a, int32_t most) {
  const int64_t cus = device_cu_count(), pairs = (int64_t)a.B * a.Hkv * ((a.Hq / a.Hkv + 15) / 16), walk = (int64_t)a.Lmax * a.D;
  if (decode_by_pairs(a)) return 1;
  const bool full = pairs * 20 >= (pairs + cus - 1) / cus * cus * 17;
  if (!a.step && ((walk <= 131072 && pairs * 2 >= cus) || (walk <= 262144 && pairs >= cus && full))) return 1;
  const int64_t per_pair = cus / pairs;
  if (per_pair < 4 || per_pair * pairs * 8 < cus * 7) return most;
  const int64_t chunk = std::min(std::max(a.Lmax / 1024 * 64, 128), 512);
  const int64_t chunks = std::max<int64_t>((a.Lmax + chunk - 1) / chunk, a.step ? 2 : 1);
  return (int32_t)std::min({per_pair, chunks, (int64_t)most});
}

// Validation and launch shared by lmh_decode_attn (caller-owned workspace) and lmh_decode_attn_static (the
// library's static scratch): `ws` / `ws_bytes` is the split-KV partial storage, enough for `num_splits`; `choose`: fewer will do.
static int decode_args(const lmh_decode_params *p, const char *fn, int32_t num_splits, void *ws, size_t ws_bytes,
                       const lmh_decode_step_extra *step, DecodeArgs &a, bool choose) {
  a.step = step ? 1 : 0;
  a.q_rope = (step && step->rope) ? 1 : 0;
  a.rope_interleaved = (step && step->pairing == LMH_ROPE_INTERLEAVED) ? 1 : 0;
  a.rope_log2_base = step ? log2f(step->rope_base) : 0.f;
  a.k_new = step ? step->k_new : nullptr;
  a.v_new = step ? step->v_new : nullptr;
  a.out = p->out; a.q = p->q; a.k = p->k_cache; a.v = p->v_cache; a.kv_len = p->kv_len;
  a.B = p->B; a.Hq = p->Hq; a.Hkv = p->Hkv; a.Lmax = p->Lmax; a.D = p->D;
  a.scale = p->scale; a.head_map = p->head_map;
  a.out_f32 = (p->out_f32 != 0 || p->dtype == LMH_F32) ? 1 : 0;
  if (all_zero(p->q_stride, 2)) { a.qs[0] = (int64_t)p->Hq * p->D; a.qs[1] = p->D; }
  else { a.qs[0] = p->q_stride[0]; a.qs[1] = p->q_stride[1]; }
  if (all_zero(p->o_stride, 2)) { a.os[0] = (int64_t)p->Hq * p->D; a.os[1] = p->D; }
  else { a.os[0] = p->o_stride[0]; a.os[1] = p->o_stride[1]; }
  auto fill3 = [&](int64_t *dst, const int64_t *src) {
    if (all_zero(src, 3)) {
      dst[0] = (int64_t)p->Hkv * p->Lmax * p->D; dst[1] = (int64_t)p->Lmax * p->D; dst[2] = p->D;
    } else {
      dst[0] = src[0]; dst[1] = src[1]; dst[2] = src[2];
    }
  };
  fill3(a.ks, p->k_stride);
  fill3(a.vs, p->v_stride);
  // 128-bit loads: every row start must be 16-byte aligned
  const int64_t align_elems = 16 / (int64_t)elem_bytes(p->dtype);
  if (!aligned16(p->k_cache) || !aligned16(p->v_cache))
    return fail(LMH_E_SHAPE, "%s: cache pointers must be 16-byte aligned", fn);
  for (int i = 0; i < 3; i++)
    if (a.ks[i] < 0 || a.vs[i] < 0 || a.ks[i] % align_elems != 0 || a.vs[i] % align_elems != 0)
      return fail(LMH_E_SHAPE, "%s: cache strides must be non-negative multiples of %lld elements", fn,
                  (long long)align_elems);
  if (a.ks[2] < p->D || a.vs[2] < p->D) return fail(LMH_E_SHAPE, "%s: cache row stride smaller than head dim", fn);
  if (a.qs[0] < 0 || a.qs[1] < 0 || a.os[0] < 0 || a.os[1] < 0) return fail(LMH_E_SHAPE, "%s: negative stride", fn);

  // the matrix-core kernel addresses a (b, kv head) slice with 32-bit buffer offsets
  // (a block of 32 rows is addressed even when Lmax is smaller, so bound that too)
  const int64_t rows = p->Lmax > 32 ? p->Lmax : 32;
  const bool slice_fits = rows * a.ks[2] * 2 < 0x7ffffff0 && rows * a.vs[2] * 2 < 0x7ffffff0;
  a.mfma_ok = (p->scale > 0.f && aligned16(p->q) && a.qs[0] % 8 == 0 && a.qs[1] % 8 == 0 && slice_fits) ? 1 : 0;
  a.num_splits = num_splits;
  a.ws_o = nullptr;
  a.ws_ml = nullptr;
  if (num_splits > 1) {
    const size_t need = lmh_decode_workspace_bytes(p->B, p->Hq, p->Hkv, p->Lmax, p->D, num_splits);
    if (!ws || ws_bytes < need)
      return fail(LMH_E_WORKSPACE, "%s: workspace of %zu bytes needed for %d splits, got %zu", fn, need,
                  num_splits, ws ? ws_bytes : (size_t)0);
    if (!aligned16(ws)) return fail(LMH_E_WORKSPACE, "%s: workspace must be 16-byte aligned", fn);
    if (choose) a.num_splits = decode_mfma_takes(a, p->dtype) ? decode_splits(a, num_splits) : decode_valu_splits(a, p->dtype, num_splits);
  }
  a.chunk = decode_chunk_for(p->Lmax, a.num_splits);
  if (a.num_splits > 1) {
    a.ws_o = reinterpret_cast<float *>(ws);
    a.ws_ml = a.ws_o + (size_t)p->B * p->Hq * a.num_splits * p->D;
  }
  if (step) {
    // two launches only where the split kernel can rotate q in registers and the slice fits its addressing
    if (!a.mfma_ok || !decode_mfma_supported(p->dtype, p->D, p->B))
      return fail(LMH_E_UNSUPPORTED, "%s: needs the matrix-core decode kernel (fp16 / bf16, head dim 64, 96, 128 or 256, aligned q, "
                  "batch <= 1024); use lmh_kv_append + lmh_decode_attn", fn);
    if (a.q_rope && !decode_mfma_rope_ok(p->D, a.rope_interleaved))
      return fail(LMH_E_UNSUPPORTED, "%s: head dim %d with the half-split pairing cannot be rotated in registers; use lmh_kv_append + "
                  "lmh_decode_attn", fn, p->D);
  }
  return LMH_OK;
}

static int decode_launch(const lmh_decode_params *p, const char *fn, int32_t num_splits, void *ws, size_t ws_bytes, bool choose) {
  DecodeArgs a;
  const int rc = decode_args(p, fn, num_splits, ws, ws_bytes, nullptr, a, choose);
  return rc != LMH_OK ? rc : launch_decode(a, p->dtype, (hipStream_t)p->stream);
}

static int decode_check(const lmh_decode_params *p, const char *fn) {
  if (!p) return fail(LMH_E_NULL, "%s: null params", fn);
  if (!p->out || !p->q || !p->k_cache || !p->v_cache) return fail(LMH_E_NULL, "%s: null tensor pointer", fn);
  if (p->B <= 0 || p->Hq <= 0 || p->Hkv <= 0 || p->Lmax <= 0 || p->D <= 0)
    return fail(LMH_E_SHAPE, "%s: non-positive dimension (B=%d Hq=%d Hkv=%d Lmax=%d D=%d)", fn, p->B, p->Hq,
                p->Hkv, p->Lmax, p->D);
  if (p->Hq % p->Hkv != 0) return fail(LMH_E_SHAPE, "%s: Hq=%d is not a multiple of Hkv=%d", fn, p->Hq, p->Hkv);
  if (p->dtype != LMH_F32 && p->dtype != LMH_F16 && p->dtype != LMH_BF16)
    return fail(LMH_E_UNSUPPORTED, "%s: unknown dtype %d", fn, p->dtype);
  if (p->head_map != LMH_HEADMAP_INTERLEAVED && p->head_map != LMH_HEADMAP_BLOCKED)
    return fail(LMH_E_UNSUPPORTED, "%s: unknown head_map %d", fn, p->head_map);
  const int vec = p->dtype == LMH_F32 ? 4 : 8;
  if (p->D % vec != 0 || p->D > 256)
    return fail(LMH_E_UNSUPPORTED, "%s: head dim %d must be a multiple of %d and <= 256", fn, p->D, vec);
  if (p->num_splits < 0) return fail(LMH_E_SHAPE, "%s: negative num_splits", fn);
  if (!(p->scale == p->scale)) return fail(LMH_E_SHAPE, "%s: scale is NaN", fn);
  return LMH_OK;
}

int lmh_decode_attn(const lmh_decode_params *p) {
  const int rc = decode_check(p, "lmh_decode_attn");
  if (rc != LMH_OK) return rc;
  const int32_t splits = p->num_splits == 0 ? lmh_decode_auto_splits(p->B, p->Hkv, p->Lmax) : p->num_splits;
  return decode_launch(p, "lmh_decode_attn", splits, p->workspace, p->workspace_bytes, p->num_splits == 0);
}

int lmh_decode_plan(const lmh_decode_params *p, char *plan, size_t plan_bytes) {
  if (!plan || plan_bytes < 2) return fail(LMH_E_NULL, "lmh_decode_plan: no room for the description");
  plan[0] = 0;
  g_plan_buf = plan;
  g_plan_bytes = plan_bytes;
  const int rc = lmh_decode_attn(p);
  g_plan_buf = nullptr;
  return rc;
}

int32_t lmh_decode_step_splits(int32_t B, int32_t Hkv, int32_t Lmax) {
  const int32_t s = lmh_decode_auto_splits(B, Hkv, Lmax);
  return s == 0 ? 0 : (s < 2 ? 2 : s);  // the merge launch always runs: it is what adds the new row
}

static int decode_step_args(const lmh_decode_params *p, const lmh_decode_step_extra *x, DecodeArgs &a) {
  const char *fn = "lmh_decode_step";
  const int rc = decode_check(p, fn);
  if (rc != LMH_OK) return rc;
  if (!x || !x->k_new || !x->v_new) return fail(LMH_E_NULL, "%s: null k_new / v_new", fn);
  if (!p->kv_len) return fail(LMH_E_NULL, "%s: kv_len (the rows already in the caches) is required", fn);
  if (p->dtype == LMH_F32) return fail(LMH_E_UNSUPPORTED, "%s: fp16 / bf16 only; use lmh_kv_append + lmh_decode_attn", fn);
  if (x->pairing != LMH_ROPE_HALF_SPLIT && x->pairing != LMH_ROPE_INTERLEAVED)
    return fail(LMH_E_UNSUPPORTED, "%s: unknown rope pairing %d", fn, x->pairing);
  if (x->rope && !(x->rope_base > 1.f)) return fail(LMH_E_SHAPE, "%s: rope base must be > 1", fn);
  if (p->num_splits == 1) return fail(LMH_E_SHAPE, "%s: num_splits must be 0 or >= 2", fn);
  const int32_t splits = p->num_splits == 0 ? lmh_decode_step_splits(p->B, p->Hkv, p->Lmax) : p->num_splits;
  return decode_args(p, fn, splits, p->workspace, p->workspace_bytes, x, a, p->num_splits == 0);
}

int lmh_decode_step(const lmh_decode_params *p, const lmh_decode_step_extra *x) {
  DecodeArgs a;
  const int rc = decode_step_args(p, x, a);
  return rc != LMH_OK ? rc : launch_decode(a, p->dtype, (hipStream_t)p->stream);
}

// --------------------------------------------------------------------------------------------
// decode attention for callers that cannot allocate: the split-KV partials live in a static device array
// --------------------------------------------------------------------------------------------
size_t lmh_static_scratch_bytes(void) { return LMH_STATIC_SCRATCH_BYTES; }

int32_t lmh_decode_static_splits(int32_t B, int32_t Hq, int32_t Hkv, int32_t Lmax, int32_t D) {
  int32_t splits = lmh_decode_auto_splits(B, Hkv, Lmax);
  if (splits <= 0 || Hq <= 0 || D <= 0) return 0;
  // halve the split count (double the keys per split) until the partials fit; one split needs none
  while (splits > 1 && lmh_decode_workspace_bytes(B, Hq, Hkv, Lmax, D, splits) > LMH_STATIC_SCRATCH_BYTES)
    splits = (splits + 1) / 2;
  return splits;
}

int lmh_decode_attn_static(const lmh_decode_params *p) {
  const char *fn = "lmh_decode_attn_static";
  const int rc = decode_check(p, fn);
  if (rc != LMH_OK) return rc;
  const int32_t splits = p->num_splits == 0 ? lmh_decode_static_splits(p->B, p->Hq, p->Hkv, p->Lmax, p->D) : p->num_splits;
  const size_t need = lmh_decode_workspace_bytes(p->B, p->Hq, p->Hkv, p->Lmax, p->D, splits);
  if (need > LMH_STATIC_SCRATCH_BYTES)
    return fail(LMH_E_WORKSPACE,
                "%s: %d splits of B=%d Hq=%d D=%d need %zu bytes of partials, the static scratch holds %zu; "
                "pass num_splits = 0 or a smaller count, or use lmh_decode_attn with a workspace",
                fn, splits, p->B, p->Hq, p->D, need, (size_t)LMH_STATIC_SCRATCH_BYTES);
  void *ws = nullptr;
  if (splits > 1) {
    const int rc_ws = static_scratch_for_current_device(&ws);
    if (rc_ws != LMH_OK) return rc_ws;
    const int rc_claim = static_scratch_claim((hipStream_t)p->stream, fn);
    if (rc_claim != LMH_OK) return rc_claim;
  }
  // Nothing in the scratch has to start at zero: every partial slot the merge kernel reads was written by
  // the split kernel of the same call (a result, or the "empty" marker), so no clearing is enqueued.
  const int rc_launch = decode_launch(p, fn, splits, ws, LMH_STATIC_SCRATCH_BYTES, false);
  if (rc_launch == LMH_OK && splits > 1) static_scratch_mark((hipStream_t)p->stream);
  return rc_launch;
}

// --------------------------------------------------------------------------------------------
// rotary embedding and KV-cache append
// --------------------------------------------------------------------------------------------
int lmh_rope(const lmh_rope_params *p) {
  if (!p) return fail(LMH_E_NULL, "lmh_rope: null params");
  if (!p->out || !p->x) return fail(LMH_E_NULL, "lmh_rope: null tensor pointer");
  if (p->B <= 0 || p->H <= 0 || p->S <= 0 || p->D <= 0)
    return fail(LMH_E_SHAPE, "lmh_rope: non-positive dimension (B=%d H=%d S=%d D=%d)", p->B, p->H, p->S, p->D);
  if (p->D % 2 != 0) return fail(LMH_E_SHAPE, "lmh_rope: head dim %d must be even", p->D);
  if (p->dtype != LMH_F32 && p->dtype != LMH_F16 && p->dtype != LMH_BF16)
    return fail(LMH_E_UNSUPPORTED, "lmh_rope: unknown dtype %d", p->dtype);
  if (p->pairing != LMH_ROPE_HALF_SPLIT && p->pairing != LMH_ROPE_INTERLEAVED)
    return fail(LMH_E_UNSUPPORTED, "lmh_rope: unknown pairing %d", p->pairing);
  if (!(p->base > 0.f)) return fail(LMH_E_SHAPE, "lmh_rope: base must be positive");
  RopeArgs a;
  a.out = p->out; a.x = p->x; a.pos0 = p->pos0; a.prev_seq = p->prev_seq;
  a.B = p->B; a.H = p->H; a.S = p->S; a.D = p->D;
  auto fill = [&](int64_t *dst, const int64_t *src) {
    if (all_zero(src, 3)) { dst[0] = (int64_t)p->H * p->S * p->D; dst[1] = (int64_t)p->S * p->D; dst[2] = p->D; }
    else { dst[0] = src[0]; dst[1] = src[1]; dst[2] = src[2]; }
  };
  fill(a.xs, p->x_stride);
  fill(a.os, p->o_stride);
  for (int i = 0; i < 3; i++)
    if (a.xs[i] < 0 || a.os[i] < 0) return fail(LMH_E_SHAPE, "lmh_rope: negative stride");
  a.log2_base = log2f(p->base);
  a.interleaved = p->pairing == LMH_ROPE_INTERLEAVED;
  return launch_rope(a, p->dtype, (hipStream_t)p->stream);
}

static int append_args(const lmh_kv_append_params *p, KvAppendArgs &a) {
  if (!p) return fail(LMH_E_NULL, "lmh_kv_append: null params");
  if (!p->k_cache || !p->v_cache || !p->k_new || !p->v_new) return fail(LMH_E_NULL, "lmh_kv_append: null tensor pointer");
  if (p->B <= 0 || p->Hkv <= 0 || p->T <= 0 || p->D <= 0 || p->Lmax <= 0)
    return fail(LMH_E_SHAPE, "lmh_kv_append: non-positive dimension (B=%d Hkv=%d T=%d D=%d Lmax=%d)", p->B, p->Hkv, p->T,
                p->D, p->Lmax);
  if (p->dtype != LMH_F32 && p->dtype != LMH_F16 && p->dtype != LMH_BF16)
    return fail(LMH_E_UNSUPPORTED, "lmh_kv_append: unknown dtype %d", p->dtype);
  if (p->q_rope && p->Hq <= 0) return fail(LMH_E_SHAPE, "lmh_kv_append: q_rope given with Hq=%d", p->Hq);
  if (p->rope_k || p->q_rope) {
    if (p->D % 2 != 0) return fail(LMH_E_SHAPE, "lmh_kv_append: head dim %d must be even for the rotary embedding", p->D);
    if (p->pairing != LMH_ROPE_HALF_SPLIT && p->pairing != LMH_ROPE_INTERLEAVED)
      return fail(LMH_E_UNSUPPORTED, "lmh_kv_append: unknown pairing %d", p->pairing);
    if (!(p->base > 0.f)) return fail(LMH_E_SHAPE, "lmh_kv_append: base must be positive");
  }
  a.k_cache = p->k_cache; a.v_cache = p->v_cache; a.k_new = p->k_new; a.v_new = p->v_new;
  a.pos = p->pos; a.pos_all = p->pos_all;
  a.B = p->B; a.Hkv = p->Hkv; a.T = p->T; a.D = p->D; a.Lmax = p->Lmax;
  auto fill = [&](int64_t *dst, const int64_t *src) {
    if (all_zero(src, 3)) { dst[0] = (int64_t)p->Hkv * p->Lmax * p->D; dst[1] = (int64_t)p->Lmax * p->D; dst[2] = p->D; }
    else { dst[0] = src[0]; dst[1] = src[1]; dst[2] = src[2]; }
  };
  fill(a.ks, p->k_stride);
  fill(a.vs, p->v_stride);
  for (int i = 0; i < 3; i++)
    if (a.ks[i] < 0 || a.vs[i] < 0) return fail(LMH_E_SHAPE, "lmh_kv_append: negative stride");
  if (a.ks[2] < p->D || a.vs[2] < p->D) return fail(LMH_E_SHAPE, "lmh_kv_append: cache row stride smaller than head dim");
  a.rope_k = p->rope_k ? 1 : 0;
  a.interleaved = p->pairing == LMH_ROPE_INTERLEAVED;
  a.log2_base = (p->rope_k || p->q_rope) ? log2f(p->base) : 0.f;
  a.q = p->q_rope;
  a.Hq = p->q_rope ? p->Hq : 0;
  return LMH_OK;
}

int lmh_kv_append(const lmh_kv_append_params *p) {
  KvAppendArgs a;
  const int rc = append_args(p, a);
  return rc != LMH_OK ? rc : launch_kv_append(a, p->dtype, (hipStream_t)p->stream);
}

// --------------------------------------------------------------------------------------------
// the nodes around attention
// --------------------------------------------------------------------------------------------
static bool graph_dtype(int d) { return d == LMH_F32 || d == LMH_F16 || d == LMH_BF16 || d == LMH_I32; }

static int matmul_args(const lmh_matmul_params *ps, int32_t n, MatmulArgs &args) {
  static_assert(LMH_MATMUL_GROUP == kMatmulGroup, "header and kernel agree");
  if (!ps) return fail(LMH_E_NULL, "lmh_matmul: null params");
  if (n < 1 || n > LMH_MATMUL_GROUP) return fail(LMH_E_SHAPE, "lmh_matmul: %d products, 1 to %d fit a launch", n, LMH_MATMUL_GROUP);
  for (int i = 0; i < n; i++) {
    const lmh_matmul_params &p = ps[i];
    if (!p.c || !p.a || !p.b) return fail(LMH_E_NULL, "lmh_matmul: null tensor pointer");
    if (p.batch <= 0 || p.M <= 0 || p.N <= 0 || p.K <= 0)
      return fail(LMH_E_SHAPE, "lmh_matmul: non-positive dimension (batch=%d M=%d N=%d K=%d)", p.batch, p.M, p.N, p.K);
    if (!graph_dtype(p.a_dtype) || !graph_dtype(p.b_dtype) || !graph_dtype(p.c_dtype) || p.c_dtype == LMH_I32 ||
        (p.bias && !graph_dtype(p.bias_dtype)))
      return fail(LMH_E_UNSUPPORTED, "lmh_matmul: unknown element type");
    for (int d = 0; d < 3; d++)
      if (p.a_stride[d] < 0 || p.b_stride[d] < 0) return fail(LMH_E_SHAPE, "lmh_matmul: negative stride");
    if (p.heads < 0 || (p.heads > 0 && (p.batch != 1 || p.seq <= 0 || p.M % p.seq != 0 || p.N % p.heads != 0)))
      return fail(LMH_E_SHAPE, "lmh_matmul: %d heads of %d rows do not divide c (batch=%d M=%d N=%d)", p.heads, p.seq, p.batch, p.M, p.N);
    MatmulProblem &q = args.p[i];
    q.c = p.c; q.a = p.a; q.b = p.b; q.bias = p.bias;
    q.batch = p.batch; q.M = p.M; q.N = p.N; q.K = p.K;
    for (int d = 0; d < 3; d++) { q.as[d] = p.a_stride[d]; q.bs[d] = p.b_stride[d]; }
    q.a_dtype = p.a_dtype; q.b_dtype = p.b_dtype; q.c_dtype = p.c_dtype; q.bias_dtype = p.bias_dtype;
    q.heads = p.heads; q.seq = p.heads ? p.seq : 1;
    // 16-byte chunks along the contraction, addressed with 32-bit byte offsets inside a tile of 64 rows of a / inside b
    constexpr int64_t kMaxBytes = 0x7ffffff0;
    q.a_vec = p.a_dtype == LMH_F32 && p.a_stride[2] == 1 && p.K % 4 == 0 && p.a_stride[0] % 4 == 0 && p.a_stride[1] % 4 == 0 && aligned16(p.a) &&
              (64 * p.a_stride[1] + p.K) * 4 < kMaxBytes;
    q.b_vec = p.b_dtype == LMH_F32 && p.b_stride[1] == 1 && p.K % 4 == 0 && p.b_stride[0] % 4 == 0 && p.b_stride[2] % 4 == 0 && aligned16(p.b) &&
              ((int64_t)p.N * p.b_stride[2] + p.K) * 4 < kMaxBytes;
    q.b_by_column = !q.b_vec && p.b_stride[2] == 1 && p.b_stride[1] != 1;
  }
  return LMH_OK;
}

int lmh_matmul(const lmh_matmul_params *ps, int32_t n, void *stream) {
  MatmulArgs args = {};
  const int rc = matmul_args(ps, n, args);
  return rc != LMH_OK ? rc : launch_matmul(args, n, (hipStream_t)stream);
}

int lmh_map(const lmh_map_params *p, void *stream) {
  static_assert(LMH_MAP_DIMS == kMapDims, "header and kernel agree");
  if (!p) return fail(LMH_E_NULL, "lmh_map: null params");
  if (!p->out || !p->a) return fail(LMH_E_NULL, "lmh_map: null tensor pointer");
  if (p->n_dims < 1 || p->n_dims > LMH_MAP_DIMS) return fail(LMH_E_SHAPE, "lmh_map: %d dimensions, 1 to %d are taken", p->n_dims, LMH_MAP_DIMS);
  if (!graph_dtype(p->out_dtype) || p->out_dtype == LMH_I32 || !graph_dtype(p->a_dtype) || (p->b && !graph_dtype(p->b_dtype)))
    return fail(LMH_E_UNSUPPORTED, "lmh_map: unknown element type");
  MapArgs a = {};
  a.out = p->out; a.a = p->a; a.b = p->b;
  a.n_dims = p->n_dims;
  a.out_dtype = p->out_dtype; a.a_dtype = p->a_dtype; a.b_dtype = p->b_dtype;
  for (int d = 0; d < p->n_dims; d++) {
    if (p->dims[d] <= 0) return fail(LMH_E_SHAPE, "lmh_map: non-positive dimension");
    if (p->a_stride[d] < 0 || (p->b && p->b_stride[d] < 0)) return fail(LMH_E_SHAPE, "lmh_map: negative stride");
    a.dims[d] = p->dims[d];
    a.as[d] = p->a_stride[d];
    a.bs[d] = p->b ? p->b_stride[d] : 0;
  }
  return launch_map(a, (hipStream_t)stream);
}

static bool meet(const void *x, size_t nx, const void *y, size_t ny) {
  return (uintptr_t)x < (uintptr_t)y + ny && (uintptr_t)y < (uintptr_t)x + nx;
}

int lmh_copy_many(void *const *dst, const void *const *src, const size_t *bytes, int32_t n, void *stream) {
  static_assert(LMH_COPY_MANY == kCopyMany, "header and kernel agree");
  if (n < 0) return fail(LMH_E_SHAPE, "lmh_copy_many: negative count");
  if (n > 0 && (!dst || !src || !bytes)) return fail(LMH_E_NULL, "lmh_copy_many: null list");
  for (int32_t i = 0; i < n; i++)
    if (bytes[i] && (!dst[i] || !src[i])) return fail(LMH_E_NULL, "lmh_copy_many: null pointer");
  CopyManyArgs a = {};
  int m = 0;  // ranges of the launch that is being put together
  auto launch = [&]() {
    const int count = m;
    m = 0;
    return count ? launch_copy_many(a, count, (hipStream_t)stream) : LMH_OK;
  };
  for (int32_t i = 0; i < n; i++) {
    const size_t len = bytes[i];
    if (!len || dst[i] == src[i]) continue;
    // a range that meets one of the launch waits for it
    bool wait = m == LMH_COPY_MANY;
    for (int j = 0; j < m && !wait; j++)
      wait = meet(dst[i], len, a.dst[j], a.bytes[j]) || meet(dst[i], len, a.src[j], a.bytes[j]) || meet(src[i], len, a.dst[j], a.bytes[j]);
    const bool itself = meet(dst[i], len, src[i], len);
    if (wait || itself) {
      const int rc = launch();
      if (rc != LMH_OK) return rc;
    }
    if (itself) {  // the runtime's copy, as lmh_memcpy_d2d
      LMH_HIP_TRY(hipMemcpyAsync(dst[i], src[i], len, hipMemcpyDeviceToDevice, (hipStream_t)stream));
      continue;
    }
    a.dst[m] = dst[i]; a.src[m] = src[i]; a.bytes[m] = (int64_t)len;
    m++;
  }
  return launch();
}

}  // extern "C"

// --------------------------------------------------------------------------------------------
// launches that take their operands from the caller's arrays and copy those into the graph's buffers on the side
// --------------------------------------------------------------------------------------------
namespace {

// The bytes from the first element to the last one of a tensor.
template <int N>
int64_t extent(const int64_t (&stride)[N], std::initializer_list<int64_t> dims, int64_t D, int64_t esz) {
  int64_t last = D - 1;
  int i = 0;
  for (int64_t n : dims) last += (n - 1) * stride[i++];
  return (last + 1) * esz;
}

// Copies whose order among themselves and against the launch that carries them does not matter.
struct Feed {
  CopyManyArgs a = {};
  int n = 0;

  // Whether the copies may all run at once; from then on `a` holds those that move something.
  bool apart(void *const *dst, const void *const *src, const size_t *bytes, int32_t count) {
    if (count < 0 || (count > 0 && (!dst || !src || !bytes))) return false;
    for (int32_t i = 0; i < count; i++) {
      if (!bytes[i] || dst[i] == src[i]) continue;
      if (!dst[i] || !src[i] || n == kCopyMany || touches(dst[i], bytes[i]) || writes(src[i], bytes[i]) || meet(dst[i], bytes[i], src[i], bytes[i]))
        return false;
      a.dst[n] = dst[i]; a.src[n] = src[i]; a.bytes[n] = (int64_t)bytes[i];
      n++;
    }
    return true;
  }
  bool writes(const void *p, int64_t bytes) const {
    for (int j = 0; j < n; j++)
      if (meet(p, bytes, a.dst[j], a.bytes[j])) return true;
    return false;
  }
  bool touches(const void *p, int64_t bytes) const {
    for (int j = 0; j < n; j++)
      if (meet(p, bytes, a.src[j], a.bytes[j])) return true;
    return writes(p, bytes);
  }
  // Sends an operand inside one of the destinations to where its values come from, which has to be as aligned as the
  // destination is; false for one that lies across an end.
  template <typename T>
  bool redirect(T *&p, int64_t bytes) const {
    for (int j = 0; j < n; j++) {
      if (!meet(p, bytes, a.dst[j], a.bytes[j])) continue;
      const intptr_t at = (intptr_t)p - (intptr_t)a.dst[j];
      if (at < 0 || at + bytes > a.bytes[j] || !aligned16(a.src[j]) || !aligned16(a.dst[j])) return false;
      p = (T *)((const char *)a.src[j] + at);
      return true;
    }
    return true;
  }
  // Copies that a launch has workgroups for, beside its own.
  bool some() {
    const int64_t blocks = number_copy_blocks(a, n);
    return blocks > 0 && blocks <= 32768;
  }
  // The copy that fills exactly this tensor, both ends 16-byte aligned; -1: there is none.
  int of(const void *p, int64_t bytes) const {
    for (int j = 0; j < n; j++)
      if (p == a.dst[j] && bytes == a.bytes[j] && aligned16(a.dst[j]) && aligned16(a.src[j])) return j;
    return -1;
  }
  void drop(int j) {
    n--;
    a.dst[j] = a.dst[n]; a.src[j] = a.src[n]; a.bytes[j] = a.bytes[n];
  }
};

}  // namespace

extern "C" {

int lmh_decode_step_fed(const lmh_decode_params *p, const lmh_decode_step_extra *x, void *const *dst, const void *const *src,
                        const size_t *bytes, int32_t n) {
  DecodeArgs a;
  Feed feed;
  if (feed.apart(dst, src, bytes, n) && feed.n && decode_step_args(p, x, a) == LMH_OK) {
    const int64_t esz = (int64_t)elem_bytes(p->dtype), rows = (int64_t)p->B * p->Hkv * p->D * esz;
    bool ok = feed.some() && !feed.touches(a.out, extent(a.os, {p->B, p->Hq}, p->D, a.out_f32 ? 4 : esz)) &&
              !feed.touches(a.k, extent(a.ks, {p->B, p->Hkv, p->Lmax}, p->D, esz)) &&
              !feed.touches(a.v, extent(a.vs, {p->B, p->Hkv, p->Lmax}, p->D, esz)) &&
              !feed.touches(a.ws_o, (int64_t)lmh_decode_workspace_bytes(p->B, p->Hq, p->Hkv, p->Lmax, p->D, a.num_splits));
    ok = ok && feed.redirect(a.q, extent(a.qs, {p->B, p->Hq}, p->D, esz)) && feed.redirect(a.k_new, rows) &&
         feed.redirect(a.v_new, rows) && feed.redirect(a.kv_len, (int64_t)p->B * 4);
    if (ok) return launch_decode(a, p->dtype, (hipStream_t)p->stream, &feed.a, feed.n);
  }
  const int rc = lmh_copy_many(dst, src, bytes, n, p ? p->stream : nullptr);
  return rc != LMH_OK ? rc : lmh_decode_step(p, x);
}

// Lets an attention launch read its queries from the caller's array and store them itself: under a causal mask on the
// 16-bit matrix-core kernels up to head dim 128, whole contiguous tensors that nothing of this launch or the append in front of it lies in.
static void attention_stores_queries(const lmh_kv_append_params *p, Feed &feed, PrefillArgs &f, int dtype, bool mfma_ok, QueryCopy &queries) {
#ifdef LMH_W64_KERNEL
  return;
#endif
  const int64_t esz = (int64_t)elem_bytes(dtype), bytes = (int64_t)f.B * f.Hq * f.Sq * f.D * esz;
  if (!mfma_ok || dtype == LMH_F32 || !f.causal || f.D > 128 || f.qs[2] != f.D || f.qs[1] != (int64_t)f.Sq * f.D || f.qs[0] != (int64_t)f.Hq * f.Sq * f.D)
    return;
  const int j = feed.of(f.q, bytes);
  if (j < 0) return;
  const int64_t rows = (int64_t)p->B * p->Hkv * p->T * p->D * (int64_t)elem_bytes(p->dtype);
  const struct { const void *at; int64_t bytes; } others[] = {
      {f.out, extent(f.os, {f.B, f.Hq, f.Sq}, f.D, f.out_f32 ? 4 : esz)}, {f.k, extent(f.ks, {f.B, f.Hkv, f.Sk}, f.D, esz)},
      {f.v, extent(f.vs, {f.B, f.Hkv, f.Sk}, f.D, esz)}, {f.kv_len, (int64_t)f.B * 4}, {f.q_pos0, (int64_t)f.B * 4},
      {p->k_new, rows}, {p->v_new, rows}, {p->pos, (int64_t)p->B * 4}};
  for (const auto &o : others)
    if (o.at && (meet(o.at, o.bytes, feed.a.dst[j], bytes) || meet(o.at, o.bytes, feed.a.src[j], bytes))) return;
  f.q = queries.src = feed.a.src[j];
  queries.dst = feed.a.dst[j];
  feed.drop(j);
}

int lmh_kv_append_fed(const lmh_kv_append_params *p, const lmh_attn_params *attn, void *const *dst, const void *const *src,
                      const size_t *bytes, int32_t n) {
  KvAppendArgs a;
  PrefillArgs f;
  bool mfma_ok = false;
  Feed feed;
  if (feed.apart(dst, src, bytes, n) && append_args(p, a) == LMH_OK &&
      (!attn || (attn->stream == p->stream && attn_args(attn, f, mfma_ok) == LMH_OK))) {
    const int64_t esz = (int64_t)elem_bytes(p->dtype), rows = (int64_t)p->B * p->Hkv * p->T * p->D * esz;
    bool ok = feed.some() && !feed.touches(a.k_cache, extent(a.ks, {p->B, p->Hkv, p->Lmax}, p->D, esz)) &&
              !feed.touches(a.v_cache, extent(a.vs, {p->B, p->Hkv, p->Lmax}, p->D, esz));
    if (ok && a.q) {  // rotated on the way from the caller's array, where that is all that is made of it
      const int64_t q_bytes = (int64_t)p->B * p->Hq * p->T * p->D * esz;
      const int j = feed.of(a.q, q_bytes);
      ok = j >= 0 && !meet(a.q, q_bytes, p->k_new, rows) && !meet(a.q, q_bytes, p->v_new, rows) &&
           !(p->pos && meet(a.q, q_bytes, p->pos, (int64_t)p->B * 4));
      if (ok) a.q_from = feed.a.src[j], feed.drop(j);
    }
    ok = ok && feed.redirect(a.k_new, rows) && feed.redirect(a.v_new, rows) && (!a.pos || feed.redirect(a.pos, (int64_t)p->B * 4));
    if (ok) {
      QueryCopy queries;
      if (attn) attention_stores_queries(p, feed, f, attn->dtype, mfma_ok, queries);
      const int rc = launch_kv_append(a, p->dtype, (hipStream_t)p->stream, &feed.a, feed.n);
      if (rc != LMH_OK || !attn) return rc;
      return queries.dst ? launch_prefill_mfma(f, attn->dtype, (hipStream_t)p->stream, queries) : launch_attn(f, attn->dtype, mfma_ok, (hipStream_t)p->stream);
    }
  }
  int rc = lmh_copy_many(dst, src, bytes, n, p ? p->stream : nullptr);
  if (rc == LMH_OK) rc = lmh_kv_append(p);
  return rc != LMH_OK || !attn ? rc : lmh_flash_attn_fwd(attn);
}

int lmh_matmul_fed(const lmh_matmul_params *ps, int32_t n, void *stream, void *const *dst, const void *const *src, const size_t *bytes,
                   int32_t n_copies) {
  MatmulArgs args = {};
  Feed feed;
  if (feed.apart(dst, src, bytes, n_copies) && matmul_args(ps, n, args) == LMH_OK && feed.some()) {
    bool ok = true;
    for (int i = 0; i < n && ok; i++) {
      MatmulProblem &q = args.p[i];
      auto size = [](int dtype) -> int64_t { return dtype == LMH_F32 || dtype == LMH_I32 ? 4 : 2; };
      ok = !feed.touches(q.c, (int64_t)q.batch * q.M * q.N * size(q.c_dtype)) &&
           feed.redirect(q.a, ((q.batch - 1) * q.as[0] + (q.M - 1) * q.as[1] + (q.K - 1) * q.as[2] + 1) * size(q.a_dtype)) &&
           feed.redirect(q.b, ((q.batch - 1) * q.bs[0] + (q.K - 1) * q.bs[1] + (q.N - 1) * q.bs[2] + 1) * size(q.b_dtype)) &&
           (!q.bias || feed.redirect(q.bias, q.N * size(q.bias_dtype)));
    }
    if (ok) return launch_matmul(args, n, (hipStream_t)stream, &feed.a, feed.n);
  }
  const int rc = lmh_copy_many(dst, src, bytes, n_copies, stream);
  return rc != LMH_OK ? rc : lmh_matmul(ps, n, stream);
}

}  // extern "C"
