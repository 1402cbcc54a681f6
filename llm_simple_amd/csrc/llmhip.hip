// C ABI of libllmhip.so (declared in include/llmhip.h): argument validation,
// dispatch to the gfx950 kernels, and thin wrappers over the HIP runtime so
// that the C++ device layer above needs no HIP header.
#include "../../include/llmhip.h"

#include <hip/hip_runtime.h>

#include <mutex>

#include "kernels.hpp"
#include "stream_scratch.hpp"

using namespace llmhip;

namespace {

constexpr int kMaxDecodeCols = 16;
constexpr int kMaxDecodeSplits = 256;

inline hipStream_t as_stream(void *s) { return static_cast<hipStream_t>(s); }
inline int from_hip(hipError_t e) { return e == hipSuccess ? LLMHIP_OK : (int)e; }
inline bool dtype_ok(int dt) { return dt == LLMHIP_DT_FLOAT16 || dt == LLMHIP_DT_BFLOAT16; }
// every kernel moves 16-byte pieces: a misaligned base pointer would fault on the device
inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
template <typename... P> inline bool all_aligned16(P... ptrs) { return (aligned16(ptrs) && ...); }

// Split-KV scratch for the entry points that mirror the reference signatures
// and therefore have no workspace argument: see stream_scratch.hpp.  It goes with
// llmhip_stream_destroy / llmhip_release_internal_workspace.
class OnDevice {  // makes a device the current one for a while
 public:
  explicit OnDevice(int device) {
    if (hipGetDevice(&before_) == hipSuccess && before_ != device && hipSetDevice(device) == hipSuccess) moved_ = true;
  }
  ~OnDevice() {
    if (moved_) (void)hipSetDevice(before_);
  }

 private:
  int before_ = 0;
  bool moved_ = false;
};
struct HipScratch {
  // (of the null stream and its likes: the current device)
  static int device_of(void *stream) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) (void)hipGetLastError();
    const hipStream_t s = as_stream(stream);
    hipDevice_t of_stream;
    if (s == nullptr || s == hipStreamLegacy || s == hipStreamPerThread) return device;
    if (hipStreamGetDevice(s, &of_stream) == hipSuccess) return of_stream;
    (void)hipGetLastError();
    return device;
  }
  // hipMalloc that another stream's capture does not forbid.
  static int allocate(int device, void **ptr, size_t bytes) {
    const OnDevice on(device);
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    const hipError_t e = hipMalloc(ptr, bytes);
    if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) (void)hipGetLastError();  // handled here: not for the next launch to report
    return (int)e;
  }
  static int release(void *ptr) { return (int)hipFree(ptr); }
  static bool capturing(void *stream) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(as_stream(stream), &cap) != hipSuccess) (void)hipGetLastError();
    return cap != hipStreamCaptureStatusNone;
  }
  static void wait_stream(int device, void *stream) {
    const OnDevice on(device);
    (void)hipStreamSynchronize(as_stream(stream));
  }
  static int wait_device(int device) {
    const OnDevice on(device);
    return (int)hipDeviceSynchronize();
  }
};
std::mutex g_scratch_mu;
// Partials; and what workgroups of an eager launch pass each other, which captured launches do not.  A captured graph keeps its stream's partials
// buffer and may be replayed on any other stream: calls that need no partials stay safe beside it.
ScratchTable<HipScratch> g_scratch, g_exchange;

int attn_common(void *out, const void *q, const void *k, const void *v, int m, int n,
                int offset, int group_size, int kv_head_num, int head_dim, int dt,
                void *stream) {
  if (!out || !q || !k || !v || !all_aligned16(out, q, k, v)) return LLMHIP_ERR_INVALID_ARG;
  if (m < 1 || n < 1 || offset < 0 || group_size < 1 || kv_head_num < 1)
    return LLMHIP_ERR_INVALID_ARG;
  if (!dtype_ok(dt)) return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128) return LLMHIP_ERR_UNSUPPORTED;
  // grid dimensions and the 32-bit row offsets of the tile loader
  if (kv_head_num > 65535 || (long long)group_size * kv_head_num > 65535) return LLMHIP_ERR_UNSUPPORTED;
  if ((long long)m * group_size <= kMaxDecodeCols) {
    // few query rows: stream the cache once with the split-KV kernel
    const int n_vis = (n < m + offset) ? n : m + offset;  // keys any row can see
    int splits = flash_decode_default_splits(1, n_vis, kv_head_num, m * group_size);
    const size_t need = flash_decode_workspace_bytes(1, m, group_size, kv_head_num, splits);
    if (!need)
      return from_hip(launch_flash_decode(out, q, k, v, nullptr, 0, 1, m, n_vis, offset, n_vis, group_size,
                                          kv_head_num, splits, dt, as_stream(stream)));
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    StreamScratch *ws = nullptr;
    int rc = g_scratch.get(
        stream, need, [&] { return flash_decode_least_workspace_bytes(1, n_vis, kv_head_num); }, &ws);
    if (rc != LLMHIP_OK) return rc;
    if (ws->bytes < need) splits = flash_decode_splits_within(1, n_vis, kv_head_num, m * group_size, ws->bytes);
    return from_hip(launch_flash_decode(out, q, k, v, ws->ptr, ws->bytes, 1, m, n_vis, offset, n_vis,
                                        group_size, kv_head_num, splits, dt,
                                        as_stream(stream)));
  }
  const int n_vis = (n < m + offset) ? n : m + offset;
  if (flash_decode_takes_tiles(m, n_vis, group_size, kv_head_num)) {
    // some more of them over a short cache: the same in tiles of rows, if the scratch is there or can be had
    const int tiles = flash_decode_tiles(m, group_size);
    const int splits = flash_decode_default_splits(tiles, n_vis, kv_head_num, kMaxDecodeCols);
    const size_t need = flash_decode_workspace_bytes(tiles, m, group_size, kv_head_num, splits);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    StreamScratch *ws = nullptr;
    if (need) (void)g_scratch.get(stream, need, [] { return (size_t)0; }, &ws);
    if (!need || ws->bytes >= need)
      return from_hip(launch_flash_decode_tiles(out, q, k, v, need ? ws->ptr : nullptr, need ? ws->bytes : 0, m, n_vis, offset,
                                                group_size, kv_head_num, splits, dt, as_stream(stream)));
  }
  // a chunk of few rows over a long cache is split over the key range: fp32 partials in the
  // per-stream scratch
  const size_t need = flash_prefill_workspace_bytes(m, n, offset, group_size, kv_head_num);
  if (!need) {
    // a prompt: its longest rows shared by two workgroups, if the scratch is there or can be had.  Not on hipStreamPerThread,
    // where calls of several threads have one buffer and no order.
    const size_t halves = flash_prefill_halves_bytes(m, n, offset, group_size, kv_head_num);
    if (halves && as_stream(stream) != hipStreamPerThread && !may_be_capturing(as_stream(stream))) {
      std::lock_guard<std::mutex> lk(g_scratch_mu);
      StreamScratch *ws = nullptr;
      (void)g_exchange.get(stream, halves, [] { return (size_t)0; }, &ws);
      if (ws->bytes >= halves)
        return from_hip(launch_flash_prefill(out, q, k, v, m, n, offset, group_size, kv_head_num, dt, as_stream(stream), ws->ptr, ws->bytes));
    }
    return from_hip(launch_flash_prefill(out, q, k, v, m, n, offset, group_size, kv_head_num, dt,
                                         as_stream(stream), nullptr, 0));
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  StreamScratch *ws = nullptr;
  int rc = g_scratch.get(
      stream, need, [&] { return flash_prefill_least_workspace_bytes(m, n, offset, group_size, kv_head_num); }, &ws);
  if (rc != LLMHIP_OK) return rc;
  return from_hip(launch_flash_prefill(out, q, k, v, m, n, offset, group_size, kv_head_num, dt,
                                       as_stream(stream), ws->ptr, ws->bytes));
}

}  // namespace

extern "C" {

int llmhip_flash_attn(void *out, const void *q, const void *k, const void *v, int m, int n,
                      int offset, int head_num, int head_dim, int dt, void *stream) {
  return attn_common(out, q, k, v, m, n, offset, 1, head_num, head_dim, dt, stream);
}

int llmhip_flash_attn_gqa(void *out, const void *q, const void *k, const void *v, int m,
                          int n, int offset, int group_size, int kv_head_num, int head_dim,
                          int dt, void *stream) {
  return attn_common(out, q, k, v, m, n, offset, group_size, kv_head_num, head_dim, dt, stream);
}

int llmhip_flash_attn_opt_prefill(void *out, const void *q, const void *k, const void *v,
                                  int m, int n, int offset, int head_num, int head_dim,
                                  int dt, void *stream) {
  return attn_common(out, q, k, v, m, n, offset, 1, head_num, head_dim, dt, stream);
}

size_t llmhip_flash_attn_scratch_bytes(int m, int n, int offset, int group_size, int kv_head_num) {
  if (m < 1 || n < 1 || offset < 0 || group_size < 1 || kv_head_num < 1) return 0;
  if ((long long)m * group_size <= kMaxDecodeCols) {
    const int n_vis = (n < m + offset) ? n : m + offset;
    return flash_decode_workspace_bytes(1, m, group_size, kv_head_num,
                                        flash_decode_default_splits(1, n_vis, kv_head_num, m * group_size));
  }
  const int n_vis = (n < m + offset) ? n : m + offset;
  if (flash_decode_takes_tiles(m, n_vis, group_size, kv_head_num)) {
    const int tiles = flash_decode_tiles(m, group_size);
    return flash_decode_workspace_bytes(tiles, m, group_size, kv_head_num,
                                        flash_decode_default_splits(tiles, n_vis, kv_head_num, kMaxDecodeCols));
  }
  return flash_prefill_workspace_bytes(m, n, offset, group_size, kv_head_num);
}

int llmhip_flash_decode_default_splits(int batch, int n, int kv_head_num) {
  if (batch < 1 || n < 1 || kv_head_num < 1) return LLMHIP_ERR_INVALID_ARG;
  return flash_decode_default_splits(batch, n, kv_head_num, 1);
}

size_t llmhip_flash_decode_workspace_bytes(int batch, int group_size, int kv_head_num,
                                           int head_dim, int num_splits) {
  if (batch < 1 || group_size < 1 || kv_head_num < 1 || head_dim != 128) return 0;
  if (num_splits <= 0) {
    // the largest count the default rule picks for any KV length
    num_splits = flash_decode_max_default_splits((long long)batch * kv_head_num);
  }
  if (num_splits > kMaxDecodeSplits) num_splits = kMaxDecodeSplits;
  return flash_decode_workspace_bytes(batch, 1, group_size, kv_head_num, num_splits);
}

int llmhip_flash_decode_gqa(void *out, const void *q, const void *k_cache,
                            const void *v_cache, void *workspace, size_t workspace_bytes,
                            int batch, int n, int64_t kv_seq_stride, int group_size,
                            int kv_head_num, int head_dim, int num_splits, int dt,
                            void *stream) {
  if (!out || !q || !k_cache || !v_cache || !all_aligned16(out, q, k_cache, v_cache, workspace))
    return LLMHIP_ERR_INVALID_ARG;
  if (batch < 1 || n < 1 || group_size < 1 || kv_head_num < 1 || kv_seq_stride < n)
    return LLMHIP_ERR_INVALID_ARG;
  if (!dtype_ok(dt)) return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128 || group_size > kMaxDecodeCols) return LLMHIP_ERR_UNSUPPORTED;
  if (batch > 65535 || kv_head_num > 65535) return LLMHIP_ERR_UNSUPPORTED;
  const size_t room = workspace ? workspace_bytes : 0;
  if (num_splits <= 0) {
    // the default count, or the best one the workspace holds, unless that is less than a call may insist on
    num_splits = flash_decode_default_splits(batch, n, kv_head_num, group_size);
    if (flash_decode_workspace_bytes(batch, 1, group_size, kv_head_num, num_splits) > room &&
        flash_decode_least_workspace_bytes(batch, n, kv_head_num) <= room)
      num_splits = flash_decode_splits_within(batch, n, kv_head_num, group_size, room);
  }
  if (num_splits > kMaxDecodeSplits) num_splits = kMaxDecodeSplits;  // the combine kernel's limit
  const size_t need = flash_decode_workspace_bytes(batch, 1, group_size, kv_head_num, num_splits);
  if (need > room) return LLMHIP_ERR_WORKSPACE;
  return from_hip(launch_flash_decode(out, q, k_cache, v_cache, workspace, room, batch, 1, n, n - 1,
                                      kv_seq_stride, group_size, kv_head_num, num_splits, dt,
                                      as_stream(stream)));
}

int llmhip_flash_decode_gqa_static(void *out, const void *q, const void *k_cache, const void *v_cache,
                                   int batch, int n, int64_t kv_seq_stride, int group_size,
                                   int kv_head_num, int head_dim, int num_splits, int dt, void *stream) {
  if (!out || !q || !k_cache || !v_cache || !all_aligned16(out, q, k_cache, v_cache))
    return LLMHIP_ERR_INVALID_ARG;
  if (batch < 1 || n < 1 || group_size < 1 || kv_head_num < 1 || kv_seq_stride < n)
    return LLMHIP_ERR_INVALID_ARG;
  if (!dtype_ok(dt)) return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128 || group_size > kMaxDecodeCols) return LLMHIP_ERR_UNSUPPORTED;
  if (batch > 65535 || kv_head_num > 65535) return LLMHIP_ERR_UNSUPPORTED;
  if (num_splits <= 0) {
    // the default count, lowered until its partials fit the fixed array (one split needs none)
    num_splits = flash_decode_default_splits(batch, n, kv_head_num, group_size);
    while (num_splits > 1 &&
           flash_decode_workspace_bytes(batch, 1, group_size, kv_head_num, num_splits) > kStaticDecodeScratchBytes)
      --num_splits;
  }
  if (num_splits > kMaxDecodeSplits) num_splits = kMaxDecodeSplits;
  // the launch uses at most one split per 128 keys: a larger count is judged by what it becomes
  num_splits = flash_decode_effective_splits(num_splits, n);
  // the fixed array must hold the partials of every (sequence, kv head, split)
  if (flash_decode_workspace_bytes(batch, 1, group_size, kv_head_num, num_splits) > kStaticDecodeScratchBytes)
    return LLMHIP_ERR_WORKSPACE;
  return from_hip(launch_flash_decode_static(out, q, k_cache, v_cache, batch, n, kv_seq_stride, group_size,
                                             kv_head_num, num_splits, dt, as_stream(stream)));
}

size_t llmhip_flash_decode_static_scratch_bytes(void) { return kStaticDecodeScratchBytes; }

int llmhip_decode_step_gqa(void *out, void *k_cache, void *v_cache, const void *freq_cis, const void *in_q,
                           const void *in_k, const void *in_v, int pos, int group_size, int kv_head_num,
                           int head_dim, int is_neox_style, int dt, void *stream) {
  if (!out || !k_cache || !v_cache || !freq_cis || !in_q || !in_k || !in_v ||
      !all_aligned16(out, k_cache, v_cache, freq_cis, in_q, in_k, in_v))
    return LLMHIP_ERR_INVALID_ARG;
  if (pos < 0 || pos == INT32_MAX || group_size < 1 || kv_head_num < 1 || !dtype_ok(dt)) return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128 || group_size > kMaxDecodeCols) return LLMHIP_ERR_UNSUPPORTED;
  if (kv_head_num > 65535) return LLMHIP_ERR_UNSUPPORTED;
  const int n = pos + 1;
  int splits = flash_decode_default_splits(1, n, kv_head_num, group_size);
  const size_t need = flash_decode_workspace_bytes(1, 1, group_size, kv_head_num, splits);
  if (!need)
    return from_hip(launch_flash_decode_step(out, k_cache, v_cache, freq_cis, in_q, in_k, in_v, nullptr, 0, pos,
                                             group_size, kv_head_num, is_neox_style, splits, dt,
                                             as_stream(stream)));
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  StreamScratch *ws = nullptr;
  int rc = g_scratch.get(
      stream, need, [&] { return flash_decode_least_workspace_bytes(1, n, kv_head_num); }, &ws);
  if (rc != LLMHIP_OK) return rc;
  if (ws->bytes < need) splits = flash_decode_splits_within(1, n, kv_head_num, group_size, ws->bytes);
  return from_hip(launch_flash_decode_step(out, k_cache, v_cache, freq_cis, in_q, in_k, in_v, ws->ptr, ws->bytes, pos, group_size,
                                           kv_head_num, is_neox_style, splits, dt, as_stream(stream)));
}

int llmhip_rope(void *out_q, void *out_k, const void *freq_cis, const void *in_q,
                const void *in_k, int start_pos, int cur_size, int n_heads, int hidden_dim,
                int is_neox_style, int dt, void *stream) {
  if (!out_q || !out_k || !freq_cis || !in_q || !in_k || !all_aligned16(out_q, out_k, freq_cis, in_q, in_k))
    return LLMHIP_ERR_INVALID_ARG;
  if (start_pos < 0 || cur_size < 1 || n_heads < 1 || !dtype_ok(dt))
    return LLMHIP_ERR_INVALID_ARG;
  if (hidden_dim != n_heads * 128) return LLMHIP_ERR_UNSUPPORTED;
  return from_hip(launch_rope_kv_append(out_q, out_k, nullptr, freq_cis, in_q, in_k, nullptr,
                                        start_pos, cur_size, n_heads, n_heads, 0,
                                        is_neox_style, dt, as_stream(stream)));
}

int llmhip_rope_single(void *out, const void *freq_cis, const void *in, int start_pos,
                       int cur_size, int n_heads, int hidden_dim, int is_neox_style, int dt,
                       void *stream) {
  if (!out || !freq_cis || !in || !all_aligned16(out, freq_cis, in)) return LLMHIP_ERR_INVALID_ARG;
  if (start_pos < 0 || cur_size < 1 || n_heads < 1 || !dtype_ok(dt))
    return LLMHIP_ERR_INVALID_ARG;
  if (hidden_dim != n_heads * 128) return LLMHIP_ERR_UNSUPPORTED;
  return from_hip(launch_rope_kv_append(out, nullptr, nullptr, freq_cis, in, nullptr, nullptr,
                                        start_pos, cur_size, n_heads, 0, 0, is_neox_style, dt,
                                        as_stream(stream)));
}

int llmhip_rope_kv_append(void *out_q, void *k_cache, void *v_cache, const void *freq_cis,
                          const void *in_q, const void *in_k, const void *in_v,
                          int start_pos, int cur_size, int n_heads, int n_kv_heads,
                          int head_dim, int is_neox_style, int dt, void *stream) {
  if (!out_q || !k_cache || !v_cache || !freq_cis || !in_q || !in_k || !in_v ||
      !all_aligned16(out_q, k_cache, v_cache, freq_cis, in_q, in_k, in_v))
    return LLMHIP_ERR_INVALID_ARG;
  if (start_pos < 0 || cur_size < 1 || n_heads < 1 || n_kv_heads < 1 || !dtype_ok(dt))
    return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128) return LLMHIP_ERR_UNSUPPORTED;
  return from_hip(launch_rope_kv_append(out_q, k_cache, v_cache, freq_cis, in_q, in_k, in_v,
                                        start_pos, cur_size, n_heads, n_kv_heads, start_pos,
                                        is_neox_style, dt, as_stream(stream)));
}

/* ---------------- runtime surface ---------------- */

int llmhip_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}
int llmhip_device_props(int device, int *compute_units, int *max_clock_khz, size_t *total_mem_bytes) {
  if (llmhip_device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  hipDeviceProp_t prop;
  hipError_t e = hipGetDeviceProperties(&prop, device);
  if (e != hipSuccess) return (int)e;
  if (compute_units) *compute_units = prop.multiProcessorCount;
  if (max_clock_khz) *max_clock_khz = prop.clockRate;
  if (total_mem_bytes) *total_mem_bytes = prop.totalGlobalMem;
  return LLMHIP_OK;
}
int llmhip_set_device(int device) {
  if (llmhip_device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(hipSetDevice(device));
}
int llmhip_malloc(void **ptr, size_t bytes) {
  if (!ptr) return LLMHIP_ERR_INVALID_ARG;
  if (llmhip_device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(hipMalloc(ptr, bytes));
}
int llmhip_free(void *ptr) { return from_hip(hipFree(ptr)); }
int llmhip_memcpy_h2d(void *dst, const void *src, size_t bytes) {
  if (!dst || !src) return LLMHIP_ERR_INVALID_ARG;
  return from_hip(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
}
int llmhip_memcpy_d2h(void *dst, const void *src, size_t bytes) {
  if (!dst || !src) return LLMHIP_ERR_INVALID_ARG;
  return from_hip(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
}
int llmhip_memcpy_d2d_async(void *dst, const void *src, size_t bytes, void *stream) {
  if (!dst || !src) return LLMHIP_ERR_INVALID_ARG;
  return from_hip(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
}
int llmhip_memset_async(void *dst, int value, size_t bytes, void *stream) {
  if (!dst) return LLMHIP_ERR_INVALID_ARG;
  // a fill kernel, not hipMemsetAsync: the call may be captured into a HIP graph
  return from_hip(launch_fill(dst, value, bytes, as_stream(stream)));
}
int llmhip_stream_create(void **stream) {
  if (!stream) return LLMHIP_ERR_INVALID_ARG;
  if (llmhip_device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  hipStream_t s;
  hipError_t e = hipStreamCreate(&s);  // default priority
  if (e != hipSuccess) return (int)e;
  *stream = s;
  return LLMHIP_OK;
}
int llmhip_stream_destroy(void *stream) {
  {
    // the scratch kept for this stream goes with it
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    g_scratch.drop(stream);
    g_exchange.drop(stream);
  }
  return from_hip(hipStreamDestroy(as_stream(stream)));
}
int llmhip_stream_sync(void *stream) { return from_hip(hipStreamSynchronize(as_stream(stream))); }
int llmhip_device_sync(void) { return from_hip(hipDeviceSynchronize()); }
int llmhip_event_create(void **event) {
  if (!event) return LLMHIP_ERR_INVALID_ARG;
  if (llmhip_device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  hipEvent_t ev;
  hipError_t e = hipEventCreate(&ev);
  if (e != hipSuccess) return (int)e;
  *event = ev;
  return LLMHIP_OK;
}
int llmhip_event_destroy(void *event) {
  return from_hip(hipEventDestroy(static_cast<hipEvent_t>(event)));
}
int llmhip_event_record(void *event, void *stream) {
  return from_hip(hipEventRecord(static_cast<hipEvent_t>(event), as_stream(stream)));
}
int llmhip_event_sync(void *event) {
  return from_hip(hipEventSynchronize(static_cast<hipEvent_t>(event)));
}
int llmhip_event_query(void *event) {
  const hipError_t e = hipEventQuery(static_cast<hipEvent_t>(event));
  if (e == hipErrorNotReady) {
    (void)hipGetLastError();  // not an error: leave nothing behind for the next call to report
    return LLMHIP_NOT_READY;
  }
  return from_hip(e);
}
int llmhip_event_elapsed_ms(float *ms, void *start, void *stop) {
  if (!ms) return LLMHIP_ERR_INVALID_ARG;
  return from_hip(
      hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
}
const char *llmhip_error_string(int status) {
  switch (status) {
    case LLMHIP_OK: return "ok";
    case LLMHIP_ERR_INVALID_ARG: return "invalid argument";
    case LLMHIP_ERR_UNSUPPORTED: return "unsupported shape (head_dim must be 128)";
    case LLMHIP_ERR_WORKSPACE:
      return "workspace missing or too small (or batch * kv heads * splits beyond the fixed scratch of the "
             "allocation-free decode)";
    case LLMHIP_ERR_NO_DEVICE: return "no HIP device";
    case LLMHIP_NOT_READY: return "event not complete yet";
    default: break;
  }
  if (status > 0) return hipGetErrorString(static_cast<hipError_t>(status));
  return "unknown status";
}
int llmhip_release_internal_workspace(void) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  const int kept = g_scratch.release(), passed = g_exchange.release(), rc = kept ? kept : passed;
  release_matmul_resources();
  return rc;
}

static int matmul_common(void *out, const void *lhs, const void *weight, const void *bias, int m,
                         int n, int k, int dt, void *stream) {
  if (!out || !lhs || !weight) return LLMHIP_ERR_INVALID_ARG;
  if (m < 1 || n < 1 || k < 1 || !dtype_ok(dt)) return LLMHIP_ERR_INVALID_ARG;
  if (n % 16 != 0 || k % 16 != 0) return LLMHIP_ERR_UNSUPPORTED;
  // Up to 16 rows one MFMA column block holds every lhs row and the call is a read of W; beyond that lhs, which
  // every workgroup of that kernel reads whole, outweighs W, and tiles are shared.  From 9 rows on that is so already where W has
  // more than one round of its workgroups takes, 16 rows per CU, or where rows times W rows per CU, its work beside the stream,
  // pass a bound, lower over a long k (W from HBM, us, few-row kernel / tiles: 4352 x 5120, 9 rows 15.3 / 12.3; 5120 x 3584 11.6 /
  // 9.6; 4096 x 4096, 12 rows 10.5 / 9.6; 3584 x 3584, 9 rows 8.2 / 9.0, 16 rows 9.5 / 9.6; 2560 x 3584 7.0 / 8.4, 8.5 / 9.1; long:
  // 4096 x 11008, 9 rows 28.4 / 22.5, 3584 x 18944, 12 rows 39.1 / 38.0, 2560 x 8192, 9 rows 13.4 / 15.5).  Over 322 sizes of
  // 512-11008 W rows, k of 1536-18944 and 9-16 rows the kernel chosen is 0.4 % slower than the better one on average, 16 % at most (3072
  // x 11008, 9 rows); by a line at 16 rows per CU alone 1.8 %, at 8 2.7 %.  With 8 rows neither is ahead by much: 4352 x 5120 13.1
  // / 12.4, 11008 x 18944 75.4 / 79.4.  (With W in the last-level cache the tiles are ahead earlier, 3584 x 3584, 9 rows 7.3 / 6.8,
  // but the weights of a model's other layers lie between two calls.)  Both kernels move 16-byte pieces; hipBLASLt takes any
  // base.
  if (all_aligned16(out, lhs, weight)) {
    const float *b = static_cast<const float *>(bias);
    // Few tiles over a long k in pieces, if the scratch is there or can be had (not on hipStreamPerThread, see attn_common)
    const int pieces = matmul_tile_pieces(m, n, k);
    if (pieces > 1 && as_stream(stream) != hipStreamPerThread && !may_be_capturing(as_stream(stream))) {
      const size_t need = matmul_pieces_bytes(m, n, pieces);
      std::lock_guard<std::mutex> lk(g_scratch_mu);
      StreamScratch *ws = nullptr;
      (void)g_exchange.get(stream, need, [] { return (size_t)0; }, &ws);
      if (ws->bytes >= need) return from_hip(launch_matmul_tile(out, lhs, weight, b, m, n, k, dt, as_stream(stream), pieces, ws->ptr));
    }
    const bool tiles = m > 8 && matmul_tile_takes(m, n, k);
    const long long per_cu = (n + device_compute_units() - 1) / device_compute_units();
    if (m <= 16 && !(tiles && (per_cu > 16 || m * per_cu > (k > 7168 ? 130 : 190))))
      return from_hip(launch_matmul_skinny(out, lhs, weight, b, m, n, k, dt, as_stream(stream)));
    if (tiles)
      return from_hip(launch_matmul_tile(out, lhs, weight, b, m, n, k, dt, as_stream(stream)));
  }
  return from_hip(launch_matmul_bias(out, lhs, weight, static_cast<const float *>(bias), m, n, k, dt,
                                     as_stream(stream)));
}
int llmhip_matmul(void *out, const void *lhs, const void *weight, int m, int n, int k, int dt,
                  void *stream) {
  return matmul_common(out, lhs, weight, nullptr, m, n, k, dt, stream);
}
int llmhip_matmul_bias(void *out, const void *lhs, const void *weight, const void *bias_f32, int m,
                       int n, int k, int dt, void *stream) {
  if (!bias_f32) return LLMHIP_ERR_INVALID_ARG;
  return matmul_common(out, lhs, weight, bias_f32, m, n, k, dt, stream);
}
int llmhip_add(void *out, const void *lhs, const void *rhs, long long total_size, int dt,
               void *stream) {
  if (!out || !lhs || !rhs || total_size < 0 || !dtype_ok(dt) || !all_aligned16(out, lhs, rhs))
    return LLMHIP_ERR_INVALID_ARG;
  return from_hip(launch_add(out, lhs, rhs, (size_t)total_size, dt, as_stream(stream)));
}

}  // extern "C"
