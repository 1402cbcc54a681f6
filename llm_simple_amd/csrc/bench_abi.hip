// C ABI of libllmhip_bench.so (declared in include/llmhip_bench.h): the measurement aids of the
// benchmark.  Built with LLMHIP_BENCH defined, so the prefill kernel linked here is the library's own
// copy with the clock stamp; the product library libllmhip.so holds none of this.
#include "../../include/llmhip_bench.h"

#include <hip/hip_runtime.h>

#include "bench_kernels.hpp"
#include "kernels.hpp"

using namespace LLMHIP_NS;

namespace {
inline int from_hip(hipError_t e) { return e == hipSuccess ? LLMHIP_OK : (int)e; }
inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline int device_count() {
  int n = 0;
  return hipGetDeviceCount(&n) == hipSuccess ? n : 0;
}
}  // namespace

extern "C" {

int llmhip_bench_flash_attn_gqa_clocked(void *out, const void *q, const void *k, const void *v, int m, int n,
                                        int offset, int group_size, int kv_head_num, int head_dim, int dt,
                                        void *clock_probe, void *stream) {
  if (!out || !q || !k || !v || !clock_probe || !aligned16(out) || !aligned16(q) || !aligned16(k) ||
      !aligned16(v) || (reinterpret_cast<uintptr_t>(clock_probe) & 7u))
    return LLMHIP_ERR_INVALID_ARG;
  if (m < 1 || n < 1 || offset < 0 || group_size < 1 || kv_head_num < 1 ||
      (dt != LLMHIP_DT_FLOAT16 && dt != LLMHIP_DT_BFLOAT16))
    return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128) return LLMHIP_ERR_UNSUPPORTED;
  if (kv_head_num > 65535 || (long long)group_size * kv_head_num > 65535) return LLMHIP_ERR_UNSUPPORTED;
  if ((long long)m * group_size <= 16) return LLMHIP_ERR_UNSUPPORTED;  // prefill kernel only
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(launch_flash_prefill(out, q, k, v, m, n, offset, group_size, kv_head_num, dt,
                                       static_cast<hipStream_t>(stream), nullptr, 0, clock_probe));
}

int llmhip_bench_flash_attn_gqa_alone(void *out, const void *q, const void *k, const void *v, void *workspace, size_t workspace_bytes,
                                      int m, int n, int offset, int group_size, int kv_head_num, int head_dim, int dt, void *stream) {
  if (!out || !q || !k || !v || !workspace || !aligned16(out) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(workspace))
    return LLMHIP_ERR_INVALID_ARG;
  if (m < 1 || n < 1 || offset < 0 || group_size < 1 || kv_head_num < 1 ||
      (dt != LLMHIP_DT_FLOAT16 && dt != LLMHIP_DT_BFLOAT16))
    return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128 || kv_head_num > 65535 || (long long)group_size * kv_head_num > 65535 || (long long)m * group_size <= 16)
    return LLMHIP_ERR_UNSUPPORTED;
  const size_t need = flash_prefill_halves_bytes(m, n, offset, group_size, kv_head_num);
  if (!need) return LLMHIP_ERR_UNSUPPORTED;
  if (need > workspace_bytes) return LLMHIP_ERR_WORKSPACE;
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(launch_flash_prefill(out, q, k, v, m, n, offset, group_size, kv_head_num, dt, static_cast<hipStream_t>(stream),
                                       workspace, workspace_bytes, nullptr));
}

int llmhip_bench_flash_decode_gqa_alone(void *out, const void *q, const void *k_cache, const void *v_cache, void *workspace,
                                        size_t workspace_bytes, int batch, int n, int64_t kv_seq_stride, int group_size,
                                        int kv_head_num, int head_dim, int num_splits, int dt, void *stream) {
  if (!out || !q || !k_cache || !v_cache || !workspace || !aligned16(out) || !aligned16(q) || !aligned16(k_cache) ||
      !aligned16(v_cache) || !aligned16(workspace))
    return LLMHIP_ERR_INVALID_ARG;
  if (batch < 1 || n < 1 || group_size < 1 || kv_head_num < 1 || kv_seq_stride < n || num_splits < 1 ||
      (dt != LLMHIP_DT_FLOAT16 && dt != LLMHIP_DT_BFLOAT16))
    return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128 || group_size > 16 || batch > 65535 || kv_head_num > 65535 || num_splits > 256) return LLMHIP_ERR_UNSUPPORTED;
  if (flash_decode_workspace_bytes(batch, 1, group_size, kv_head_num, num_splits) > workspace_bytes) return LLMHIP_ERR_WORKSPACE;
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(launch_flash_decode(out, q, k_cache, v_cache, workspace, workspace_bytes, batch, 1, n, n - 1, kv_seq_stride,
                                      group_size, kv_head_num, num_splits, dt, static_cast<hipStream_t>(stream)));
}

int llmhip_bench_decode_step_gqa_alone(void *out, void *k_cache, void *v_cache, const void *freq_cis, const void *in_q,
                                       const void *in_k, const void *in_v, void *workspace, size_t workspace_bytes, int pos,
                                       int group_size, int kv_head_num, int head_dim, int is_neox_style, int num_splits, int dt,
                                       void *stream) {
  if (!out || !k_cache || !v_cache || !freq_cis || !in_q || !in_k || !in_v || !workspace || !aligned16(out) || !aligned16(k_cache) ||
      !aligned16(v_cache) || !aligned16(freq_cis) || !aligned16(in_q) || !aligned16(in_k) || !aligned16(in_v) || !aligned16(workspace))
    return LLMHIP_ERR_INVALID_ARG;
  if (pos < 0 || pos == INT32_MAX || group_size < 1 || kv_head_num < 1 || num_splits < 1 ||
      (dt != LLMHIP_DT_FLOAT16 && dt != LLMHIP_DT_BFLOAT16))
    return LLMHIP_ERR_INVALID_ARG;
  if (head_dim != 128 || group_size > 16 || kv_head_num > 65535 || num_splits > 256) return LLMHIP_ERR_UNSUPPORTED;
  if (flash_decode_workspace_bytes(1, 1, group_size, kv_head_num, num_splits) > workspace_bytes) return LLMHIP_ERR_WORKSPACE;
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(launch_flash_decode_step(out, k_cache, v_cache, freq_cis, in_q, in_k, in_v, workspace, workspace_bytes, pos,
                                           group_size, kv_head_num, is_neox_style, num_splits, dt,
                                           static_cast<hipStream_t>(stream)));
}

int llmhip_bench_matmul_alone(void *out, const void *lhs, const void *weight, const void *bias_f32, void *workspace, size_t workspace_bytes,
                              int m, int n, int k, int dt, void *stream) {
  if (!out || !lhs || !weight || !workspace || !aligned16(out) || !aligned16(lhs) || !aligned16(weight) || !aligned16(workspace))
    return LLMHIP_ERR_INVALID_ARG;
  if (m < 1 || n < 1 || k < 1 || (dt != LLMHIP_DT_FLOAT16 && dt != LLMHIP_DT_BFLOAT16)) return LLMHIP_ERR_INVALID_ARG;
  if (n % 16 != 0 || k % 16 != 0) return LLMHIP_ERR_UNSUPPORTED;
  const int pieces = matmul_tile_pieces(m, n, k);
  if (pieces < 2) return LLMHIP_ERR_UNSUPPORTED;
  if (matmul_pieces_bytes(m, n, pieces) > workspace_bytes) return LLMHIP_ERR_WORKSPACE;
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(launch_matmul_tile(out, lhs, weight, static_cast<const float *>(bias_f32), m, n, k, dt, static_cast<hipStream_t>(stream),
                                     pieces, workspace));
}

int llmhip_bench_matmul_tile(int m, int n, int k) { return m < 1 || n < 1 || k < 1 ? LLMHIP_ERR_INVALID_ARG : matmul_tile_size(m, n, k); }

int llmhip_bench_mfma_ceiling(int mix, double target_ms, double *tflops) {
  if (!tflops || (mix != 0 && mix != 1) || target_ms < 0.0 || target_ms > 2000.0) return LLMHIP_ERR_INVALID_ARG;
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(run_mfma_ceiling(mix, target_ms, tflops));
}

int llmhip_bench_stream_read(const void *src_a, const void *src_b, size_t bytes_each, void *sink, size_t sink_bytes,
                             int variant, void *stream) {
  if (!src_a || !src_b || !sink || bytes_each == 0 || bytes_each % 16 != 0 || (variant != 0 && variant != 1))
    return LLMHIP_ERR_INVALID_ARG;
  if (sink_bytes < kStreamReadSinkBytes) return LLMHIP_ERR_WORKSPACE;
  if (!aligned16(src_a) || !aligned16(src_b) || !aligned16(sink)) return LLMHIP_ERR_INVALID_ARG;
  if (device_count() < 1) return LLMHIP_ERR_NO_DEVICE;
  return from_hip(launch_stream_read(src_a, src_b, bytes_each, sink, variant, static_cast<hipStream_t>(stream)));
}

}  // extern "C"
