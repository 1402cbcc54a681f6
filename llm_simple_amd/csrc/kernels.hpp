// Launchers of the gfx950 kernels; called only by the C ABI in llmhip.hip after
// it has validated every argument.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "common.hpp"
#include "launch.hpp"

namespace LLMHIP_NS {

// workspace, workspace_bytes: device memory for the fp32 partials of a key-range split; the call takes the fastest
// plan that fits (null: unsplit).  flash_prefill_workspace_bytes: what the fastest plan of all takes (0: none needed);
// flash_prefill_least_workspace_bytes: below this a call with no way to get more is to be refused.
size_t flash_prefill_workspace_bytes(int m, int n, int offset, int group_size, int kv_head_num);
size_t flash_prefill_least_workspace_bytes(int m, int n, int offset, int group_size, int kv_head_num);
// What a prompt whose longest rows two workgroups share takes for the halves that are passed on (0: none do).  Without it they are not
// shared; nor are they on a stream that may be capturing.
size_t flash_prefill_halves_bytes(int m, int n, int offset, int group_size, int kv_head_num);
#ifdef LLMHIP_BENCH
// The measurement library's copy: clock_probe is null or a device pointer to two 64-bit counters that
// workgroup 0 fills with the shader-clock ticks and the reference-clock ticks of its lifetime; where rows are shared,
// who began second of a pair does not wait for the other one's half.
hipError_t launch_flash_prefill(void *out, const void *q, const void *k, const void *v, int m,
                                int n, int offset, int group_size, int kv_head_num, int dt,
                                hipStream_t stream, void *workspace, size_t workspace_bytes, void *clock_probe);
#else
hipError_t launch_flash_prefill(void *out, const void *q, const void *k, const void *v, int m,
                                int n, int offset, int group_size, int kv_head_num, int dt,
                                hipStream_t stream, void *workspace, size_t workspace_bytes);
#endif

// What the launch of a prompt does and the rope launch before it counts on.  A call is a prompt if no more tokens are cached than
// new.  Workgroup b runs on XCD b % 8; the query heads of a kv head are dealt to one XCD (of several kv heads each), or to 2^share_log2 of
// them, as long as kv heads and XCDs divide; else (share_log2 < 0) workgroups are not dealt at all.
inline bool prefill_is_prompt(long long new_tokens, long long visible_keys) { return visible_keys < 2 * new_tokens; }
inline int prefill_xcd_share_log2(int kv_head_num) {
  if (kv_head_num % 8 == 0) return 0;
  return kv_head_num == 4 ? 1 : kv_head_num == 2 ? 2 : kv_head_num == 1 ? 3 : -1;
}

// A number that no workspace holds: of a launch, see launch_number.hpp.  (A replayed graph launches with the number of its
// capture, and words of the replay before would pass for new ones: not for a stream that may be capturing.)
uint64_t launch_number();
bool may_be_capturing(hipStream_t stream);

// Compute units of the current device, cached per device; 256 when no device can be asked.
int device_compute_units();

// Split-KV decode.  rows = m * group_size <= 16 query rows per kv head.
size_t flash_decode_workspace_bytes(int batch, int m, int group_size, int kv_head_num,
                                    int num_splits);
// rows: query rows of a kv head
int flash_decode_default_splits(int batch, int n, int kv_head_num, int rows);
int flash_decode_max_default_splits(long long pairs);
// The best count whose partials fit `bytes`; the size below which a call that leaves the count to the
// library and has no way to get more is to be refused.
int flash_decode_splits_within(int batch, int n, int kv_head_num, int rows, size_t bytes);
size_t flash_decode_least_workspace_bytes(int batch, int n, int kv_head_num);
// The split count a launch really uses for n keys: at most one split per block of 128 keys.
int flash_decode_effective_splits(int num_splits, int n);
hipError_t launch_flash_decode(void *out, const void *q, const void *k, const void *v,
                               void *workspace, size_t workspace_bytes, int batch, int m, int n, int offset,
                               int64_t kv_seq_stride, int group_size, int kv_head_num,
                               int num_splits, int dt, hipStream_t stream);

// m tokens of one sequence with more query rows than 16: as tiles of up to 16 rows, each with workgroups of its own, over
// visible keys n.  Partials as of flash_decode_tiles(m, group_size) sequences.
int flash_decode_tiles(int m, int group_size);
bool flash_decode_takes_tiles(int m, int n_vis, int group_size, int kv_head_num);
hipError_t launch_flash_decode_tiles(void *out, const void *q, const void *k, const void *v, void *workspace, size_t workspace_bytes,
                                     int m, int n, int offset, int group_size, int kv_head_num, int num_splits, int dt,
                                     hipStream_t stream);

// One decode step of one sequence, rotary embedding and cache append fused into the decode kernel:
// q and the new K row are rotated with row `pos` of the table as they are loaded, the workgroups that own
// the last key range write row pos of both caches, attention runs over rows [0, pos].
hipError_t launch_flash_decode_step(void *out, void *k_cache, void *v_cache, const void *freq_cis,
                                    const void *in_q, const void *in_k, const void *in_v, void *workspace,
                                    size_t workspace_bytes, int pos, int group_size, int kv_head_num, int is_neox, int num_splits,
                                    int dt, hipStream_t stream);

// Same decode with the split-KV partials in a fixed device array of kStaticDecodeScratchBytes inside
// the library: no allocation, no workspace argument.  The caller checks the size beforehand.
constexpr size_t kStaticDecodeScratchBytes = 4u << 20;
hipError_t launch_flash_decode_static(void *out, const void *q, const void *k, const void *v,
                                      int batch, int n, int64_t kv_seq_stride, int group_size,
                                      int kv_head_num, int num_splits, int dt, hipStream_t stream);

// q_heads may be 0 (rotate K only) and cache pointers may be null (no append):
// covers rope, rope_single and the fused rope + KV append.
hipError_t launch_rope_kv_append(void *out_q, void *out_k, void *out_v, const void *freq_cis,
                                 const void *in_q, const void *in_k, const void *in_v,
                                 int start_pos, int cur_size, int q_heads, int k_heads,
                                 int k_out_row_offset, int is_neox, int dt, hipStream_t stream);

// Projection out[m][n] = round(lhs[m][k] . weight[n][k]^T + bias), bias fp32 [n] or null; n and k multiples
// of 16.  matmul_skinny: m <= 16, pointers 16-byte aligned.  matmul_tile: the sizes that matmul_tile_takes
// accepts, pointers 16-byte aligned; with more than one of matmul_tile_pieces' pieces of k a workspace of matmul_pieces_bytes, and not on a
// stream that may be capturing.  matmul_bias: hipBLASLt, whose handle and 64 MiB
// workspace the first call creates.
hipError_t launch_matmul_skinny(void *out, const void *lhs, const void *weight, const float *bias,
                                int m, int n, int k, int dt, hipStream_t stream);
bool matmul_tile_takes(int m, int n, int k);
int matmul_tile_size(int m, int n, int k);  // lhs rows << 16 | features; 0: not taken
int matmul_tile_pieces(int m, int n, int k);
size_t matmul_pieces_bytes(int m, int n, int pieces);
hipError_t launch_matmul_tile(void *out, const void *lhs, const void *weight, const float *bias,
                              int m, int n, int k, int dt, hipStream_t stream, int pieces = 1, void *workspace = nullptr);
hipError_t launch_matmul_bias(void *out, const void *lhs, const void *weight, const float *bias,
                              int m, int n, int k, int dt, hipStream_t stream);
void release_matmul_resources();
hipError_t launch_add(void *out, const void *lhs, const void *rhs, size_t total, int dt,
                      hipStream_t stream);
// dst[0 .. bytes) = (unsigned char)value with a kernel (safe to capture into a HIP graph).
hipError_t launch_fill(void *dst, int value, size_t bytes, hipStream_t stream);

}  // namespace LLMHIP_NS
