/*
 * llmhip_bench.h -- C ABI of libllmhip_bench.so: measurement aids of the benchmark.
 *
 * None of these has a counterpart in the reference and none is part of the product library
 * (libllmhip.so, include/llmhip.h): they exist so that the benchmark can print, next to each
 * kernel's figure, what the machine it ran on delivers -- the shader clock under the prefill
 * kernel's load, the rate the matrix pipe sustains, the rate of a kernel that only reads.  Status
 * codes and the dtype numbering are those of llmhip.h.
 */
#ifndef LLMHIP_BENCH_H_
#define LLMHIP_BENCH_H_

#include "llmhip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* llmhip_flash_attn_gqa (llmhip.h) on this library's own copy of the prefill kernel
 * (m * group_size > 16, LLMHIP_ERR_UNSUPPORTED otherwise; square and ragged prefill shapes, no
 * key-range split), which also makes the first scheduled workgroup store two 64-bit counters at
 * clock_probe (device memory, 16 bytes): the shader-clock ticks and the ticks of the constant
 * 100 MHz reference clock between its start and its end.  Their ratio x 100 MHz is the shader
 * clock under this kernel's load. */
int llmhip_bench_flash_attn_gqa_clocked(void *out, const void *q, const void *k, const void *v, int m,
                                        int n, int offset, int group_size, int kv_head_num, int head_dim,
                                        int dt, void *clock_probe, void *stream);

/* llmhip_flash_attn_gqa of a prompt whose longest rows two workgroups share, on this library's own copy of the kernel, in which the second one of a
 * pair to begin does not wait for the first one's half of the keys but goes over both by itself, as the product's does when it has looked for it in
 * vain for some 0.1 s: the results are those of whole rows.  LLMHIP_ERR_UNSUPPORTED for other sizes; LLMHIP_ERR_WORKSPACE if workspace is too small (16 MiB
 * are enough for any on 256 compute units).  On a capturing stream no rows are shared. */
int llmhip_bench_flash_attn_gqa_alone(void *out, const void *q, const void *k, const void *v, void *workspace, size_t workspace_bytes,
                                      int m, int n, int offset, int group_size, int kv_head_num, int head_dim, int dt, void *stream);

/* llmhip_flash_decode_gqa and llmhip_decode_step_gqa (llmhip.h) on this library's own copy of the decode kernel, in which the
 * workgroups that fold partials do not wait for them: each computes its rows from the caches by itself, as the product's do
 * when they have looked for partials in vain for some 50 ms.  num_splits >= 1 and a workspace of
 * llmhip_flash_decode_workspace_bytes in both. */
int llmhip_bench_flash_decode_gqa_alone(void *out, const void *q, const void *k_cache, const void *v_cache, void *workspace,
                                        size_t workspace_bytes, int batch, int n, int64_t kv_seq_stride, int group_size,
                                        int kv_head_num, int head_dim, int num_splits, int dt, void *stream);
int llmhip_bench_decode_step_gqa_alone(void *out, void *k_cache, void *v_cache, const void *freq_cis, const void *in_q,
                                       const void *in_k, const void *in_v, void *workspace, size_t workspace_bytes, int pos,
                                       int group_size, int kv_head_num, int head_dim, int is_neox_style, int num_splits, int dt,
                                       void *stream);

/* llmhip_matmul_bias (bias_f32 null: llmhip_matmul) of a size that is computed in pieces of k, by a copy of that kernel whose adding workgroups
 * do not wait for the other pieces' sums but make all of them by themselves, as they do after waiting in vain: the same bits.  LLMHIP_ERR_UNSUPPORTED for
 * other sizes; workspace: 2 MiB are enough for any. */
int llmhip_bench_matmul_alone(void *out, const void *lhs, const void *weight, const void *bias_f32, void *workspace, size_t workspace_bytes,
                              int m, int n, int k, int dt, void *stream);

/* The tile by which llmhip_matmul(_bias) of 17 rows or more goes where k is not cut, lhs rows << 16 | features; 0: not by tiles. */
int llmhip_bench_matmul_tile(int m, int n, int k);

/* Runs, for about target_ms (<= 2000), a loop of back-to-back bf16 32x32x16 MFMAs on N(0,1)
 * operands on every CU and returns the sustained TFLOP/s.  mix 0: the MFMAs alone (what the matrix
 * pipe sustains at the clock its own power draw allows); mix 1: the same MFMAs with the LDS
 * fragment reads and vector instructions of a flash-attention inner loop beside them, no memory
 * traffic, no barriers, no dependences.  Allocates and frees two small device buffers; runs on the
 * default stream. */
int llmhip_bench_mfma_ceiling(int mix, double target_ms, double *tflops);

/* A plain streaming read of two device arrays of bytes_each bytes (a multiple of 16), every byte
 * read once and nothing else done -- what the memory system delivers to a kernel that only reads,
 * to set beside the decode kernel's rate on the same byte count.  variant 0: one workgroup per CU
 * with 8 loads in flight per thread; variant 1: two per CU with 4 (the better one below about
 * 256 MiB).  sink: LLMHIP_BENCH_STREAM_READ_SINK_BYTES bytes of device memory that receive a
 * checksum per wave.  Asynchronous on `stream`; allocates nothing. */
#define LLMHIP_BENCH_STREAM_READ_SINK_BYTES 65536
int llmhip_bench_stream_read(const void *src_a, const void *src_b, size_t bytes_each, void *sink,
                             size_t sink_bytes, int variant, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* LLMHIP_BENCH_H_ */
