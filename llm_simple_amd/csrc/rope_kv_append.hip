// Rotary embedding on Q and K fused with the KV-cache append, gfx950.
//
// Replaces, in one launch, what the reference does with two (or one) rope
// launches plus two device-to-device copies per layer and step
// (src/llama2_layer_npu.cpp:790-798 + :830-844; Llama :206-208 + :325-339):
//   out_q[s][h][:]              = rope(in_q[s][h][:], freq_cis[start_pos+s])
//   out_k[row_off + s][h][:]    = rope(in_k[s][h][:], freq_cis[start_pos+s])
//   out_v[row_off + s][h][:]    = in_v[s][h][:]                    (bytes)
// with out_k / out_v the cache base pointers and row_off = start_pos for the
// append, or plain output tensors with row_off = 0 for the stand-alone rope
// entry points.
//
// Arithmetic follows src/llama2_layer_cpu.cpp:835-856 with the position
// offset of the device contract (tests/rope_single_layer_test.cpp:78-97):
// widen to fp32, (a*c - b*d, a*d + b*c) with every product and sum rounded
// separately (this file is compiled with -ffp-contract=off), one rounding to
// the storage type.  Pairing: interleaved (2f, 2f+1) or neox (f, f + 64).
//
// Pure streaming: a thread takes 32 bytes of a 256-byte head row, 16 of either half (8 pairs: two 128-bit
// loads, 64 bytes of the fp32 table, two 128-bit stores; 8 lanes per row, whole lines in either pairing style), Q, K and
// V rows alike -- a V row is copied by the same 8 lanes without the arithmetic.  The pairing style is a template
// parameter, the storage type is rounded by the hardware conversion (equal to round-to-nearest-even on the bit pattern for
// every non-NaN fp32), the token of a row comes from a multiply-shift division.
//
// Bound by the memory path of three separate streams of 256-byte rows.  4096 tokens of 28 + 2 x 4 heads (75.5 MB): 11.7 us
// with the buffers in the last-level cache, 14.4 from and to HBM, where a plain device copy of the same bytes takes
// 10.2-11.7 and 16-16.6; 256 tokens of 32 + 2 x 32 heads 2.85 us, of which an empty launch is 1.55.  One piece to a thread: two, a
// grid apart, kept half as many waves (a layer's rope and attention, us, two / one: 64 tokens of 32 heads 8.29 / 8.02,
// 256 10.80 / 10.52, 1500 41.9 / 40.9, 256 of 12 9.03 / 8.61).
#include "common.hpp"
#include "kernels.hpp"

namespace llmhip {

// Where the rows of the first token go: fetched from memory while the loads are under way.
struct RopeOut {
  char *q, *k, *v;
};

// The 8 pairs of one thread: a = elements of the first 16-byte chunk, b = of the second.  NEOX: pair i
// = (a[i], b[i]) (dims f, f + 64); interleaved: pair i = elements 2i, 2i+1 of the 16 contiguous ones.
// Arithmetic of src/llama2_layer_cpu.cpp:835-856: every product and sum rounded on its own.
template <typename T, bool NEOX>
__device__ __forceinline__ void rotate8(u32x4_t &va, u32x4_t &vb, const f32x4_t (&cs)[4]) {
  using E = Elem<T>;
  float r0[8], r1[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    uint16_t xa, xb;
    if (NEOX) {
      xa = (uint16_t)(va[i >> 1] >> ((i & 1) * 16));
      xb = (uint16_t)(vb[i >> 1] >> ((i & 1) * 16));
    } else {
      const uint32_t w = (i < 4) ? va[i] : vb[i - 4];
      xa = (uint16_t)w;
      xb = (uint16_t)(w >> 16);
    }
    const float a = E::widen(xa), b = E::widen(xb);
    const float c = cs[i >> 1][2 * (i & 1)], d = cs[i >> 1][2 * (i & 1) + 1];
    r0[i] = a * c - b * d;
    r1[i] = a * d + b * c;
  }
  if (NEOX) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      va[j] = E::pack2(r0[2 * j], r0[2 * j + 1]);
      vb[j] = E::pack2(r1[2 * j], r1[2 * j + 1]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      va[j] = E::pack2(r0[j], r1[j]);
      vb[j] = E::pack2(r0[j + 4], r1[j + 4]);
    }
  }
}

enum RopeWay { kInOrder, kPlaced, kOrdinaryStores };  // (in order too)

// kPlaced: workgroup b works for XCD b % 8, on rows that the attention launch to come reads there (prefill_xcd_share_log2): the
// heads of that XCD's kv heads, or, where two XCDs share one, those of every second token.  What these stores leave in an XCD's L2 is
// valid and clean, and Q, K and V are then read from there; where two XCDs share a kv head, half of what each reads (attention deals
// tiles and heads to the two, and either reads every K and V row).  Which rows go where is nothing but speed.
template <typename T, bool NEOX, RopeWay WAY>
__global__ __launch_bounds__(256) void rope_kv_append_kernel(addresses_t in_, u32x4_t size, u32x2_t heads_, RopeOut to) {
  // in_: q, k, v, the table; size: tokens (kPlaced) or threads, factor and shift of the division by a token's rows in a list (bit 8:
  // there is a V; kPlaced, from bit 9 on: logarithm of the XCDs that share a list), start_pos
  constexpr bool PLACED = WAY == kPlaced;
  const int start_pos = size[3], q_heads = heads_[0], k_heads = heads_[1];
  const uint32_t share = PLACED ? size[2] >> 9 : 0, xcd = PLACED ? blockIdx.x & 7u : 0, lists = PLACED ? 3 - share : 0;
  const uint32_t gid = (PLACED ? blockIdx.x >> 3 : blockIdx.x) * 256u + threadIdx.x;
  if (!PLACED && gid >= size[0]) return;
  const int q_list = q_heads >> lists, k_list = k_heads >> lists;
  const FastDiv rows_per_token = {(uint32_t)(q_list + k_list + (size[2] & 256u ? k_list : 0)), size[1], size[2] & 255u};
  const uint32_t j = gid & 7u, rowid = gid >> 3, t = fast_div(rowid, rows_per_token);
  const uint32_t s = PLACED ? (t << share) + (xcd & ((1u << share) - 1)) : t;
  if (PLACED && s >= size[0]) return;
  const int r = (int)(rowid - t * rows_per_token.d), list = xcd >> share;
  const bool is_q = r < q_list, rotated = r < q_list + k_list;
  const int heads = is_q ? q_heads : k_heads;  // V has as many as K
  const int h = is_q ? list * q_list + r : list * k_list + r - q_list - (rotated ? 0 : k_list);
  const char *in = at_address<const char>(is_q ? in_[0] : rotated ? in_[1] : in_[2]);
  in += ((size_t)s * heads + h) * kRowBytes + j * 16;
  const float *tab = at_address<const float>(in_[3]) + (size_t)(start_pos + s) * kHeadDim + (NEOX ? 16 : 8) * j;
  // All loads go out before anything is waited for, the table's included (a V row's are not used)
  u32x4_t a = global_load_b128(in), b = global_load_b128(in + 128);
  f32x4_t cs[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) cs[i] = *reinterpret_cast<const f32x4_t *>(tab + (NEOX ? 4 * i : 64 * (i >> 1) + 4 * (i & 1)));
  __builtin_amdgcn_sched_barrier(0);
  char *out = is_q ? to.q : rotated ? to.k : to.v;
  out += ((size_t)s * heads + h) * kRowBytes + j * 16;
  if (rotated) rotate8<T, NEOX>(a, b, cs);
  // Past the L2: the attention launch that follows finds nothing to wait for, and every instruction writes whole lines
  // (interleaved pairs used to be 32 bytes of a lane, stored by halves: 1019 tokens of 32 heads then take 32.8 us this way).
  // Rope and attention, us, ordinary stores / these: 256 tokens of 28 heads 9.88 / 9.38, 1019 of 28 21.9 / 20.8, 400 of 40
  // 13.7 / 12.7, 4096 of 28 130.8 / 130.1; whole lines alone 256 tokens of 32 heads, interleaved, 11.7 -> 11.3, both 10.6.
  // (Non-temporal stores are shorter still by themselves, and the rows then come back from HBM: 1019 tokens 24.3.)
  if constexpr (WAY == kOrdinaryStores) {
    *reinterpret_cast<u32x4_t *>(out) = a;
    *reinterpret_cast<u32x4_t *>(out + 128) = b;
  } else {
    store_device_b128(out, a);
    store_device_b128(out + 128, b);
  }
}

constexpr int kPlacedTokens = 64;
constexpr long long kPlacedBytes = 13 << 19;
constexpr long long kOffSectorBytes = 11 << 20;

template <typename T> static auto kernel_of(bool neox, RopeWay way) {
  if (way == kPlaced) return neox ? rope_kv_append_kernel<T, true, kPlaced> : rope_kv_append_kernel<T, false, kPlaced>;
  if (way == kOrdinaryStores) return neox ? rope_kv_append_kernel<T, true, kOrdinaryStores> : rope_kv_append_kernel<T, false, kOrdinaryStores>;
  return neox ? rope_kv_append_kernel<T, true, kInOrder> : rope_kv_append_kernel<T, false, kInOrder>;
}

hipError_t launch_rope_kv_append(void *out_q, void *out_k, void *out_v, const void *freq_cis,
                                 const void *in_q, const void *in_k, const void *in_v,
                                 int start_pos, int cur_size, int q_heads, int k_heads,
                                 int k_out_row_offset, int is_neox, int dt, hipStream_t stream) {
  const long long rows = (long long)q_heads + k_heads + (in_v != nullptr ? k_heads : 0);
  const long long total = (long long)cur_size * rows * 8;
  if (total == 0) return hipSuccess;
  if (rows > 0x7FFFFFFFLL || total > 0x7FFFFFFFLL) return hipErrorInvalidValue;  // 32-bit thread index
  // Rows placed: a prompt (a chunk's workgroups are dealt otherwise) of kv heads that make whole lists, where what is written fits
  // the L2s beside what is read.  Rope and attention, us, in order / placed: 128 tokens of 32 kv heads 8.19 / 7.15, 256 9.47 / 9.10,
  // 300 10.42 / 10.42, 512 13.66 / 13.87; 200 of 8 (40 heads) 8.52 / 8.05, 400 11.28 / 11.04, 600 14.07 / 14.17; 200 of 4 (28) 8.00 / 7.76,
  // 512 11.59 / 11.21, 700 14.01 / 14.06, 1019 18.12 / 18.21; 20 of 4 6.21 / 6.32.  Four XCDs to a kv head: nothing (256 of 2 7.73 / 7.79).
  const int share = k_heads > 0 ? prefill_xcd_share_log2(k_heads) : -1;  // logarithm of the XCDs of a list
  const bool placed = cur_size >= kPlacedTokens && prefill_is_prompt(cur_size, (long long)start_pos + cur_size) &&
                      total * 32 <= kPlacedBytes && (share == 0 || share == 1) && q_heads % k_heads == 0;
  const uint32_t list_rows = (uint32_t)(placed ? rows >> (3 - share) : rows);
  const FastDiv div = make_fast_div(list_rows);
  const size_t first = (size_t)k_out_row_offset * k_heads * kRowBytes;
  const RopeOut to = {static_cast<char *>(out_q), static_cast<char *>(out_k) + first, static_cast<char *>(out_v) + first};
  // An output that does not begin on a 64-byte sector shares the first and the last one of every 128 bytes with the next store, and
  // past the L2 both halves are a write to memory of their own; up to some MB that is hidden.  Ordinary stores where more than
  // 11 MiB go to such outputs (us, past the L2 / ordinary, base 16 bytes off: 1200 tokens of 28 + 2 x 4 heads, 11.1 MB, with attention
  // 25.9 / 26.2, 1400 30.2 / 30.25, 1700 39.1 / 37.7, 4096 136.5 / 133.9, alone 16.45 / 13.2; 256 of 32 + 2 x 32 10.59 / 10.57, 512, 12.6
  // MB, 16.2 / 15.1, 1019 30.7 / 28.65; 32 off 512 of them 15.5 / 15.1.  64 off: 512 14.3 / 14.8, 2048 of 28 44.8 / 45.5.)
  auto off_sector = [&](const void *p, long long heads) { return (address(p) & 63) != 0 ? cur_size * heads * kRowBytes : 0; };
  const long long off = off_sector(out_q, q_heads) + off_sector(to.k, k_heads) + off_sector(to.v, in_v != nullptr ? k_heads : 0);
  const RopeWay way = placed ? kPlaced : off > kOffSectorBytes ? kOrdinaryStores : kInOrder;
  const long long threads = placed ? (long long)((cur_size + (1 << share) - 1) >> share) * list_rows * 8 : total;
  const int grid = (int)((threads + 255) / 256) * (placed ? 8 : 1);
  const auto kern = (dt == kDtFloat16) ? kernel_of<_Float16>(is_neox, way) : kernel_of<__bf16>(is_neox, way);
  return launch(kern, dim3(grid), 256, 0, stream, addresses_t{address(in_q), address(in_k), address(in_v), address(freq_cis)},
                u32x4_t{(uint32_t)(placed ? cur_size : total), div.m,
                        div.l | (in_v != nullptr ? 256u : 0u) | (placed ? (uint32_t)share << 9 : 0u), (uint32_t)start_pos},
                u32x2_t{(uint32_t)q_heads, (uint32_t)k_heads}, to);
}

}  // namespace llmhip
