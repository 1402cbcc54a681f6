// GQA-aware split-KV decode attention for gfx950 (MI355X).
//
// The reference decodes with the same operator as prefill, m = 1 and offset =
// n - 1 (npu_flash_attn_gqa_layer, src/llama2_layer_npu.cpp:866-869): one
// softmax row per head over the whole contiguous KV cache
// [max_seq_len][Hkv][128] (src/llama2_layer_npu.cpp:1148-1149).  That is a
// pure stream of K and V through the chip, so the kernel is organised around
// HBM: grid = (KV split, kv head, sequence); a workgroup takes every
// num_splits-th block of 128 keys of one kv head (the workgroups of a sequence
// walk through its cache side by side), each of its 4 waves 32 keys of a block,
// and K and V of every key are read from HBM exactly once for all group_size
// query heads (and all m <= 16/group_size query rows) that share the kv head.
//
// The m*group_size query rows are the 16 columns of mfma_f32_16x16x32
// (S^T = K Q^T, O^T += V^T P^T); unused columns are zero.  Every load
// instruction fetches whole 256-byte head rows (16 lanes per row); K and V are
// staged in wave-private LDS regions, K read back in the A-operand layout
// (loading K straight into that layout -- 16 rows x 16 bytes per quarter wave --
// costs the texture cache 16 tag look-ups where this costs 2, and measured 1-2 %
// slower), V read transposed with ds_read_b64_tr_b16.  K and V are read once, so
// their loads are non-temporal (7.1 TB/s at 2 GiB where ordinary loads give 6.2),
// and K and V of a step are fetched one after the other so that a CU has 32 KiB
// in flight, not 64 (see the loop).  Each wave keeps its own running (max, sum,
// O); the
// waves are merged through LDS at the end and the workgroup writes the final rows (one split) or an
// fp32 partial (max, sum, unnormalised O).
//
// Up to 128 partials of a (sequence, kv head) are folded (log-sum-exp) by workgroups of the same launch that do nothing else
// (folders): every word of a partial goes past the XCD's L2 (sc1 stores) with half of the launch's number beside it, and a folder
// looks at all of them until it finds the number everywhere.  That is one way to memory and one back; no fence, no flag, no atomic.
// Folders have the highest workgroup numbers, so that an XCD dispatches them after the workgroups of their own launch, and on
// idle CUs if there are any.  Of launches on two streams one's folders can hold the CUs that the other's workgroups wait for, and the other way
// round on another XCD: a folder that has looked in vain for long (see fold_looks) computes its rows from the caches by itself, so that nothing
// depends on the order of dispatch but time, and a row's last bits.  A look costs what its loads cost: a wave per row, two dims per lane, the maxima and
// sums of all partials in one load (two rows per wave with three loads per partial: 1.5 us a look, 0.6 now).
// (Fused step, us, the last workgroup to store folds / folders: 384 keys of 2 kv heads 5.52 / 4.85, 512 of 32 5.23 / 5.01, 32768 of 8, with
// a combine launch before, 24.25 / 23.93; 5 x 2999 keys of 8 13.9 / 13.1; beyond 32 partials, a combine launch / folders: 4700 keys of
// 4 kv heads 7.92 / 7.06, 14000 10.45 / 9.62, 31000 15.2 / 14.5, 6000 of 2 7.77 / 6.68, 20000 10.25 / 9.58.  Since a folder reads the sums of
// its parts at once, 32768 of 8 23.9 -> 23.5.)
// More than 8 query rows (a few tokens checked at once) take folders where the room is there, with tags twice that of the partials (rope
// and attention, us, flags or a combine launch / folders: 2 tokens past 1200 keys of 28 + 4 heads 10.1 / 7.8, past 20000 14.1 / 13.3, 3 past
// 1500 of 40 + 8 11.1 / 8.4, 12 past 900 of 32 + 32 10.9 / 9.15).
// Where the number would be that of a replay, or without that room, few partials of few rows are folded by the workgroup that finds them all
// stored: partials, then a flag, then a look at the other flags, then the partials, four round trips to memory.  Beyond that, or
// beyond 128 partials, there is a second launch.  (Device-scope fences instead of sc1 accesses write back and invalidate the XCD's L2: 91 us
// against 33 at batch 1, 32768 keys.)
//
// A short cache is bound by the length of one workgroup's chain, not by bytes: at 32 keys, one sequence, the
// kernel took 6.3 us, 2.5 us of them the launch.  A wave issues a vector instruction every 4-5 cycles, so the
// chain is kept short: the query (and table) loads go out before the first keys and are waited for after
// them, the new K row of a fused step is rotated in a spare query column, bf16 results are rounded by the conversion
// instruction, K and V rows are read through buffer descriptors (the hardware bounds them, no clamps), integer
// divisions are prepared by the host, the column maximum goes through permlane swaps, masks and the
// rescaling of O run only where they change something, and the merge of the waves is free of bank conflicts (it cost
// 1.4 us).  4.1 us now.
//
// (Eight-wave workgroups, half as many, merging pairs of splits through LDS: 4.5 TB/s against 6.0 at the time.)
#include <atomic>
#include <chrono>
#include <random>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "launch_number.hpp"

namespace LLMHIP_NS {

constexpr int kDecWaveKeys = 32;                  // keys per wave per step
constexpr int kDecStepKeys = 4 * kDecWaveKeys;    // keys per workgroup per step (half of it in short caches)
constexpr int kDecCols = 16;                      // query rows per kv head (MFMA N)
constexpr int kDecWaveLds = kDecWaveKeys * kRowBytes;  // 8 KiB of staging per wave, for K and for V
constexpr int kDecLdsPad = 24 * 1024;             // with the 64 KiB of staging: more than half a CU's LDS

// What a launch is told.  What its first loads need is packed into the first 14 words of a kernel's arguments, which are in
// registers when it starts (DecodeEarly); the rest comes as a struct, fetched while those loads are under way.  (Fused step, us,
// all in the struct / this: 384 keys of 2 kv heads 5.94 / 5.52, 512 of 32 5.72 / 5.36, 4096 of 8 8.58 / 8.03, 32768 of 8 24.94 /
// 24.36; 5 x 2999 keys of 8 14.1 / 13.9.)
struct DecodeLate {
  char *out;
  float *ws_o;   // [batch][Hkv][splits][cols][128]
  float *ws_ml;  // [batch][Hkv][splits][cols][2]; fold: the last column's place is the flag of the split
  int num_splits;
  int iters_each, iters_rest;  // blocks per split: iters_each, one more for the first iters_rest splits
  int fold_rows, folders;  // by tags: rows of a folder and, 8 bits on, the looks that it takes; folders of a (sequence, kv head)
  FastDiv folders_div;
  uint64_t fold;  // the launch's number: what the flags hold, or halves of it beside the words of a partial
};
// rows = m * g query rows of a kv head, at most 16.  Fused decode step (FUSED kernels only): the token at row n - 1 is not in the
// cache yet.  q, new_k and new_v hold the unrotated projections of that token ([H][128], [Hkv][128] twice);
// q and the new K row are rotated with table row freq_row (64 (cos, sin) pairs) as they are loaded,
// and the workgroup that owns the last key range writes the rotated K row and the V row to the cache.
struct DecodeParams : DecodeLate {
  const void *q, *k, *v;
  const void *freq_row, *new_k, *new_v;
  int batch, m, n, offset;
  int64_t kv_seq_stride;  // 0: the sequences are tiles of m tokens of one
  int tokens;             // of all sequences or tiles: the last tile may be short
  int g, Hkv, rows;
  int is_neox;
  bool fused;
  bool two;  // workgroups to a CU
  int cols;  // columns of a partial's slot: 16, or 8 of workgroups of two waves
};
// a: q, K, V, then freq_row or kv_seq_stride; b: new_k and new_v, or rows | m << 8 | tokens << 16, 2^16 / g + 1, offset, pairs | 2^20 / Hkv (rounded
// up) << 10 (pairs = batch * Hkv, where the partials are folded by tags: at most kTaggedPairs); c: n, Hkv | g << 16 | is_neox << 31
struct DecodeEarly {
  addresses_t a;
  u32x4_t b;
  u32x2_t c;
  explicit DecodeEarly(const DecodeParams &p) {
    a = addresses_t{address(p.q), address(p.k), address(p.v), p.fused ? address(p.freq_row) : (uint64_t)p.kv_seq_stride};
    const uint64_t nk = address(p.new_k), nv = address(p.new_v);
    b = p.fused ? u32x4_t{(uint32_t)nk, (uint32_t)(nk >> 32), (uint32_t)nv, (uint32_t)(nv >> 32)}
                : u32x4_t{(uint32_t)(p.rows | p.m << 8) | (uint32_t)p.tokens << 16, 65536u / p.g + 1, (uint32_t)p.offset,
                          (uint32_t)(p.batch * p.Hkv) | ((1u << 20) + p.Hkv - 1) / p.Hkv << 10};
    c = u32x2_t{(uint32_t)p.n, (uint32_t)p.Hkv | (uint32_t)p.g << 16 | (uint32_t)p.is_neox << 31};
  }
};

// RoPE of the four 16-byte fragments a lane holds of one head row: fragment kk = dims 8*cg + 32*kk .. +7.
// Arithmetic of the rotary kernel, unfused products and sums (src/llama2_layer_cpu.cpp:835-856):
// (a*c - b*s, a*s + b*c) rounded once; interleaved pairs (2f, 2f+1), neox pairs (f, f+64).
// The lane's 16 (cos, sin) pairs are 8 pieces of 16 bytes of the table row.
__device__ __forceinline__ void load_rotation(f32x4_t (&t)[8], const float *row, int cg, int is_neox) {
  const float *at = row + (is_neox ? 16 * cg : 8 * cg);
  const int far = is_neox ? 64 : 32, near = is_neox ? 4 : 2;  // floats between groups, pieces of a group
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = *reinterpret_cast<const f32x4_t *>(at + far * (is_neox ? i >> 2 : i >> 1) + 4 * (i & (near - 1)));
}
template <typename T>
__device__ __forceinline__ void rotate_frags(u32x4_t (&f)[4], const f32x4_t (&t)[8], int is_neox) {
#pragma clang fp contract(off)
  using E = Elem<T>;
  auto lo = [](uint32_t w) { return E::widen((uint16_t)(w & 0xffffu)); };
  auto hi = [](uint32_t w) { return E::widen((uint16_t)(w >> 16)); };
  if (is_neox) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4_t cs = t[4 * kk + j];
        const float a0 = lo(f[kk][j]), a1 = hi(f[kk][j]), b0 = lo(f[kk + 2][j]), b1 = hi(f[kk + 2][j]);
        f[kk][j] = E::pack2(a0 * cs[0] - b0 * cs[1], a1 * cs[2] - b1 * cs[3]);
        f[kk + 2][j] = E::pack2(a0 * cs[1] + b0 * cs[0], a1 * cs[3] + b1 * cs[2]);
      }
  } else {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float c = t[2 * kk + (j >> 1)][2 * (j & 1)], sn = t[2 * kk + (j >> 1)][2 * (j & 1) + 1];
        const float x = lo(f[kk][j]), y = hi(f[kk][j]);
        f[kk][j] = E::pack2(x * c - y * sn, x * sn + y * c);
      }
  }
}

// Maximum / sum over the four lanes that hold one column (they differ in bits 4 and 5 of the lane index):
// v_permlane16_swap and v_permlane32_swap, no LDS crossbar.
template <typename F> __device__ __forceinline__ float quad_reduce(float x, F f) {
  typedef __attribute__((ext_vector_type(2))) unsigned u2;
  unsigned u = __builtin_bit_cast(unsigned, x);
  u2 r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  unsigned r0 = r[0], r1 = r[1];
  u = __builtin_bit_cast(unsigned, f(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1)));
  r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  r0 = r[0];
  r1 = r[1];
  return f(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}
__device__ __forceinline__ float quad_max(float x) {
  return quad_reduce(x, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float quad_sum(float x) {
  return quad_reduce(x, [](float a, float b) { return a + b; });
}

// V staging swizzle for the 16x16x32 transposed reads: one instruction touches
// 8 rows x 32 bytes per half-wave, so the 32-byte slot index is XORed with
// row%8.
__device__ __forceinline__ int v_swizzle32_off(int row, int granule) {
  return row * kRowBytes + ((((granule >> 1) ^ (row & 7)) << 5) | ((granule & 1) << 4));
}

constexpr int kMaxTaggedSplits = 128;
constexpr int kTaggedBytes = (kHeadDim + 2) * 8;  // a row of a partial whose words carry a tag
constexpr int kTaggedPairs = 1023;                // (sequence, kv head) pairs, at most
constexpr int kFoldDepth = 8;                     // partials that are summed in one part
// Looks that a folder takes, 0.6 us each or more: what its whole cache takes one workgroup, eight times over, and 0.3 ms.  It is there for
// launches on two streams (see above), which a wait of any length only holds up; too short a wait makes work, and rows summed in another order,
// where other kernels hold the workgroups up that it waits for.
static int fold_looks(int nblocks) {
#ifdef LLMHIP_BENCH
  return 0;  // (the measurement library's copy: every folder computes its rows by itself)
#else
  constexpr double kBlockUs = 2.0 * kRowBytes * kDecStepKeys * 1e-3 / 27.9, kLookUs = 0.6;  // (a CU's share of the memory system, see split_model_us)
  const double looks = (300.0 + 8.0 * kBlockUs * nblocks) / kLookUs;
  return looks < 1 << 16 ? (int)looks : 1 << 16;
#endif
}
// Parts that a row's partials are summed in before those sums are: part i has splits i, i + parts, ...  That is the order of the
// combine launch, so that all ways to fold give the same bits.
constexpr int kParts = 8;
__host__ __device__ constexpr int fold_parts(int splits) { return splits <= kFoldDepth ? 1 : kParts; }

__device__ __forceinline__ float bits_float(uint32_t u) { return __builtin_bit_cast(float, u); }

// The sum of partials, four dims of it per thread.
struct PartialSum {
  float M = -INFINITY, L = 0.0f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
  template <int D> __device__ __forceinline__ void take(const u32x2_t (&ml)[D], const f32x4_t (&ov)[D], int have) {
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (j < have) M = fmaxf(M, bits_float(ml[j][0]));
    const float M_use = (M == -INFINITY) ? 0.0f : M;
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const float wt = (j < have) ? fast_exp2(bits_float(ml[j][0]) - M_use) : 0.0f;
      L += wt * bits_float(ml[j][1]);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] += wt * ov[j][i];
    }
  }
};

// Maximum over each N = 2, 4 or 8 lanes.
template <int N> __device__ __forceinline__ float max_of_lanes(float x) {
  auto with = [&](auto control) {
    const int i = __builtin_bit_cast(int, x);
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, decltype(control)::value, 0xf, 0xf, false)));
  };
  with(std::integral_constant<int, 0xB1>());                     // quad_perm: lane ^ 1
  if (N >= 4) with(std::integral_constant<int, 0x4E>());         // quad_perm: lane ^ 2
  if (N == 8) with(std::integral_constant<int, 0x141>());        // row_half_mirror: the other quad
  return x;
}
__device__ __forceinline__ float lane_value(float x, int lane) {
  return bits_float(__builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// A folder: rows c0 .. c0 + fold_rows - 1 of a pair, from partials whose words carry this launch's tags.  A wave has a row, two
// dims per lane, and PARTS of the fold_parts() parts of its partials, DEPTH in all.  It looks at all of them until it finds the tags
// at every word.  A part's partials are summed ROUND at a time, as in the combine launch.  have_rows: of the pair's rows, those that
// are there (a short last tile).  A bit per row c0 + i that was not stored: its partials were not there after all looks.
template <typename T, int NW, int DEPTH, int PARTS, int ROUND>
__device__ __forceinline__ uint32_t fold_tagged(const DecodeLate &p, uint32_t row_part, char *lds, int pair, int token, int kvh, int c0, int rows,
                                                int have_rows, int Hkv, int g) {
  constexpr int EACH = DEPTH / PARTS;  // (PARTS 1: of one part, else of kParts)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, S = p.num_splits;
  constexpr int parts = PARTS > 1 ? kParts : 1, per_row = parts / PARTS, at_once = NW / per_row;
  const int part = wave / at_once, c = c0 + wave % at_once;
  const bool mine = wave % at_once < (p.fold_rows & 0xff) && c < have_rows;  // (of the wave)
  const int bytes = S * rows * kTaggedBytes;
  const __amdgpu_buffer_rsrc_t pt = byte_buffer(reinterpret_cast<char *>(p.ws_o) + (size_t)pair * bytes, bytes);
  const uint32_t tag0 = (uint32_t)p.fold, tag1 = (uint32_t)(p.fold >> 32);
  float M[PARTS], L[PARTS], x[PARTS], y[PARTS];
  bool there = true;
#pragma unroll
  for (int i = 0; i < PARTS; ++i) {
    M[i] = -INFINITY;
    L[i] = x[i] = y[i] = 0.0f;
  }
  if (mine) {
    // (no branches: past the splits the offset is past the buffer, and the load is not made)
    auto split_of = [&](int j) { return part + per_row * (j / EACH) + parts * (j % EACH); };
    int at[DEPTH];
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) at[j] = split_of(j) < S ? (split_of(j) * rows + c) * kTaggedBytes + lane * 16 : 0x40000000;
    const int my_split = split_of(lane & (DEPTH - 1));
    const bool have = my_split < S;
    const int at_ml = have ? (my_split * rows + c) * kTaggedBytes + kHeadDim * 8 : 0x40000000;
    u32x4_t a[DEPTH] = {}, ml = {};
    there = false;
    for (int looks = p.fold_rows >> 8; looks > 0; --looks) {
      asm volatile("" ::: "memory");  // (the loads are made again)
      ml = __builtin_bit_cast(u32x4_t, load_device(pt, at_ml));
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) a[j] = __builtin_bit_cast(u32x4_t, load_device(pt, at[j]));
      uint32_t differs = have ? (ml[1] ^ tag0) | (ml[3] ^ tag1) : 0u;
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) differs |= split_of(j) < S ? (a[j][1] ^ tag0) | (a[j][3] ^ tag1) : 0u;
      there = __builtin_amdgcn_ballot_w64(differs != 0) == 0;
      if (there) break;
      __builtin_amdgcn_s_sleep(1);
    }
    // the maximum of each round of partials, then, in the lanes of a round, that of its part up to there
    const float my_m = have ? bits_float(ml[0]) : -INFINITY, my_l = have ? bits_float(ml[2]) : 0.0f;
    const float of_round = max_of_lanes<ROUND>(my_m);
    float upto[DEPTH / ROUND], mine_upto = of_round;
#pragma unroll
    for (int r = 0; r < DEPTH / ROUND; ++r) {
      upto[r] = lane_value(of_round, r * ROUND);
      if (r * ROUND % EACH != 0) upto[r] = fmaxf(upto[r], upto[r - 1]);
      if (ROUND < EACH && (lane & (DEPTH - 1)) / ROUND == r) mine_upto = upto[r];
    }
    const float wt = have ? fast_exp2(my_m - (mine_upto == -INFINITY ? 0.0f : mine_upto)) : 0.0f;
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      const int i = j / EACH, r = j / ROUND;
      if (j % ROUND == 0) {
        if (j % EACH != 0) {
          const float resc = fast_exp2(M[i] - (upto[r] == -INFINITY ? 0.0f : upto[r]));
          L[i] *= resc;
          x[i] *= resc;
          y[i] *= resc;
        }
        M[i] = upto[r];
      }
      const float w = lane_value(wt, j);
      L[i] += w * lane_value(my_l, j);
      x[i] += w * bits_float(a[j][0]);
      y[i] += w * bits_float(a[j][2]);
    }
  }
  uint32_t *failed = reinterpret_cast<uint32_t *>(lds);  // of each wave, the bit of its row
  if (lane == 0) failed[wave] = there ? 0u : 1u << (c - c0);
  bool whole = there;  // of the row's waves
  if constexpr (PARTS > 1) {
    // part i of row `wave` is in place wave + i * at_once
    float part_m[kParts], part_l[kParts], part_x[kParts], part_y[kParts];
    if constexpr (PARTS == kParts) {
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        part_m[i] = M[i];
        part_l[i] = L[i];
        part_x[i] = x[i];
        part_y[i] = y[i];
      }
    } else {
      float *red_ml = reinterpret_cast<float *>(lds) + 16, *red_o = red_ml + 2 * NW * PARTS;
#pragma unroll
      for (int i = 0; i < PARTS; ++i) {
        const int place = wave + i * NW;
        if (lane == 0) *reinterpret_cast<float2 *>(red_ml + 2 * place) = float2{M[i], there ? L[i] : -1.0f};
        *reinterpret_cast<float2 *>(red_o + place * kHeadDim + 2 * lane) = float2{x[i], y[i]};
      }
      __syncthreads();
      // (all of them read before the first is used: in a loop a turn is a trip to LDS, 32768 keys of 8 kv heads 23.0 us, 22.5 so)
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        const int place = part == 0 ? wave + i * at_once : 0;
        const float2 ml_i = *reinterpret_cast<const float2 *>(red_ml + 2 * place), o = *reinterpret_cast<const float2 *>(red_o + place * kHeadDim + 2 * lane);
        part_m[i] = ml_i.x;
        part_l[i] = ml_i.y;
        part_x[i] = o.x;
        part_y[i] = o.y;
        if (part_l[i] < 0.0f) whole = false;
      }
    }
    M[0] = -INFINITY;
#pragma unroll
    for (int i = 0; i < kParts; ++i) M[0] = fmaxf(M[0], part_m[i]);
    const float M_use = (M[0] == -INFINITY) ? 0.0f : M[0];
    L[0] = x[0] = y[0] = 0.0f;
#pragma unroll
    for (int i = 0; i < kParts; ++i) {
      const float wt = fast_exp2(part_m[i] - M_use);  // 0 for a part without splits (-inf)
      L[0] += wt * part_l[i];
      x[0] += wt * part_x[i];
      y[0] += wt * part_y[i];
    }
  }
  if (mine && part == 0 && whole) {
    const int r = (int)(c * row_part >> 16);  // (c / g)
    const float inv = (L[0] > 0.0f) ? 1.0f / L[0] : 0.0f;
    char *row = p.out + (((size_t)token + r) * Hkv * g + kvh * g + c - r * g) * kRowBytes;
    *reinterpret_cast<uint32_t *>(row + (lane & 15) * 16 + (lane >> 4) * 4) = Elem<T>::pack2(x[0] * inv, y[0] * inv);
  }
  __syncthreads();
  uint32_t missing = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) missing |= failed[w];
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(missing);
}

// The argument struct of the running kernel, asked for here (as a parameter that two branches use it is fetched, and waited
// for, before they part).
__device__ __forceinline__ DecodeLate fetch_late() {
  constexpr int at = sizeof(addresses_t) + sizeof(u32x4_t) + sizeof(u32x2_t);
  static_assert(at % alignof(DecodeLate) == 0);
  auto arguments = (__attribute__((address_space(4))) const char *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(arguments));
  struct Words {
    uint64_t w[sizeof(DecodeLate) / 8];
  } words;
#pragma unroll
  for (size_t i = 0; i < sizeof(DecodeLate) / 8; ++i)
    words.w[i] = ((__attribute__((address_space(4))) const uint64_t *)(arguments + at))[i];
  DecodeLate p = __builtin_bit_cast(DecodeLate, words);
  p.out = at_address<char>((uint64_t)p.out);
  p.ws_o = at_address<float>((uint64_t)p.ws_o);
  p.ws_ml = at_address<float>((uint64_t)p.ws_ml);
  return p;
}

// How the partials of a (sequence, kv head) become rows: not here (one split, or the combine launch), by the workgroup that
// finds all flags up, by folders that look for tags.  A kernel each: the code of the others in the way costs a call of 4 us 0.05.
enum FoldMode { kNoFold, kFoldByFlags, kFoldByTags };

template <typename T, bool FUSED, int NW, bool LONG, FoldMode FOLD>
__global__ __launch_bounds__(64 * NW) void flash_decode_kernel(addresses_t ea, u32x4_t eb, u32x2_t ec, DecodeLate late) {
  using E = Elem<T>;
  const int n = ec[0], Hkv = ec[1] & 0xffffu, g = ec[1] >> 16 & 0xffu, H = g * Hkv;
  const bool is_neox = ec[1] >> 31;
  const int all_rows = FUSED ? g : eb[0] & 0xffu, m = FUSED ? 1 : eb[0] >> 8 & 0xffu;
  const uint32_t row_part = FUSED ? 0u : eb[1];  // (of a column, 16 bits on: its query row)
  constexpr int cols = NW == 2 ? kDecCols / 2 : kDecCols;
  auto token_of = [&](int seq) { return FUSED ? 0 : seq * m; };  // first token of a sequence, or of a tile of one
  auto rows_from = [&](int token) { return FUSED ? g : min(all_rows, ((int)(eb[0] >> 16) - token) * g); };  // (the last tile may be short)
  const int fused_pos = n - 1;
  constexpr int kStepKeys = NW * kDecWaveKeys;
  __shared__ __attribute__((aligned(16))) char lds[2 * NW * kDecWaveLds];

  int split = blockIdx.x, kvh = blockIdx.y, b = FUSED ? 0 : blockIdx.z;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int col = lane & 15, cg = lane >> 4;
  bool lone = false;  // a folder that stopped waiting: all keys of its (sequence, kv head)
  uint32_t lone_rows = 0;  // and its own rows that are not stored yet.  (Not those of other folders, which may be stored: out may be q.)
  if constexpr (FOLD == kFoldByTags) {
    const int pairs = FUSED ? Hkv : eb[3] & 0x3ffu;
    int pair = blockIdx.y;
    if (__builtin_expect(pair >= pairs, 0)) {
      const DecodeLate f = fetch_late();
      const int e = (pair - pairs) * f.num_splits + split;
      if (e >= pairs * f.folders) return;
      pair = (int)fast_div(e, f.folders_div);
      b = FUSED ? 0 : (int)(pair * (eb[3] >> 10) >> 20);
      const int c0 = (e - pair * f.folders) * (f.fold_rows & 0xff);
      auto fold = [&](auto depth, auto parts, auto round) {
        return fold_tagged<T, NW, decltype(depth)::value, decltype(parts)::value, decltype(round)::value>(f, row_part, lds, pair, token_of(b), pair - b * Hkv,
                                                                                                          c0, all_rows, rows_from(token_of(b)), Hkv, g);
      };
      using std::integral_constant;
      const integral_constant<int, 1> one;
      const integral_constant<int, 2> two;
      const integral_constant<int, 4> four;
      const integral_constant<int, 8> eight;
      const integral_constant<int, 16> sixteen;
      const int S = f.num_splits;
      uint32_t missing;
      if constexpr (NW == 4)
        missing = S > 64           ? fold(integral_constant<int, 32>(), two, four)
                  : S > 32         ? fold(sixteen, two, four)
                  : S > 16         ? fold(eight, two, four)
                  : S > kFoldDepth ? fold(sixteen, eight, two)
                  : S > 4          ? fold(eight, one, eight)
                                   : fold(four, one, four);
      else
        missing = S > 16           ? fold(sixteen, four, four)
                  : S > kFoldDepth ? fold(sixteen, eight, two)
                  : S > 4          ? fold(eight, one, eight)
                                   : fold(four, one, four);
      if (missing == 0)
        return;
      lone = true;
      lone_rows = missing << c0;
      split = 0;
    }
    b = FUSED ? 0 : (int)(pair * (eb[3] >> 10) >> 20);
    kvh = pair - b * Hkv;
  }
  const int token = token_of(b), rows = rows_from(token);
  const int offset = FUSED ? n - 1 : (int)eb[2] + (ea[3] == 0 ? token : 0);
  const DecodeLate p = FOLD == kFoldByTags ? fetch_late() : late;
  const int num_splits = lone ? 1 : p.num_splits;

  const int row_bytes = Hkv * kRowBytes;
  const size_t seq_off = ((FUSED ? 0 : (size_t)b * ea[3] * Hkv) + kvh) * kRowBytes;
  const char *kbase = at_address<const char>(ea[1]) + seq_off, *vbase = at_address<const char>(ea[2]) + seq_off;
  const int stored = FUSED ? n - 1 : n;  // rows that are in the cache

  // query column of this lane
  const bool col_valid = col < rows;
  const int c_row = FUSED || !col_valid ? 0 : (int)(col * eb[1] >> 16);  // (col / g)
  const int c_head = kvh * g + (col_valid ? col - c_row * g : 0);
  const int c_limit = c_row + offset;  // last visible key of this column
  const bool new_col = FUSED && col == rows;  // this column carries the new K row through the rotation
  const char *new_k_row = nullptr;
  const float *freq_row = nullptr;

  u32x4_t qf[4];
  f32x4_t tab[8];
  u32x4_t new_v;
  {
    const char *qp = at_address<const char>(ea[0]) + (size_t)token * H * kRowBytes;
    uint32_t qo = (c_row * H + c_head) * kRowBytes + cg * 16;
    if (FUSED) {
      new_k_row = at_address<const char>(eb[0] | (uint64_t)eb[1] << 32) + kvh * kRowBytes;
      freq_row = at_address<const float>(ea[3]);
    }
    if (new_col) {
      qp = new_k_row;
      qo = cg * 16;
    }
    qp += qo;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[kk] = u32x4_t{0u, 0u, 0u, 0u};
    if (col_valid || new_col) {
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) qf[kk] = global_load_b128(qp + kk * 64);
    }
    if (FUSED) {
      load_rotation(tab, freq_row, cg, is_neox);
      new_v = global_load_b128(at_address<const char>(eb[2] | (uint64_t)eb[3] << 32) + kvh * kRowBytes + col * 16);
    }
  }

  int voff[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) voff[i] = (wave * kDecWaveKeys + 4 * i + cg) * row_bytes + col * 16;
  u32x4_t kn[8], vn[8];
  auto block_buffer = [&](const char *base, int it) {
    const int first = (it * num_splits + split) * kStepKeys;
    const int have = min(stored - first, kStepKeys);
    const unsigned records = have > 0 ? (unsigned)(have - 1) * row_bytes + kRowBytes : 0u;
    return byte_buffer(base + (size_t)first * row_bytes, records);
  };
  auto issue_k = [&](int it) {
    const __amdgpu_buffer_rsrc_t r = block_buffer(kbase, it);
#pragma unroll
    for (int i = 0; i < 8; ++i) kn[i] = stream_load(r, voff[i]);
  };
  auto issue_v = [&](int it) {
    const __amdgpu_buffer_rsrc_t r = block_buffer(vbase, it);
#pragma unroll
    for (int i = 0; i < 8; ++i) vn[i] = stream_load(r, voff[i]);
  };
  // The first step's K and V start together.  From then on they are fetched one after the other, each while the other
  // half of the step is computed: 32 KiB in flight per CU is where this memory system streams fastest (64 KiB:
  // every large shape 2-3 % slower; a plain read kernel shows the same optimum).  LONG, a workgroup with many
  // blocks: V is asked for only after K's MFMAs and the next K after V's, a little less in flight (16 x 32768
  // keys 303.1 -> 297.2 us, 1 x 32768 keys 25.1 -> 24.8).  With few blocks each goes out as soon as its
  // registers are free (5 x 2999 keys, 4 blocks each: 15.6 -> 14.9 us).
  issue_k(0);
  issue_v(0);
  f32x4_t o[8];
#pragma unroll
  for (int d = 0; d < 8; ++d) o[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.0f;
  char *vl = lds + wave * kDecWaveLds;
  char *kl = lds + (NW + wave) * kDecWaveLds;
  if (FUSED) rotate_frags<T>(qf, tab, is_neox);

  const int iters = lone ? p.iters_each * p.num_splits + p.iters_rest
                         : p.iters_each + (split < p.iters_rest);  // blocks split, split + S, ...
  for (int it = 0; it < iters; ++it) {
    const int kb0 = (it * num_splits + split) * kStepKeys + wave * kDecWaveKeys;
    const int at = fused_pos - kb0;               // FUSED: where in the wave's keys the new row is
    const bool owner = FUSED && at >= 0 && at < kDecWaveKeys;
    u32x4_t kc[2][4];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 8; ++i) lds_write_b128(kl, (4 * i + cg) * kRowBytes + ((col ^ ((4 * i + cg) & 15)) << 4), kn[i]);
    if (owner) {
      // the new token's K row takes its place among the staged rows and goes to the cache
      u32x4_t nk[4] = {qf[0], qf[1], qf[2], qf[3]};
      bool mine = new_col;
      if (rows == kDecCols) {  // no spare column: one more rotation
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) nk[kk] = global_load_b128(new_k_row + cg * 16 + kk * 64);
        load_rotation(tab, freq_row, cg, is_neox);
        rotate_frags<T>(nk, tab, is_neox);
        mine = col == 0;
      }
      if (mine) {
        char *dst = const_cast<char *>(kbase) + (size_t)fused_pos * row_bytes + cg * 16;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          lds_write_b128(kl, at * kRowBytes + (((4 * kk + cg) ^ (at & 15)) << 4), nk[kk]);
          *reinterpret_cast<u32x4_t *>(dst + kk * 64) = nk[kk];
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (!LONG && it > 0) issue_v(it);
    // K fragments (A operand): key blk*16+col, dims 32kk + 8cg .. +7
#pragma unroll
    for (int blk = 0; blk < 2; ++blk)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        kc[blk][kk] = lds_read_b128(kl, (blk * 16 + col) * kRowBytes + (((4 * kk + cg) ^ col) << 4));

    if (kb0 < n) {
      // ---- S^T = K Q^T : 2 blocks of 16 keys ----
      f32x4_t s[2];
#pragma unroll
      for (int blk = 0; blk < 2; ++blk) {
        s[blk] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) s[blk] = E::mfma16(kc[blk][kk], qf[kk], s[blk]);
      }
      if (LONG && it > 0) {
        __builtin_amdgcn_sched_barrier(0);
        issue_v(it);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (kb0 + kDecWaveKeys - 1 > min(offset, n - 1)) {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = kb0 + blk * 16 + 4 * cg + i;
            if (key >= n || key > c_limit) s[blk][i] = -INFINITY;
          }
      }
      float mloc = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                         fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
      mloc = quad_max(mloc);
      const float m_new = fmaxf(m_run, mloc * kScaleLog2e);
      const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
      if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {
        const float alpha = fast_exp2(m_run - m_use);
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < 8; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[d][i] *= alpha;
        m_run = m_new;
      }
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[blk][i] = fast_exp2(__builtin_fmaf(s[blk][i], kScaleLog2e, -m_use));
      // P^T as B operand: slot e<4 -> block 0 key 4cg+e, e>=4 -> block 1 key 4cg+e-4
      u32x4_t pf;
      pf[0] = E::pack2(s[0][0], s[0][1]);
      pf[1] = E::pack2(s[0][2], s[0][3]);
      pf[2] = E::pack2(s[1][0], s[1][1]);
      pf[3] = E::pack2(s[1][2], s[1][3]);
      // the row sum takes the ROUNDED probabilities, the values P.V uses: numerator and
      // denominator then carry the same rounding (as in the prefill kernel)
      float psum = dot2_ones<T>(pf[0], 0.0f);
      psum = dot2_ones<T>(pf[1], psum);
      psum = dot2_ones<T>(pf[2], psum);
      psum = dot2_ones<T>(pf[3], psum);
      l_run += psum;
      // ---- O^T += V^T P^T ----
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 8; ++i) lds_write_b128(vl, v_swizzle32_off(4 * i + cg, col), vn[i]);
      if (owner && cg == (at & 3)) {  // the new token's V row, likewise
        lds_write_b128(vl, v_swizzle32_off(at, col), new_v);
        *reinterpret_cast<u32x4_t *>(const_cast<char *>(vbase) + (size_t)fused_pos * row_bytes + col * 16) = new_v;
      }
      __builtin_amdgcn_wave_barrier();
      if (it + 1 < iters && !LONG) issue_k(it + 1);
      const int vr = 4 * cg + (col >> 2);
      const int sub = (col & 1) * 8;
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const int gran = 2 * d + ((col & 3) >> 1);
        const u32x2_t lo = lds_read_tr16(vl, v_swizzle32_off(vr, gran) + sub);
        const u32x2_t hi = lds_read_tr16(vl, v_swizzle32_off(vr + 16, gran) + sub);
        const u32x4_t vf = {lo[0], lo[1], hi[0], hi[1]};
        o[d] = E::mfma16(vf, pf, o[d]);
      }
      if (it + 1 < iters && LONG) {
        __builtin_amdgcn_sched_barrier(0);
        issue_k(it + 1);
      }
    } else if (it + 1 < iters) {
      issue_k(it + 1);
    }
  }

  // ---- merge the waves ----
  const float l_tot = quad_sum(l_run);
  __syncthreads();
  // [wave][col][128]; the 16-byte pieces of a row are XORed with the column, so that neither the columns of a
  // write nor the pieces of a read meet in one bank
  float *lo_f = reinterpret_cast<float *>(lds);
  float *lml = reinterpret_cast<float *>(lds + NW * kDecWaveLds);    // [wave][col][2] (the K staging space)
#pragma unroll
  for (int d = 0; d < 8; ++d)
    *reinterpret_cast<f32x4_t *>(lo_f + (wave * kDecCols + col) * kHeadDim + (((4 * d + cg) ^ col) << 2)) = o[d];
  if (cg == 0) {
    lml[(wave * kDecCols + col) * 2] = m_run;
    lml[(wave * kDecCols + col) * 2 + 1] = l_tot;
  }
  __syncthreads();

  const size_t pair = (size_t)b * Hkv + kvh;
  const int pair_slots = p.num_splits * cols;
  const __amdgpu_buffer_rsrc_t po = byte_buffer(p.ws_o + pair * pair_slots * kHeadDim, pair_slots * kHeadDim * 4);
  const __amdgpu_buffer_rsrc_t pml = byte_buffer(p.ws_ml + pair * pair_slots * 2, pair_slots * 8);
  const int tagged_bytes = p.num_splits * all_rows * kTaggedBytes;
  const __amdgpu_buffer_rsrc_t pt = byte_buffer(reinterpret_cast<char *>(p.ws_o) + pair * tagged_bytes, tagged_bytes);
  const uint32_t tag0 = (uint32_t)p.fold, tag1 = (uint32_t)(p.fold >> 32);
  auto tagged = [&](float x, float y) {
    return __builtin_bit_cast(f32x4_t, u32x4_t{__builtin_bit_cast(uint32_t, x), tag0, __builtin_bit_cast(uint32_t, y), tag1});
  };
  for (int c = tid >> 4; c < rows; c += 4 * NW) {
    const int dch = tid & 15;  // 8-wide d chunk of column c
    float mw[NW], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = lml[(w * kDecCols + c) * 2];
      M = fmaxf(M, mw[w]);
    }
    const float M_use = (M == -INFINITY) ? 0.0f : M;
    float L = 0.0f, acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float wt = fast_exp2(mw[w] - M_use);
      L += wt * lml[(w * kDecCols + c) * 2 + 1];
      const float *src = lo_f + (w * kDecCols + c) * kHeadDim;
      const f32x4_t s0 = *reinterpret_cast<const f32x4_t *>(src + (((2 * dch) ^ c) << 2));
      const f32x4_t s1 = *reinterpret_cast<const f32x4_t *>(src + (((2 * dch + 1) ^ c) << 2));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[j] += wt * s0[j];
        acc[4 + j] += wt * s1[j];
      }
    }
    if (FOLD == kNoFold ? num_splits == 1 : lone) {
      if (lone && !(lone_rows >> c & 1)) continue;
      const float inv = (L > 0.0f) ? 1.0f / L : 0.0f;
      const int r = (int)(c * row_part >> 16), hq = c - r * g;
      char *op = p.out + (((size_t)token + r) * H + kvh * g + hq) * kRowBytes + dch * 16;
      u32x4_t w;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = E::pack2(acc[2 * j] * inv, acc[2 * j + 1] * inv);
      *reinterpret_cast<u32x4_t *>(op) = w;
      continue;
    }
    const int slot = split * cols + c;
    const f32x4_t a0 = {acc[0], acc[1], acc[2], acc[3]}, a1 = {acc[4], acc[5], acc[6], acc[7]};
    const u32x2_t ml = {__builtin_bit_cast(uint32_t, M), __builtin_bit_cast(uint32_t, L)};
    if constexpr (FOLD == kFoldByTags) {
      const int at = (split * all_rows + c) * kTaggedBytes;
#pragma unroll
      for (int j = 0; j < 4; ++j) store_device(pt, at + j * 256 + dch * 16, tagged(acc[2 * j], acc[2 * j + 1]));
      if (dch == 0) store_device(pt, at + kHeadDim * 8, tagged(M, L));
    } else if constexpr (FOLD == kFoldByFlags) {
      store_device(po, slot * kHeadDim * 4 + dch * 32, a0);
      store_device(po, slot * kHeadDim * 4 + dch * 32 + 16, a1);
      if (dch == 0) store_device(pml, slot * 8, ml);
    } else {
      float *wo = p.ws_o + (pair * pair_slots + slot) * kHeadDim + 8 * dch;
      *reinterpret_cast<f32x4_t *>(wo) = a0;
      *reinterpret_cast<f32x4_t *>(wo + 4) = a1;
      if (dch == 0) *reinterpret_cast<u32x2_t *>(p.ws_ml + (pair * pair_slots + slot) * 2) = ml;
    }
  }
  if constexpr (FOLD != kFoldByFlags) return;

  // ---- fold in the workgroup that finds every partial of its (sequence, kv head) stored ----
  // Each workgroup raises its flag once its partial has reached the point where all XCDs see it, and looks at the
  // others' after that: the last one to raise its flag finds all of them up (if two do, both write the
  // same rows).  A flag is up if it holds this launch's number, whatever the workspace held before; the folding
  // workgroup takes them down for a replay of the same launch.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  unsigned *all_up = reinterpret_cast<unsigned *>(lds);
  const u32x2_t up = {(uint32_t)p.fold, (uint32_t)(p.fold >> 32)};
  if (wave == 0) {
    const int my_flag = (split * cols + cols - 1) * 8;
    if (lane == 0) store_device(pml, my_flag, up);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const u32x2_t f = load_device2(pml, (min(lane, p.num_splits - 1) * cols + cols - 1) * 8);
    const bool down = f[0] != up[0] || f[1] != up[1];
    if (lane == 0) *all_up = 0;
    if (__builtin_amdgcn_ballot_w64(down) == 0 && lane == 0) *all_up = 1;
  }
  __syncthreads();
  if (*all_up == 0) return;
  if (tid < p.num_splits) store_device(pml, (tid * cols + cols - 1) * 8, u32x2_t{0u, 0u});
  // Every partial of a thread's share is asked for before the first is used: up to 8 of a row are a group of 32 threads' each, more of up
  // to 4 rows have a part in each group (NW = 4).
  const int c = tid >> 5, d4 = tid & 31;
  auto ask = [&](int s, int row, u32x2_t &ml, f32x4_t &ov) {
    const int slot = min(s, p.num_splits - 1) * cols + min(row, rows - 1);
    ml = load_device2(pml, slot * 8);
    ov = load_device(po, slot * kHeadDim * 4 + d4 * 16);
  };
  PartialSum sum;
  if (NW == 2 || p.num_splits <= kFoldDepth) {
    u32x2_t ml[kFoldDepth];
    f32x4_t ov[kFoldDepth];
#pragma unroll
    for (int j = 0; j < kFoldDepth; ++j) ask(j, c, ml[j], ov[j]);
    sum.take(ml, ov, p.num_splits);
  } else {
    constexpr int kRows = 4;
    static_assert(NW == 2 || kParts == 2 * NW, "a part per group");
    u32x2_t ml[kRows][2], part_ml[kParts];
    f32x4_t ov[kRows][2], part_o[kParts];
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int j = 0; j < 2; ++j) ask(c + kParts * j, r, ml[r][j], ov[r][j]);
    float *red_ml = reinterpret_cast<float *>(lds) + 16, *red_o = red_ml + 2 * kRows * kParts;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      PartialSum of_part;
      of_part.take(ml[r], ov[r], c + kParts < p.num_splits ? 2 : 1);
      if (d4 == 0) *reinterpret_cast<float2 *>(red_ml + 2 * (r * kParts + c)) = float2{of_part.M, of_part.L};
      *reinterpret_cast<f32x4_t *>(red_o + (r * kParts + c) * kHeadDim + 4 * d4) = of_part.o;
    }
    __syncthreads();
    if (c < rows) {
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        part_ml[i] = *reinterpret_cast<const u32x2_t *>(red_ml + 2 * (c * kParts + i));
        part_o[i] = *reinterpret_cast<const f32x4_t *>(red_o + (c * kParts + i) * kHeadDim + 4 * d4);
      }
      sum.take(part_ml, part_o, kParts);
    }
  }
  if (c < rows) {
    const int r = (int)(c * row_part >> 16);
    const float inv = (sum.L > 0.0f) ? 1.0f / sum.L : 0.0f;
    u32x2_t w;
    w[0] = E::pack2(sum.o[0] * inv, sum.o[1] * inv);
    w[1] = E::pack2(sum.o[2] * inv, sum.o[3] * inv);
    *reinterpret_cast<u32x2_t *>(p.out + (((size_t)token + r) * H + kvh * g + c - r * g) * kRowBytes + d4 * 8) = w;
  }
}

// Folds the splits of one output row (one query row of one head) with the log-sum-exp rule.
// grid (rows, Hkv, batch), 256 threads = 8 groups of 32: group sg takes splits sg, sg+8, ... (four
// dims per thread, all of a thread's loads issued before any is used), then the 8 groups are merged
// through LDS.  With few splits the surplus groups have nothing to load.
constexpr int kMaxSplits = 256;

template <typename T>
__global__ __launch_bounds__(256) void flash_decode_combine_kernel(addresses_t a, u32x4_t size, u32x2_t heads) {
  // a: partials, their maxima and sums, out, tokens; size: splits, columns of a slot, Hkv, m; heads: g, 2^16 / g + 1
  using E = Elem<T>;
  const float *ws_o = at_address<const float>(a[0]), *ws_ml = at_address<const float>(a[1]);
  char *out = at_address<char>(a[2]);
  const int cols = size[1], Hkv = size[2], m = size[3], g = heads[0], H = g * Hkv;
  __shared__ float red_m[8], red_l[8];
  __shared__ f32x4_t red_o[8][32];
  const int c = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  if (c >= ((int)a[3] - b * m) * g) return;  // (past a short last tile)
  const int sg = threadIdx.x >> 5, d4 = threadIdx.x & 31;
  const int S = size[0];
  const size_t base = ((size_t)b * Hkv + kvh) * S;
  const float *ml = ws_ml + (base * cols + c) * 2;
  const float *src = ws_o + (base * cols + c) * kHeadDim + 4 * d4;
  const size_t ml_stride = (size_t)cols * 2, o_stride = (size_t)cols * kHeadDim;
  float M = -INFINITY, L = 0.0f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = sg; s0 < S; s0 += 32) {  // rounds of up to 4 splits per thread
    float mv[4], lv[4];
    f32x4_t ov[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = min(s0 + 8 * j, S - 1);
      mv[j] = ml[s * ml_stride];
      lv[j] = ml[s * ml_stride + 1];
      ov[j] = *reinterpret_cast<const f32x4_t *>(src + s * o_stride);
    }
    float Mn = M;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s0 + 8 * j < S) Mn = fmaxf(Mn, mv[j]);
    const float M_use = (Mn == -INFINITY) ? 0.0f : Mn;
    const float resc = fast_exp2(M - M_use);  // 0 on the first round (M = -inf)
    L *= resc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= resc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float wt = (s0 + 8 * j < S) ? fast_exp2(mv[j] - M_use) : 0.0f;
      L += wt * lv[j];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += wt * ov[j][i];
    }
    M = Mn;
  }
  if (d4 == 0) {
    red_m[sg] = M;
    red_l[sg] = L;
  }
  red_o[sg][d4] = acc;
  __syncthreads();
  if (sg != 0) return;
  float Mt = -INFINITY;
#pragma unroll
  for (int g8 = 0; g8 < 8; ++g8) Mt = fmaxf(Mt, red_m[g8]);
  const float Mt_use = (Mt == -INFINITY) ? 0.0f : Mt;
  float Lt = 0.0f;
  f32x4_t tot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int g8 = 0; g8 < 8; ++g8) {
    const float wt = fast_exp2(red_m[g8] - Mt_use);  // 0 for a group without splits (-inf)
    Lt += wt * red_l[g8];
    const f32x4_t o = red_o[g8][d4];
#pragma unroll
    for (int i = 0; i < 4; ++i) tot[i] += wt * o[i];
  }
  const float inv = (Lt > 0.0f) ? 1.0f / Lt : 0.0f;
  const int r = (int)(c * heads[1] >> 16), hq = c - r * g;  // (c / g, c below 16)
  u32x2_t w;
  w[0] = E::pack2(tot[0] * inv, tot[1] * inv);
  w[1] = E::pack2(tot[2] * inv, tot[3] * inv);
  const size_t token = (unsigned)(b * m);
  *reinterpret_cast<u32x2_t *>(out + ((token + r) * H + kvh * g + hq) * kRowBytes + d4 * 8) = w;
}

// Largest split count the default rule considers for batch * kv heads = pairs (any KV length): one
// round of workgroups, one workgroup per CU of the current device.
int flash_decode_max_default_splits(long long pairs) {
  const long long cus = device_compute_units();
  long long base = (cus + pairs - 1) / pairs;
  if (base < 8) base = 8;
  if (base > kMaxSplits) base = kMaxSplits;
  return (int)base;
}

// Split count that a simple model of the launch makes fastest.  One workgroup to a CU (two: the next model).  While each has a CU of its own, a CU
// streams the more the fewer they are (32 KiB in flight, over a latency that grows with the load); beyond that a CU streams 27.9
// GB/s (all 256 of an MI355X together 7.1 TB/s, what its memory system gives a kernel that only reads) and the launch takes
// something between the rounds that the fullest CU runs and the mean of all.  A fold by folders costs 0.9 us in blocks of 64
// keys, else 2.0 for up to 8 partials, 1.8 for up to 16 and 1.4 beyond (what more of them cost is in the workgroups).  Of counts within 0.5 % of the best one that gives every CU one
// workgroup is taken, else the smallest.  Fitted over 563 shapes of batch 1-16 x 2-32 kv heads x 130-32000 keys and up to 40 counts each: the
// count chosen is 0.25 % slower than the fastest on average, 0.7 % at the 90th percentile, 17 % at most (2 x 188 of 32), where the model before, which
// added whole rounds up and took a fold by folders for a second launch, was 1.2, 4.4 and 18 % (us: 250 keys of 4 kv heads
// 5.47 -> 4.63, 3 x 4200 of 32 38.6 -> 34.2, 11 x 2983 of 8 28.7 -> 25.3, 6 x 4566 of 8 22.6 -> 20.3).
static double split_model_us(long long pairs, int nblocks, int s, int cus, int rows) {
  const long long wgs = pairs * s;
  const int blocks = (nblocks + s - 1) / s;
  constexpr double kBlockKb = 2.0 * kRowBytes * kDecStepKeys * 1e-3;  // K and V rows of one kv head
  double t;
  if (wgs <= cus) {
    t = kBlockKb * blocks / ((blocks >= 8 ? 46.8 : 52.4) - 18.5 * (double)wgs / cus) + 2.63;
  } else {
    const double rounds = 0.41 * (double)((wgs + cus - 1) / cus) + 0.59 * (double)wgs / cus;
    t = rounds * (kBlockKb * (0.46 * blocks + 0.54 * nblocks / s) / 27.9 + 0.93) + 1.44;
  }
  if (s == 1) return t;
  if (s == nblocks && 2 * s <= kFoldDepth && pairs * (s == 2 ? 6 : 2 * s) <= cus && rows < kDecCols / 2) return t + 0.9;
  return t + (s <= kFoldDepth ? 2.0 : s <= 16 ? 1.8 : 1.4);
}
// Two workgroups to a CU, where there are more of them than CUs: what one does not stream while it begins, merges its waves and stores, the other one
// does, and it is that which short rounds lose most to; 64 KiB are in flight then, with which a stream is slower (us, one to a CU / two, each with
// its best count: 10 sequences of 32 kv heads, 300 keys 14.2 / 12.2, 700 25.8 / 21.9, 1024 32.6 / 29.3, 1500 43.0 / 40.5, 3000 78.5 / 76.8; 2 blocks,
// 480 pairs 11.85 / 9.0; but 16 x 1500 of 32 kv heads, two even rounds, 58.2 / 61.6, 16 x 32768 of 8 295 / 325).  A workgroup's number within its XCD's
// share repeats with the split, so that the XCD of the longer ones counts.  Fitted over 1261 shapes of 1-16 sequences, 2-32 kv heads, 64-32768 keys, up to 1.1 GB
// and 17 counts each.  Two are taken where the model has them 4 % ahead, 160 of the shapes: 0.865 of the time there on average, none of all slower
// by 2 %.  Not for one sequence: the fused step's kernels take more than half of a CU's registers, and its unfused equal, which gives the same bits, has the same
// count (fused / unfused, us, count for one / for two: 2000 keys of 100 kv heads 21.1 / 22.1, 20.25 / 20.35, 3072 of 66 21.05 / 22.15, 20.2 / 19.3; but 2000
// of 88 22.8 / 20.75, 21.6 / 18.65; below 65 kv heads the counts are the same).
static double two_model_us(long long pairs, int nblocks, int s, int cus) {
  const long long wgs = pairs * s;
  if (wgs <= cus || (s > 1 && nblocks < 2 * s)) return 1e30;  // (one block each: the fold is the larger part)
  constexpr double kBlockKb = 2.0 * kRowBytes * kDecStepKeys * 1e-3;
  const int classes = s % 8 == 0 ? 8 : s % 4 == 0 ? 4 : s % 2 == 0 ? 2 : 1;  // of splits, an XCD's each
  const double mean = nblocks / s + (double)((nblocks % s + classes - 1) / classes * classes) / s;
  const double rounds = 0.28 * 2 * (double)((wgs + 2 * cus - 1) / (2 * cus)) + 0.72 * (double)wgs / cus;
  return rounds * kBlockKb * (0.05 * ((nblocks + s - 1) / s) + 0.95 * mean) / 27.1 + 1.92 + (s > 1 ? 2.46 : 0.0);
}
constexpr double kTwoMargin = 0.96;
// The smallest count within `tolerance` of the best, or one that fills up to full_rounds rounds exactly.
template <typename Model>
static int best_splits(long long pairs, int smax, int cus, double tolerance, long long full_rounds, Model model) {
  double t_min = model(1);
  for (int s = 2; s <= smax; ++s) {
    const double t = model(s);
    if (t < t_min) t_min = t;
  }
  int first = 0;
  for (int s = 1; s <= smax; ++s) {
    if (model(s) > t_min * tolerance) continue;
    if (first == 0) first = s;
    if ((pairs * s) % cus == 0 && pairs * s / cus <= full_rounds) return s;
  }
  return first;
}
static int default_splits_model(long long pairs, int nblocks, int cus, int most, int rows, bool may_two) {
  int smax = flash_decode_max_default_splits(pairs);
  if (smax > nblocks) smax = nblocks;
  if (smax > most) smax = most;
  const int one = best_splits(pairs, smax, cus, 1.005, 1, [&](int s) { return split_model_us(pairs, nblocks, s, cus, rows); });
  double least = kTwoMargin * split_model_us(pairs, nblocks, one, cus, rows);
  int best = one;
  for (int s = 1; may_two && s <= smax; ++s) {
    const double t = two_model_us(pairs, nblocks, s, cus);
    if (t < least) {
      least = t;
      best = s;
    }
  }
  return best;
}
static bool two_to_a_cu(int batch, long long pairs, int nblocks, int s, int cus, int rows) {
  return batch > 1 && two_model_us(pairs, nblocks, s, cus) < kTwoMargin * split_model_us(pairs, nblocks, s, cus, rows);
}

// The model is evaluated a few hundred times per call; a decode loop asks for the same (pairs, key
// blocks) at every layer and for the next block count only every 128 tokens, so the last answers are
// kept per thread.
int flash_decode_default_splits(int batch, int n, int kv_head_num, int rows) {
  rows = rows < kDecCols / 2 ? 1 : kDecCols;  // (what the model tells apart)
  const long long pairs = (long long)batch * kv_head_num;
  const int nblocks = (n + kDecStepKeys - 1) / kDecStepKeys;
  const int cus = device_compute_units();
  struct Memo {
    long long pairs;
    int nblocks, cus, splits;
    int rows;
    bool one;  // sequence
  };
  constexpr int kMemo = 8;
  static thread_local Memo memo[kMemo] = {};
  static thread_local unsigned next = 0;
  for (const Memo &e : memo)
    if (e.splits > 0 && e.pairs == pairs && e.nblocks == nblocks && e.cus == cus && e.rows == rows && e.one == (batch == 1)) return e.splits;
  const int s = default_splits_model(pairs, nblocks, cus, kMaxSplits, rows, batch > 1);
  memo[next++ % kMemo] = Memo{pairs, nblocks, cus, s, rows, batch == 1};
  return s;
}

int flash_decode_splits_within(int batch, int n, int kv_head_num, int rows, size_t bytes) {
  const int s = flash_decode_default_splits(batch, n, kv_head_num, rows);
  if (flash_decode_workspace_bytes(batch, 1, 1, kv_head_num, s) <= bytes) return s;
  int fits = s - 1;
  while (fits > 1 && flash_decode_workspace_bytes(batch, 1, 1, kv_head_num, fits) > bytes) --fits;
  return default_splits_model((long long)batch * kv_head_num, (n + kDecStepKeys - 1) / kDecStepKeys,
                              device_compute_units(), fits, rows, batch > 1);
}

// What a call may insist on is counted with coarser figures than the default: 27.7 GB/s per CU in a full round and at most
// 32 in a thin one, 3 us per workgroup, 5 for a fold.  Callers were promised that calls which are not worth a split by
// these need no room; the promise does not move with the model above.  Nor does it move for callers whose workspace was sized by the default
// count of a model before (whole rounds, folds of 1.2 to 2.6 us, or one workgroup to a CU only): the smallest of the three is enough (3 x 3584 keys of 8
// kv heads: 10 of the second, 7 of the first, 10 by the coarser figures).
size_t flash_decode_least_workspace_bytes(int batch, int n, int kv_head_num) {
  const long long pairs = (long long)batch * kv_head_num;
  const int nblocks = (n + kDecStepKeys - 1) / kDecStepKeys, cus = device_compute_units();
  int smax = flash_decode_max_default_splits(pairs);
  if (smax > nblocks) smax = nblocks;
  auto kb_of = [&](int splits) { return 2.0 * kRowBytes * kDecStepKeys * ((nblocks + splits - 1) / splits) * 1e-3; };
  const int coarse = best_splits(pairs, smax, cus, 1.03, pairs * smax, [&](int splits) {
    const long long full = pairs * splits / cus, rest = pairs * splits % cus;
    const double kb = kb_of(splits);
    double t = full * (kb / 27.7 + 3.0);
    if (rest > 0) {
      const double rate = 27.7 * cus / (double)rest;
      t += kb / (rate > 32.0 ? 32.0 : rate) + 3.0;
    }
    return splits > 1 ? t + 5.0 : t;
  });
  const int before = best_splits(pairs, smax, cus, 1.03, pairs * smax, [&](int splits) {
    const long long full = pairs * splits / cus, rest = pairs * splits % cus;
    double t = full * (kb_of(splits) / 27.9 + 2.7);
    if (rest > 0) t += kb_of(splits) / (((nblocks + splits - 1) / splits >= 8 ? 47.5 : 49.0) - 18.5 * (double)rest / cus) + 3.05;
    if (splits == 1) return t;
    if (splits == nblocks && 2 * splits <= kFoldDepth && 2 * pairs * splits <= cus) return t + 1.2;
    return t + (splits <= kFoldDepth ? 2.0 : splits <= 16 ? 2.6 : 2.1);
  });
  int least = default_splits_model(pairs, nblocks, cus, kMaxSplits, 1, false);
  for (const int s : {default_splits_model(pairs, nblocks, cus, kMaxSplits, kDecCols, false), coarse, before})
    if (s < least) least = s;
  return flash_decode_workspace_bytes(batch, 1, 1, kv_head_num, least);
}

int flash_decode_effective_splits(int num_splits, int n) {
  const int nblocks = (n + kDecStepKeys - 1) / kDecStepKeys;
  if (num_splits > nblocks) num_splits = nblocks;  // every split holds at least one block
  return num_splits < 1 ? 1 : num_splits;
}

size_t flash_decode_workspace_bytes(int batch, int m, int group_size, int kv_head_num,
                                    int num_splits) {
  (void)m;
  (void)group_size;
  if (num_splits <= 1) return 0;
  const size_t slots = (size_t)batch * kv_head_num * num_splits * kDecCols;
  return slots * (kHeadDim + 2) * sizeof(float);
}

// A number that no workspace holds: of a launch, see launch_number.hpp.  (By chance 2^-64, from a random start.)
uint64_t launch_number() {
  static std::atomic<uint64_t> last{[] {
    std::random_device rd;
    return ((uint64_t)rd() << 32) ^ rd() ^ (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count();
  }()};
  uint64_t before = last.load(std::memory_order_relaxed), n;
  do n = llmhip::next_launch_number(before);
  while (!last.compare_exchange_weak(before, n, std::memory_order_relaxed));
  return n;
}

bool may_be_capturing(hipStream_t stream) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) == hipSuccess) return cap != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;
}

template <typename T, bool FUSED, int NW, bool LONG, FoldMode FOLD>
static hipError_t launch_decode_t(const DecodeParams &p, hipStream_t stream) {
  // kDecLdsPad bytes of dynamic LDS that nobody touches keep a second workgroup off the CU where it is not wanted (two of
  // them put 64 KiB of loads in flight again, see two_model_us).  More than 64 KiB of LDS in total is an opt-in
  // per device and kernel.
  const int pad = NW == 4 && !p.two ? kDecLdsPad : 0;
  const auto kern = flash_decode_kernel<T, FUSED, NW, LONG, FOLD>;
  if (pad) {
    static std::atomic<uint64_t> attr_done{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(attr_done.load(std::memory_order_acquire) & bit)) {
      e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, pad);
      if (e != hipSuccess) return e;
      attr_done.fetch_or(bit, std::memory_order_release);
    }
  }
  const DecodeEarly early(p);
  dim3 grid(p.num_splits, p.Hkv, p.batch);
  if (FOLD == kFoldByTags) {
    const int pairs = p.batch * p.Hkv;
    grid = dim3(p.num_splits, pairs + (pairs * p.folders + p.num_splits - 1) / p.num_splits);
  }
  const hipError_t e = launch(kern, grid, 64 * NW, pad, stream, early.a, early.b, early.c, static_cast<const DecodeLate &>(p));
  if (e != hipSuccess || p.num_splits == 1 || FOLD != kNoFold) return e;
  return launch(flash_decode_combine_kernel<T>, dim3(p.rows, p.Hkv, p.batch), 256, 0, stream,
                addresses_t{address(p.ws_o), address(p.ws_ml), address(p.out), (uint64_t)p.tokens},
                u32x4_t{(uint32_t)p.num_splits, (uint32_t)p.cols, (uint32_t)p.Hkv, (uint32_t)p.m},
                u32x2_t{(uint32_t)p.g, 65536u / p.g + 1});
}

template <typename T, bool FUSED, FoldMode FOLD>
static hipError_t launch_decode_f(const DecodeParams &p, bool half, bool many, hipStream_t stream) {
  if (half) return launch_decode_t<T, FUSED, 2, false, FOLD>(p, stream);
  if (many) return launch_decode_t<T, FUSED, 4, true, FOLD>(p, stream);
  return launch_decode_t<T, FUSED, 4, false, FOLD>(p, stream);
}
template <typename T, bool FUSED>
static hipError_t launch_decode(const DecodeParams &p, FoldMode how, bool half, bool many, hipStream_t stream) {
  if (how == kFoldByTags) return launch_decode_f<T, FUSED, kFoldByTags>(p, half, many, stream);
  return how == kFoldByFlags ? launch_decode_f<T, FUSED, kFoldByFlags>(p, half, many, stream)
                             : launch_decode_f<T, FUSED, kNoFold>(p, half, many, stream);
}

static hipError_t launch_decode_impl(DecodeParams &p, void *workspace, size_t workspace_bytes, int num_splits, int dt, bool fused,
                                     hipStream_t stream) {
  p.num_splits = flash_decode_effective_splits(num_splits, p.n);
  p.cols = kDecCols;
  int nblocks = (p.n + kDecStepKeys - 1) / kDecStepKeys;
  // Short caches: where every workgroup has one block of 128 keys and twice as many workgroups still fit the chip at
  // once, blocks of 64 keys and workgroups of two waves.  Their slots have half the columns, so the
  // partials take no more room (one column is the flag's: up to 7 query rows).  More than 8 such blocks, with some CUs left to
  // the folders, for one token of one sequence only: in the fused step each wave of a CU takes in the query and the table beside its keys (us,
  // blocks of 128 / 64: 700 keys of 4 kv heads 5.88 / 5.6, 1500 6.28 / 5.83, 1500 of 2 5.95 / 5.54, 1200 of 8 6.21 / 5.91; but unfused 2 x 900
  // of 4 5.33 / 5.69, and without CUs for the folders 2000 of 8 6.45 / 6.57), and the unfused call gives the same bits.  They need the room that
  // folders take: in an exact workspace 5 to 7 rows keep blocks of 128, which folders fit (unfused, 28 + 4 heads, blocks of 64 by flags
  // or a second launch / so: 1000 keys 8.5 / 5.0, 1030 5.86 / 5.39).
  const int half_blocks = (p.n + kDecStepKeys / 2 - 1) / (kDecStepKeys / 2), cus = device_compute_units();
  const long long pairs = (long long)p.batch * p.Hkv, half_wgs = pairs * half_blocks;
  auto tags_fit = [&](int splits) { return pairs <= kTaggedPairs && (size_t)pairs * splits * p.rows * kTaggedBytes <= workspace_bytes; };
  const bool half = p.num_splits > 1 && p.num_splits == nblocks && p.rows < kDecCols / 2 &&
                    (half_blocks <= kFoldDepth ? half_wgs <= cus
                                               : p.batch == 1 && p.m == 1 && half_blocks <= 32 && half_wgs <= cus - cus / 16 &&
                                                     tags_fit(half_blocks));
  if (half) {
    p.num_splits = nblocks = half_blocks;
    p.cols = kDecCols / 2;
  }
  p.iters_each = nblocks / p.num_splits;
  p.iters_rest = nblocks % p.num_splits;
  // Without folders, few partials of few rows are folded by the workgroup that finds them all stored.  It takes in every one of them, and that is what
  // more of either wait for (captured calls, us, flags / a second launch, which a graph brings at no cost to the host: the fused step, 1000 keys of 28 +
  // 4 heads, 16 partials of 7 rows, 9.3 / 6.6, 2048 of 40 + 8, 16 of 5, 9.0 / 7.4, 153 of 28 + 4, 4 of 7, 6.9 / 6.4; 522 of 30 + 2, 5 of 15,
  // 7.48 / 7.06; but 474 of 32 + 32, 8 of one, 6.24 / 6.57, 496 of 16 + 2, 4 of 8, 6.57 / 6.75, 3 tokens past 3021 of 16 + 16, 16 of 3, 8.68 / 9.18).
  const int few_rows = p.num_splits <= kFoldDepth ? (half ? 4 : 8) : p.num_splits <= 16 && !half ? 4 : 0;
  FoldMode how = p.num_splits > 1 && p.rows <= few_rows ? kFoldByFlags : kNoFold;
  p.fold = how != kNoFold ? launch_number() : 0;
  // Up to 128 partials by folders (more than 8 rows where the room is larger than a call may insist on: with tags they take more, and a full round of
  // 256 workgroups with 16 rows more than a stream's first 4 MiB of scratch: 32 kv heads fold by a second launch until a call has made it grow), as many of them as
  // the CUs that the other workgroups leave idle can take, down to one row each.
  // A replayed graph launches with the number of its capture, and words of the replay before would pass for new ones.
  if (p.num_splits > 1 && p.num_splits <= kMaxTaggedSplits && tags_fit(p.num_splits) && !may_be_capturing(stream)) {
    how = kFoldByTags;
    if (p.fold == 0) p.fold = launch_number();
    const long long idle = device_compute_units() - pairs * p.num_splits;
    p.fold_rows = p.num_splits > 16 ? 1 : half || (p.num_splits > kFoldDepth && p.rows <= 8) ? 2 : 4;
    while (p.fold_rows > 1 && pairs * ((2 * p.rows + p.fold_rows - 1) / p.fold_rows) <= idle) p.fold_rows /= 2;
    p.folders = (p.rows + p.fold_rows - 1) / p.fold_rows;
    p.folders_div = make_fast_div((uint32_t)p.folders);
    p.fold_rows |= fold_looks((p.n + kDecStepKeys - 1) / kDecStepKeys) << 8;
  }
  const size_t slots = (size_t)p.batch * p.Hkv * p.num_splits * p.cols;
  p.ws_o = static_cast<float *>(workspace);
  p.ws_ml = p.ws_o ? p.ws_o + slots * kHeadDim : nullptr;
  p.two = !half && two_to_a_cu(p.batch, pairs, nblocks, p.num_splits, cus, p.rows);
  const bool many = p.iters_each >= 8;  // long enough to be bound by the stream, see the kernel
  if (dt == kDtFloat16)
    return fused ? launch_decode<_Float16, true>(p, how, half, many, stream) : launch_decode<_Float16, false>(p, how, half, many, stream);
  return fused ? launch_decode<__bf16, true>(p, how, half, many, stream) : launch_decode<__bf16, false>(p, how, half, many, stream);
}

hipError_t launch_flash_decode(void *out, const void *q, const void *k, const void *v,
                               void *workspace, size_t workspace_bytes, int batch, int m, int n, int offset,
                               int64_t kv_seq_stride, int group_size, int kv_head_num,
                               int num_splits, int dt, hipStream_t stream) {
  DecodeParams p = {};
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = static_cast<char *>(out);
  p.batch = batch;
  p.m = m;
  p.n = n;
  p.offset = offset;
  p.kv_seq_stride = kv_seq_stride;
  p.tokens = batch * m;
  p.g = group_size;
  p.Hkv = kv_head_num;
  p.rows = m * group_size;
  return launch_decode_impl(p, workspace, workspace_bytes, num_splits, dt, false, stream);
}

int flash_decode_tiles(int m, int group_size) {
  const int most = kDecCols / group_size;
  return (m + most - 1) / most;
}

// Tiles read their keys each for itself, so that it is the short calls that they are for, those that wait for one workgroup's chain and
// the fold: up to 40000 keys of all tiles and kv heads, and from where a chunk's workgroups of all keys take longer (lines measured with 256
// compute units; attention, us, key ranges and a combine launch / tiles: 3 tokens past 1000 keys of 28 + 4 heads 8.13 / 5.89, 8 past 2000 8.62 / 7.75, 6 past 1000 of 12 + 2
// 7.95 / 5.60, 4 past 4000 8.17 / 7.04, 6 past 2000 of 40 + 8 8.69 / 7.84; but 6 past 4000 of 28 + 4 8.92 / 9.50 (49000), 12 past 500 of 40 +
// 8 6.43 / 6.80, and of 32 heads of one kv head each 32 past 500 7.2 / 8.35).
bool flash_decode_takes_tiles(int m, int n_vis, int group_size, int kv_head_num) {
  if (group_size < 2 || group_size > kDecCols || m > 8 * kDecCols || prefill_is_prompt(m, n_vis)) return false;
  const int tiles = flash_decode_tiles(m, group_size);
  const long long pairs = (long long)tiles * kv_head_num;
  return tiles <= 8 && pairs * n_vis <= 40000 && n_vis >= 33 * (pairs - 8);
}

hipError_t launch_flash_decode_tiles(void *out, const void *q, const void *k, const void *v, void *workspace, size_t workspace_bytes,
                                     int m, int n, int offset, int group_size, int kv_head_num, int num_splits, int dt,
                                     hipStream_t stream) {
  DecodeParams p = {};
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = static_cast<char *>(out);
  p.batch = flash_decode_tiles(m, group_size);
  p.m = (m + p.batch - 1) / p.batch;
  p.tokens = m;
  p.n = n;
  p.offset = offset;
  p.g = group_size;
  p.Hkv = kv_head_num;
  p.rows = p.m * group_size;
  return launch_decode_impl(p, workspace, workspace_bytes, num_splits, dt, false, stream);
}

// One decode step of one sequence with the rotary embedding and the cache append inside the decode
// kernel: rows [0, pos) of the caches are read, row pos is produced from in_k / in_v and written.
hipError_t launch_flash_decode_step(void *out, void *k_cache, void *v_cache, const void *freq_cis,
                                    const void *in_q, const void *in_k, const void *in_v, void *workspace,
                                    size_t workspace_bytes, int pos, int group_size, int kv_head_num, int is_neox, int num_splits,
                                    int dt, hipStream_t stream) {
  DecodeParams p = {};
  p.q = in_q;
  p.k = k_cache;
  p.v = v_cache;
  p.out = static_cast<char *>(out);
  p.batch = 1;
  p.m = 1;
  p.tokens = 1;
  p.n = pos + 1;
  p.offset = pos;
  p.kv_seq_stride = pos + 1;
  p.g = group_size;
  p.Hkv = kv_head_num;
  p.rows = group_size;
  p.new_k = in_k;
  p.new_v = in_v;
  p.freq_row = static_cast<const float *>(freq_cis) + (size_t)pos * kHeadDim;
  p.fused = true;
  p.is_neox = is_neox ? 1 : 0;
  return launch_decode_impl(p, workspace, workspace_bytes, num_splits, dt, true, stream);
}

#ifndef LLMHIP_BENCH
// ---------------------------------------------------------------------------
// Decode without any allocation: the split-KV partials live in a fixed array in device memory
// that is part of the library's code object (every GPU the library runs on holds its own copy
// until the process ends).  In host code the array's name is only a handle for
// hipGetSymbolAddress: the device address is looked up once per device and that pointer is what
// the kernels receive, exactly as they receive the caller's workspace in launch_flash_decode.
// Nothing in the buffer has to start at zero: every (sequence, kv head, split) slot that the
// combine kernel reads is written by the decode kernel of the same call.  All calls on one GPU
// share the array, so calls that overlap on one GPU (different streams) race.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[kStaticDecodeScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void *> g_scratch_ptr[kMaxDevices];
}  // namespace

hipError_t launch_flash_decode_static(void *out, const void *q, const void *k, const void *v,
                                      int batch, int n, int64_t kv_seq_stride, int group_size,
                                      int kv_head_num, int num_splits, int dt, hipStream_t stream) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  void *ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!ptr) {
    // first call on this device (which is current): each GPU has the array at its own address
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!ptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  }
  return launch_flash_decode(out, q, k, v, ptr, kStaticDecodeScratchBytes, batch, 1, n, n - 1, kv_seq_stride, group_size,
                             kv_head_num, num_splits, dt, stream);
}
#endif  // !LLMHIP_BENCH

}  // namespace LLMHIP_NS
