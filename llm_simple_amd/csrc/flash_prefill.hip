// Causal flash-attention prefill for gfx950 (MI355X).
//
// Computes what the reference's npu_flash_attn_layer / npu_flash_attn_gqa_layer
// compute (prebuild/npu_ops.h:6-18): out[m][H*128] = softmax(scale q k^T +
// mask) v, key c masked for query r iff c > r + offset
// (src/llama2_layer_cpu.cpp:687-701), scale = 1/sqrt(128) inside
// (src/llama2_layer_cpu.cpp:177), query head h reading kv head h / group_size.
//
// Common to all workgroup shapes.  A wave owns 32 query rows.  The scores are
// produced transposed, S^T = K Q^T, with mfma_f32_32x32x16: every lane then
// holds 16 keys of ONE query column per 32-key block, so the softmax row
// reductions are in-register plus one exchange with lane^32
// (v_permlane32_swap).  The probabilities, rounded to the storage type, are
// already laid out as the B operand of O^T += V^T P^T (the contraction index is
// permuted consistently on the V side), so P never touches LDS.  K and V tiles
// of 64 keys are staged in LDS, XOR-swizzled 256-byte rows; K fragments are
// read with ds_read_b128, V^T fragments with ds_read_b64_tr_b16.  exp2 with the
// scale folded into one FMA; the reference maximum is kept in raw score units and
// moves lazily, so O is rarely rescaled.  Accumulation is fp32; out =
// O / l rounded once; l sums the ROUNDED probabilities (what P.V used).
//
// flash_prefill_kernel<T, NW, KP, NT, KEYS>: NW waves share the K/V tiles of 32*NW/KP query rows, KP of them every
// row block, each on its own 32 keys of every tile (KP = 1: on all 64).  While the chip is not full a launch
// waits for the serial chain of the waves with the most keys -- a step of a wave takes 1600-1900 cycles
// where its MFMAs take 512, and nothing else runs on its SIMD -- so that short prompts and chunks want many waves per
// row (KP = 4: 512 tokens, 28 heads 11.5 -> 9.2 us; 256 tokens, 32 heads 8.7 -> 6.7), long ones the
// cheapest step (KP = 1, 256 rows).  NT: the tile loads are non-temporal (chunks whose K/V tiles only one
// workgroup reads).  KEYS: all of them, the key range cut (rows may be packed), or the keys of the longest rows of a prompt in halves.
// Outside the loop a workgroup costs a short launch 2-3 us: indexes come from divisions prepared by the host, Q
// of shared rows is fetched once through LDS, and waves that shared rows trade pieces of O^T so that each
// folds and stores its part (epilogue of a pair 3900 -> 2200 cycles).
// Tiles travel global -> LDS without VGPR staging (buffer_load_dwordx4 ... lds), spread over the MFMA
// stream in the 8-wave kernels, issued beside the first MFMAs of a phase in the others.  The loop is
// software pipelined inside a wave: the MFMAs of S(j+1) are issued beside the
// softmax of tile j (the first ones beside the row-maximum chain, the rest, together with the
// MFMAs of P(j).V(j), beside the exponentials), so K is fetched one tile ahead of V.
// Every LDS fragment address is a loop-invariant register plus an immediate, and a
// tile load is a descriptor that walks through the cache plus a loop-invariant lane offset: the loop spends its
// vector ALU instructions on the softmax only.  That counts for more than their order: a full chip runs this loop at
// 1.6 GHz, what its power allows, and the waves of short prompts issue one instruction in 4-5 cycles.  Clamps
// and 64-bit address sums of the tile loads, a register for M0 per load, the additive term of the exponent and the
// line for its move in every tile, an addition of 0 to every V address: without these 40 of 300 instructions of a
// step (rope not counted, us) 256 tokens of 32 heads 6.6 -> 6.15, 1019 of 28 17.7 -> 16.9, 2048 40.2 -> 39.0, 4096 121.8 ->
// 118.6, 8192 445 -> 434, 200 past 16001 59.0 -> 56.7.  (The same step written out in slots of one MFMA with every
// fragment read four slots ahead of its use is not faster: 4096 tokens 115.9 / 115.7, 8192 420 / 418; nor are sums by
// shifts and additions in place of the dot instructions, which an MFMA cannot overlap: 116.2 / 119.3.)
//
// A chunk of few query rows over a long cache (chunked prefill) has its key range split over
// workgroups: each leaves an fp32 partial (reference maximum, sum, unnormalised O) and
// prefill_combine_kernel (or, for few rows and many ranges, prefill_combine_wide_kernel) folds
// them; the query heads of a kv head can share the rows of a tile.  plan_prefill decides all of this from the
// shape and the device's CU count.
#include <atomic>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace LLMHIP_NS {

constexpr int kTileN = 64;                      // keys per LDS tile (128 where four waves share the rows)
constexpr int kTileBytes = kTileN * kRowBytes;  // 16 KiB
constexpr float kLazyLog2 = 8.0f;                // rescale threshold, log2 units
constexpr int kMaxPrefillSplits = 128;           // key ranges per call
constexpr int kWholeRange = 0x7fffffc0;          // keys of a range without an end
constexpr int kFewRows = 64;                     // rows up to which partials are stored straight from registers

// Keys of a workgroup: all that its rows see; a range of them, its partial to be folded by a launch of its own; all, but a half where
// two workgroups have the longest rows (see pass_half)
enum PrefillKeys { kAllKeys, kRanges, kHalves };

// What a launch is told beyond what its first loads need (PrefillEarly): fetched while those are under way -- except with SPLIT, where
// the key range (num_splits and what stands behind it) is needed for the first address and waited for.
struct PrefillLate {
  char *out;
  // Key-range split (chunked prefill: few query rows over a long cache).  Split s of S covers the key tiles s * first_each,
  // then every following one, up to range_keys keys of them, or, if range_keys is kWholeRange, every S-th (see launch_prefill_t); with more
  // than one split every workgroup leaves an fp32 partial (reference maximum, sum, unnormalised O) that prefill_combine_kernel folds.
  float *ws_o;            // [split][m][H][128], then maxima and sums [split][m][H][2]
  int num_splits, first_each, range_keys;
  // Packed rows whose tiles are dealt to XCDs in clusters: items of an XCD's piece of the list (else 0), tiles of a cluster and, 8 bits on, of
  // the last one, 2^16 over either (rounded up)
  int per_xcd;
  uint32_t tiles, each_part, last_part;
  FastDiv splits_div, per_list;  // items per key range of an XCD's work list, or per cluster of all key ranges and kv heads
#ifdef LLMHIP_BENCH
  // measurement library only: workgroup 0 stores {shader-clock ticks, 100 MHz ticks} of its lifetime
  unsigned long long *clock_probe;
#endif
};
#ifndef LLMHIP_BENCH
static_assert(sizeof(PrefillLate) <= 72, "with what stands before it two lines of 64 bytes (common.hpp)");
#endif
// What an unsplit launch is told of it.
struct PrefillBrief {
  char *out;
#ifdef LLMHIP_BENCH
  unsigned long long *clock_probe;
#endif
  __host__ __device__ operator PrefillLate() const {
    PrefillLate p = {};
    p.out = out;
#ifdef LLMHIP_BENCH
    p.clock_probe = clock_probe;
#endif
    return p;
  }
};
struct PrefillHalves : PrefillBrief {
  char *halves;     // of a pair of workgroups a half's O, maxima and sums, words with tags (kHalfBytes), and behind all of them a word each
  uint64_t number;  // of the launch
  int pairs;
};
struct PrefillParams : PrefillLate {
  const void *q, *k, *v;
  int m, n, offset;
  int H, Hkv, g;
  int xcd_bits, sched_shift;  // workgroups dealt to XCDs: 3 bits, and the logarithm of the XCDs per kv head; else 0
  int second, second_end;    // places of a list (of the XCD, mode 0: of the launch) that are taken in reverse
  int cut, cut_at;           // query tiles of a head, from the last on, whose keys two workgroups share, and how many others come before them
  char *halves;
  uint64_t number;
  FastDiv list_heads;        // heads of an XCD's work list
  FastDiv g_div;
  // Split mode only: the rows of a tile are (token, head-in-group) pairs of ONE kv head, packed
  // token-major (row index = token * g + head % g), so a chunk shorter than a tile reads K and V of
  // its kv head once for all g query heads.
  int pack;
  int chunk;  // keys of a range: a multiple of 128
};
// What the index arithmetic and the first loads of a workgroup need (of an unsplit one: see PrefillLate), packed into the first 14
// words of a kernel's arguments, which are in registers when it starts.  With kernels of their own for key ranges, whose packed rows and partials a prompt need not step
// over (both together, attention alone, us: 32 tokens of 32 heads 4.65 -> 4.21, 256 5.85 -> 5.50, 512 of 28 8.44 -> 7.94, 1019 14.4 ->
// 14.05, 2048 35.6 -> 34.8, 4096 113.5 -> 112.8; 200 past 16001 53.1 -> 51.75, 100 past 8000 of 40 25.2 -> 24.1).  It counts
// instructions: one wave issues one in 4-5 cycles, so the lists' forms are one formula, divisions have no branch, tiles are counted by
// shifts and what a load needs of the last tile is kept (230 instead of 290 of them to the first K line: 32 tokens 4.22 -> 4.00, 256
// 5.50 -> 5.32, 512 of 28 7.93 -> 7.80; 20 past 600 7.24 -> 7.07).
struct PrefillEarly {
  addresses_t a;  // q, K, V, m | n << 32
  u32x4_t b;      // offset, Hkv | g << 16, flags, second | second_end << 16
  u32x2_t c;      // factors of the divisions by g and by the heads of a list
  // flags: xcd_bits, sched_shift << 2, pack << 4, shifts of the divisions << 5 and << 10, heads of a list << 16; with halves the places
  // are second | second_end << 10 | cut << 20 | cut_at << 26
  explicit PrefillEarly(const PrefillParams &p) {
    a = addresses_t{address(p.q), address(p.k), address(p.v), (uint32_t)p.m | (uint64_t)p.n << 32};
    b = u32x4_t{(uint32_t)p.offset, (uint32_t)p.Hkv | (uint32_t)p.g << 16,
                (uint32_t)(p.xcd_bits | p.sched_shift << 2 | p.pack << 4) | p.g_div.l << 5 | p.list_heads.l << 10 | p.list_heads.d << 16,
                p.cut ? (uint32_t)p.second | (uint32_t)p.second_end << 10 | (uint32_t)p.cut << 20 | (uint32_t)p.cut_at << 26
                      : (uint32_t)p.second | (uint32_t)p.second_end << 16};
    c = u32x2_t{p.g_div.m, p.list_heads.m};
  }
};
struct PrefillShared {  // the same, unpacked
  const char *q, *k, *v;
  int m, n, offset, H, Hkv, g, xcd_bits, sched_shift, second, second_end, cut, cut_at;
  bool pack;
  FastDiv g_div, list_heads;
  __device__ __forceinline__ PrefillShared(addresses_t a, u32x4_t b, u32x2_t c, bool halves)
      : q(at_address<const char>(a[0])), k(at_address<const char>(a[1])), v(at_address<const char>(a[2])), m((uint32_t)a[3]),
        n((uint32_t)(a[3] >> 32)), offset(b[0]), H((b[1] & 0xffffu) * (b[1] >> 16)), Hkv(b[1] & 0xffffu), g(b[1] >> 16),
        xcd_bits(b[2] & 3u), sched_shift(b[2] >> 2 & 3u), second(b[3] & (halves ? 0x3ffu : 0xffffu)),
        second_end(halves ? b[3] >> 10 & 0x3ffu : b[3] >> 16), cut(b[3] >> 20 & 63u), cut_at(b[3] >> 26), pack(b[2] & 16u),
        g_div{b[1] >> 16, c[0], b[2] >> 5 & 31u}, list_heads{b[2] >> 16, c[1], b[2] >> 10 & 31u} {}
};

// blockIdx -> (query tile, head, key range).  Workgroup ids are dealt round-robin to the 8
// XCDs by the hardware; heads that share a kv head are kept on the same XCD(s)
// so that its K/V stay in that XCD's L2, and within an XCD the heaviest (last)
// query tiles are issued first.  Key ranges (split mode) are the slowest index of an XCD's
// list, so that every XCD gets the same number of workgroups whatever the head count.
template <PrefillKeys KEYS>
__device__ __forceinline__ bool prefill_schedule(const PrefillShared &e, const PrefillLate &p, int bid, int num_q_tiles, int &tile,
                                                 int &head, int &split) {
  constexpr bool SPLIT = KEYS == kRanges;
  if (SPLIT && p.per_xcd) {
    // (cluster of tiles, kv head, key range, tile of the cluster): an XCD has a piece of the list
    const int i = bid >> 3, idx = (bid & 7) * p.per_xcd + i;
    if (i >= p.per_xcd || idx >= num_q_tiles * e.Hkv * p.num_splits) return false;
    const int each = p.tiles & 0xffu, cluster = (int)fast_div(idx, p.per_list), rem = idx - cluster * (int)p.per_list.d;
    const int first = cluster * each, whole = num_q_tiles - first >= each, size = whole ? each : (int)(p.tiles >> 8);
    const int group = (int)((uint32_t)rem * (whole ? p.each_part : p.last_part) >> 16), h = (int)fast_div(group, p.splits_div);
    split = group - h * p.num_splits;
    tile = num_q_tiles - 1 - first - (rem - group * size);
    head = h * e.g;  // first query head of the kv head
    return true;
  }
  int idx = bid >> e.xcd_bits, xcd = bid & ((1 << e.xcd_bits) - 1);
  if (idx >= e.second && idx < e.second_end) idx = e.second + e.second_end - 1 - idx;
  idx = (idx << e.sched_shift) + (xcd & ((1 << e.sched_shift) - 1));  // 2^sched_shift XCDs per kv head (one: of several heads)
  xcd >>= e.sched_shift;
  // idx: (key range, tile from the last, head among the list's `list_heads`)
  int rem = idx;
  split = 0;
  if (SPLIT) {
    if (idx >= (int)p.per_list.d * p.num_splits) return false;
    split = (int)fast_div(idx, p.per_list);
    rem = idx - split * (int)p.per_list.d;
  }
  int t = (int)fast_div(rem, e.list_heads);
  const int h = rem - t * (int)e.list_heads.d;
  if (KEYS == kHalves) {  // split: all keys, the first half, the second
    const int in = t - e.cut_at;
    const bool half = (uint32_t)in < 2u * e.cut;
    split = half ? 1 + (in & 1) : 0;
    t = half ? in >> 1 : in < 0 ? t + e.cut : t - e.cut;
  }
  if (t >= num_q_tiles) return false;
  tile = num_q_tiles - 1 - t;
  if (SPLIT && e.pack)
    head = h * e.g;  // the list holds kv heads: first query head of the kv head
  else
    head = xcd * (int)e.list_heads.d + h;
  return true;
}

// max / sum over the lane pair (l, l^32) without going through the LDS
// crossbar.  v_permlane32_swap(a, b) exchanges a[32..63] with b[0..31]; with
// a == b == x the two results are (x_lo, x_lo) and (x_hi, x_hi).  The results
// are copied to scalars before the bit cast: a bit cast applied directly to a
// vector element reads element 0.
__device__ __forceinline__ void pair_swap(float x, float &lo, float &hi) {
  typedef __attribute__((ext_vector_type(2))) unsigned u2;
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const u2 r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const unsigned r0 = r[0], r1 = r[1];
  lo = __builtin_bit_cast(float, r0);
  hi = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float pair_max(float x) {
  float lo, hi;
  pair_swap(x, lo, hi);
  return fmaxf(lo, hi);
}
__device__ __forceinline__ float pair_sum(float x) {
  float lo, hi;
  pair_swap(x, lo, hi);
  return lo + hi;
}

// LDS visibility + workgroup barrier that does not drain outstanding global loads.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// State of one wave: 32 query rows (one per lane pair), fp32 O^T accumulators.  KB = 32-key blocks
// of every 64-key tile that the wave works on: 2 normally; 1 when two waves share the rows and
// each takes one half of every tile (short sequences: halves the serial MFMA chain of a wave).
template <typename T, int KB = 2> struct WaveAttn {
  using E = Elem<T>;
  f32x16_t o[4];       // O^T: d block x (16 d rows of this lane)
  u32x4_t pf[KB][2];   // P^T packed as B operand: key block x k-step
  u32x4_t qf[8];       // Q^T fragments (B operand), loaded once
  float m_run, l_run;  // running max (raw score units) and sum of this lane's keys
  float move_above, neg_ms;  // m_run plus the slack of its move; what it adds to the exponent
  int lane, l32, hh, g16, li;
  int k_addr[8];  // LDS byte offset of this lane's K fragment kk in tile slot 0, key block 0
  uint32_t v_addr[4];  // LDS address of the V^T fragment of d block d (k-step 0, low half)

  // kb0: first 32-key block of a tile this wave works on (0, or 1 for the second wave of a pair)
  __device__ __forceinline__ void init(const char *lds, int lane_, int v_region, int kb0 = 0) {
    lane = lane_;
    l32 = lane & 31;
    hh = lane >> 5;
    g16 = lane >> 4;
    li = lane & 15;
    m_run = -INFINITY;
    move_above = -INFINITY;
    neg_ms = 0.0f;
    l_run = 0.0f;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
    // Every other fragment address of the loop is one of these plus a compile-time constant
    // that fits the 16-bit offset field of the LDS instructions; the empty asm keeps the
    // compiler from recomputing them (it otherwise spends ~50 VALU instructions per tile).
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      k_addr[kk] = k_swizzle_off(l32, 2 * kk + hh) + kb0 * 32 * kRowBytes;
      asm volatile("" : "+v"(k_addr[kk]));
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int gran = d * 4 + (g16 & 1) * 2 + ((li & 3) >> 1);
      v_addr[d] = lds_address(lds) + v_region + v_swizzle_off(4 * hh + (li >> 2), gran) + (li & 1) * 8 + kb0 * 32 * kRowBytes;
      asm volatile("" : "+v"(v_addr[d]));
    }
  }

  // Q^T fragments of 32 rows in LDS, laid out like a K tile; off: their place less this wave's first tile row
  __device__ __forceinline__ void load_q_lds(const char *lds, int off) {
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) qf[kk] = lds_read_b128(lds, k_addr[kk] + off);
  }
  struct NoHook {
    template <typename I> __device__ __forceinline__ void operator()(I) const {}
  };
  // S^T = K Q^T for the wave's keys of the K tile at byte offset `koff` of the LDS segment.
  // The fragments of step kk+1 are requested before the MFMAs of step kk.  hook(i) runs
  // after MFMA i (0..8*KB-1): the callers spread their global loads over the MFMA stream with it.
  template <int KK0 = 0, int KK1 = 8, typename Hook = NoHook>
  __device__ __forceinline__ void qk(const char *lds, int koff, f32x16_t (&s)[KB], Hook hook = Hook()) {
    static_for<KK0, KK1>([&](auto kk_) {
      constexpr int kk = decltype(kk_)::value;
      static_for<0, KB>([&](auto kb_) {
        constexpr int kb = decltype(kb_)::value;
        const u32x4_t kf = lds_read_b128(lds, k_addr[kk] + koff + kb * 32 * kRowBytes);
        if constexpr (kk == 0) {
          f32x16_t z;
#pragma unroll
          for (int i = 0; i < 16; ++i) z[i] = 0.0f;
          s[kb] = E::mfma32(kf, qf[kk], z);
        } else {
          s[kb] = E::mfma32(kf, qf[kk], s[kb]);
        }
        hook(std::integral_constant<int, kk * KB + kb>());
      });
    });
  }

  // O^T += V^T P^T over the V tile at byte offset `voff` past the start of the V region.
  // Lane (d = 32*dblk + l32, hh): element e of k-step (kb, ks2) is the key
  // 32*kb + 16*ks2 + 8*(e/4) + 4*hh + e%4 -- the key P's element e carries.
  template <typename Hook = NoHook>
  __device__ __forceinline__ void pv(int voff, Hook hook = Hook()) {
    static_for<0, 8 * KB>([&](auto i_) {
      constexpr int i = decltype(i_)::value, kb = i / 8, ks2 = i / 4 % 2, d = i % 4;
      const int c = voff + (kb * 32 + ks2 * 16) * kRowBytes;
      const u32x2_t lo = lds_read_tr16(v_addr[d], c);
      const u32x2_t hi = lds_read_tr16(v_addr[d], c + 8 * kRowBytes);
      const u32x4_t vf = {lo[0], lo[1], hi[0], hi[1]};
      o[d] = E::mfma32(vf, pf[kb][ks2], o[d]);
      hook(i_);
    });
  }

  // Causal / length mask of one tile of scores (only called for tiles that can be cut); key0 =
  // first key of the wave's part of the tile.
  __device__ __forceinline__ void mask(f32x16_t (&s)[KB], int key0, int qrow, int offset, int n) {
    const int last = min(qrow + offset, n - 1) - key0 - 4 * hh;  // the lane's last key, from its first one
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (kb * 32 + 8 * (i >> 2) + (i & 3) > last) s[kb][i] = -INFINITY;
  }

  // P = exp2(s*c + neg_ms) rounded to T and packed as the B operand; returns this lane's sum
  // of the rounded values.
  __device__ __forceinline__ float probabilities(const f32x16_t (&s)[KB], float c) {
    float ps0 = 0.0f, ps1 = 0.0f;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ks2 = 0; ks2 < 2; ++ks2) {
        u32x4_t w;
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2) {
          const float e0 = fast_exp2(__builtin_fmaf(s[kb][8 * ks2 + 2 * e2], c, neg_ms));
          const float e1 = fast_exp2(__builtin_fmaf(s[kb][8 * ks2 + 2 * e2 + 1], c, neg_ms));
          w[e2] = E::pack2(e0, e1);
          // l sums the ROUNDED probabilities, the values P.V really used: for rows that see few
          // keys the rounding errors of numerator and denominator then cancel.  (In a design that
          // separates MFMA and softmax phases these dot instructions are costly -- they queue
          // behind the MFMAs of every wave on the SIMD: a softmax pass beside an MFMA-issuing wave
          // takes 1690 cycles with them, 1070 with plain adds -- in this interleaved loop the
          // two versions time the same.)
          if (e2 & 1)
            ps1 = dot2_ones<T>(w[e2], ps1);
          else
            ps0 = dot2_ones<T>(w[e2], ps0);
        }
        pf[kb][ks2] = w;
      }
    return ps0 + ps1;
  }

  // First half of the online softmax of one tile of (already masked) scores: row maxima and,
  // rarely, the move of the reference.  m_run is the reference maximum used in the exponent,
  // in raw score units.  It moves only when a row maximum exceeds it by more than kLazyLog2
  // in log2 units (probabilities then stay below 2^kLazyLog2, harmless in fp32 sums and in
  // the 16-bit P operand); a -inf reference always moves.  O and l are rescaled only then,
  // which after the first tiles is rare: what depends on the reference alone (the line `move_above`, the additive term
  // of the exponent) is computed then too, and a lane pair compares notes only then.
  __device__ __forceinline__ void row_max(const f32x16_t (&s)[KB], float scale_log2e) {
    float m0 = -INFINITY, m1 = -INFINITY;  // two chains: half the dependent latency
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (KB == 2) {
        m0 = fmaxf(m0, s[0][i]);
        m1 = fmaxf(m1, s[KB - 1][i]);
      } else if (i & 1) {
        m1 = fmaxf(m1, s[0][i]);
      } else {
        m0 = fmaxf(m0, s[0][i]);
      }
    }
    float mloc = fmaxf(m0, m1);
    if (__builtin_amdgcn_ballot_w64(mloc > move_above) != 0) {
      mloc = pair_max(mloc);
      const bool move = mloc > move_above;
      const float m_new = move ? mloc : m_run;
      const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
      const float alpha = move ? fast_exp2((m_run - m_use) * scale_log2e) : 1.0f;
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
      m_run = m_new;
      move_above = m_new + kLazyLog2 / scale_log2e;
      neg_ms = -m_use * scale_log2e;
    }
  }

  // KP waves that shared the rows (KB == 1) trade pieces of O^T: wave `part` keeps and will store the
  // ND = 4 / KP d blocks part*ND .., and hands every other wave the blocks that one keeps, with its maximum and
  // sum.  All as 16-byte pieces, lane by lane: conflict-free.  The maxima are uniform over a lane pair in
  // all of them.  lds_rows: trade_bytes(KP) bytes of the row block.
  static constexpr int kPieceBytes = 4 * 1024;  // one d block of a wave
  static constexpr int give_bytes(int kp) { return (4 - 4 / kp) * kPieceBytes + 512; }
  static constexpr int trade_bytes(int kp) { return kp * give_bytes(kp); }
  template <int KP> __device__ __forceinline__ void give(char *lds_rows, int part) const {
    constexpr int ND = 4 / KP;
    char *mine = lds_rows + part * give_bytes(KP);
    f32x4_t *dst = reinterpret_cast<f32x4_t *>(mine) + lane;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      if (d / ND == part) continue;  // (wave-uniform)
      f32x4_t *piece = dst + (d / ND < part ? d : d - ND) * 256;
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        piece[i4 * 64] = f32x4_t{o[d][4 * i4], o[d][4 * i4 + 1], o[d][4 * i4 + 2], o[d][4 * i4 + 3]};
    }
    *reinterpret_cast<float2 *>(mine + give_bytes(KP) - 512 + lane * 8) = float2{m_run, l_run};
  }
  // Folds what the others gave into d blocks PART*ND ..
  template <int KP, int PART> __device__ __forceinline__ void take(const char *lds_rows, float scale_log2e) {
    constexpr int ND = 4 / KP;
    float2 ml[KP];
    float m_new = m_run;
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      ml[q] = float2{m_run, l_run};
      if (q != PART)
        ml[q] = *reinterpret_cast<const float2 *>(lds_rows + (q + 1) * give_bytes(KP) - 512 + lane * 8);
    }
#pragma unroll
    for (int q = 0; q < KP; ++q) m_new = fmaxf(m_new, ml[q].x);
    const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
    const float f_own = fast_exp2((m_run - m_use) * scale_log2e);
    float l = 0.0f;  // in the same order in every wave
#pragma unroll
    for (int d = PART * ND; d < PART * ND + ND; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] *= f_own;
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const float f = fast_exp2((ml[q].x - m_use) * scale_log2e);
      l = __builtin_fmaf(ml[q].y, f, l);
      if (q == PART) continue;
      const f32x4_t *src = reinterpret_cast<const f32x4_t *>(lds_rows + q * give_bytes(KP)) + lane;
#pragma unroll
      for (int d = PART * ND; d < PART * ND + ND; ++d)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const f32x4_t v = src[((d / ND < q ? d : d - ND) * 4 + i4) * 64];
#pragma unroll
          for (int i = 0; i < 4; ++i) o[d][4 * i4 + i] = __builtin_fmaf(v[i], f, o[d][4 * i4 + i]);
        }
    }
    m_run = m_new;
    l_run = l;
  }

  // out[row][head][32*D0 .. +32*ND) = O^T / l, rounded once.  The lane layout of O^T (a lane holds 4
  // contiguous dims of one row at 4*ND places) would make every store instruction touch 32
  // rows with 16 bytes each; the tile goes through 2*ND KiB of LDS of this wave instead
  // (16-byte granule XOR row: conflict-free both ways with four d blocks; rows of one or two are shorter
  // than the banks, and up to 8 lanes meet in one, 1-2 % of a launch's cycles) and leaves as whole pieces of
  // 64*ND bytes, 4*ND lanes per row, past the L2: lines that are left there are written back at the end of the launch (rope
  // and attention, us, ordinary stores / these: 256 tokens of 28 heads 9.39 / 9.20, 600 14.64 / 14.16, 1019 20.5 / 19.7, of
  // 32 26.3 / 25.7, 2048 of 28 44.5 / 43.8; up to 128 tokens and from 4096 on the same).  So too with ND = 1, pieces of 64 bytes from
  // two waves to a line: a sector is enough (attention alone, us: 256 of 32 5.44 / 5.29, 512 of 28 7.98 / 7.78, 2000 of 12 22.7 / 22.4), and
  // where the output begins off a sector (16 bytes off: 512 of 28 8.80 / 8.60, 1019 18.0 / 17.4, of 32 19.8 / 19.6, 2048 of 28 41.7 / 41.7, 4096
  // 125.4 / 125.2).  lds_wave: this wave's region; out_blk: &out[first row of the
  // wave][head]; rows_valid: how many of the wave's 32 rows exist.
  template <int D0 = 0, int ND = 4>
  __device__ __forceinline__ void store(char *lds_wave, char *out_blk, size_t row_bytes, int rows_valid) {
    constexpr int G = 4 * ND, RB_ = G * 16, RPI = 64 / G;  // granules and bytes of a row, rows per instruction
    const float l_tot = pair_sum(l_run);
    const float inv = (l_tot > 0.0f) ? 1.0f / l_tot : 0.0f;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        u32x2_t w;
        w[0] = E::pack2(o[D0 + d][4 * i4] * inv, o[D0 + d][4 * i4 + 1] * inv);
        w[1] = E::pack2(o[D0 + d][4 * i4 + 2] * inv, o[D0 + d][4 * i4 + 3] * inv);
        const int gran = 4 * d + i4;  // 16-byte granule of dims 32d + 8*i4 .. +7; hh picks its half
        *reinterpret_cast<u32x2_t *>(lds_wave + l32 * RB_ + ((gran ^ (l32 & (G - 1))) << 4) + hh * 8) = w;
      }
    __builtin_amdgcn_wave_barrier();  // wave-private region: LDS ops of one wave complete in order
    const int r0 = lane / G, g0 = lane % G;
    u32x4_t v[2 * ND];
#pragma unroll
    for (int t = 0; t < 2 * ND; ++t) {
      const int r = RPI * t + r0;
      v[t] = lds_read_b128(lds_wave, r * RB_ + ((g0 ^ (r & (G - 1))) << 4));
    }
    char *dst = out_blk + (size_t)r0 * row_bytes + D0 * 64 + g0 * 16;
#pragma unroll
    for (int t = 0; t < 2 * ND; ++t) {
      if (RPI * t + r0 < rows_valid) store_device_b128(dst, v[t]);
      dst += RPI * row_bytes;
    }
  }
};

// Partial result of one key range (see PrefillParams::num_splits): this lane's row gets d blocks D0 .. D0+ND-1 of its
// unnormalised O^T as fp32, and (reference maximum in raw score units, sum) once per lane pair.
template <int D0 = 0, int ND = 4, typename T, int KB>
__device__ __forceinline__ void store_partial(const WaveAttn<T, KB> &w, float *o_row, float *ml_row, bool row_valid) {
  const float l_tot = pair_sum(w.l_run);
  if (!row_valid) return;
#pragma unroll
  for (int d = D0; d < D0 + ND; ++d)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4_t v = {w.o[d][4 * i4], w.o[d][4 * i4 + 1], w.o[d][4 * i4 + 2], w.o[d][4 * i4 + 3]};
      *reinterpret_cast<f32x4_t *>(o_row + 32 * d + 8 * i4 + 4 * w.hh) = v;
    }
  if (D0 == 0 && w.hh == 0) {
    ml_row[0] = w.m_run;
    ml_row[1] = l_tot;
  }
}

// The same through LDS: stored straight from the accumulator layout an instruction touches 32 rows with 32 bytes each, this
// way it writes whole pieces of 128*ND bytes (us: 200 tokens past 16001, 28 heads 55.1 -> 54.6; 64 past 3936, 40 heads 18.7 ->
// 18.15; 500 past 2500, 32 heads 36.4 -> 35.8; not so where few waves have rows at all, 4 past 5396, 28 heads 9.86 ->
// 10.0: up to kFewRows rows they go straight), and past the L2 (100 past 8000, 40 heads 29.5 -> 28.7; 200 past 16001, 28 heads
// 57.8 -> 56.8; 450 past 10000 78.9 -> 78.0; 100 past 8000, 32 heads of one kv head each 43.1 -> 43.8).  lds_wave: 4*ND KiB of this
// wave's own; o_row(r): d block 0 of row r of the wave's 32, of which rows_valid exist.
template <int D0, int ND, typename T, int KB, typename Row>
__device__ __forceinline__ void store_partial_rows(const WaveAttn<T, KB> &w, char *lds_wave, Row o_row, float *ml_row, bool row_valid,
                                                   int rows_valid) {
  constexpr int G = 8 * ND, RB_ = G * 16, RPI = 64 / G;  // granules and bytes of a row, rows per instruction
  const float l_tot = pair_sum(w.l_run);
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4_t v = {w.o[D0 + d][4 * i4], w.o[D0 + d][4 * i4 + 1], w.o[D0 + d][4 * i4 + 2], w.o[D0 + d][4 * i4 + 3]};
      const int gran = 8 * d + 2 * i4 + w.hh;
      *reinterpret_cast<f32x4_t *>(lds_wave + w.l32 * RB_ + ((gran ^ (w.l32 & (G - 1))) << 4)) = v;
    }
  if (D0 == 0 && w.hh == 0 && row_valid) {
    ml_row[0] = w.m_run;
    ml_row[1] = l_tot;
  }
  __builtin_amdgcn_wave_barrier();  // wave-private region: LDS ops of one wave complete in order
  const int r0 = w.lane / G, g0 = w.lane % G;
#pragma unroll
  for (int t = 0; t < 32 / RPI; ++t) {
    const int r = RPI * t + r0;
    const u32x4_t v = lds_read_b128(lds_wave, r * RB_ + ((g0 ^ (r & (G - 1))) << 4));
    if (r < rows_valid) store_device_b128(o_row(r) + D0 * 32 + g0 * 4, v);
  }
}

// The longest rows of a prompt, dealt to two workgroups: each has half of the keys, and the one that began first passes what it has to
// the other, lane by lane as it lies in registers, every word beside half of the launch's number, past the XCD's L2.  No fence, no flag;
// the other looks at what is stored last until it finds the number, then at all.  Both in the order of the halves, whoever folds.
//   The wait has an end, 0.1 s (the other one is under way): who has looked in vain goes over all keys by itself, as where no rows are shared.
constexpr int kHalfBytes = 4 * 17 * 1024;  // 4 waves of 32 floats, a maximum and a sum to a lane
#ifdef LLMHIP_BENCH
constexpr int kHalfLooks = 0;  // (the measurement library's copy: who began second goes over all keys by itself)
#else
constexpr int kHalfLooks = 1 << 17;
#endif
template <int D0, int ND, typename T, int KB>
__device__ __forceinline__ void pass_half(const WaveAttn<T, KB> &w, __amdgpu_buffer_rsrc_t words, int wave, uint64_t number) {
  const uint32_t tag0 = (uint32_t)number, tag1 = (uint32_t)(number >> 32);
  const int at = wave * 17 * 1024 + w.lane * 16;
  auto word = [&](int i, float x, float y) {
    store_device(words, at + i * 1024, __builtin_bit_cast(f32x4_t, u32x4_t{__builtin_bit_cast(uint32_t, x), tag0, __builtin_bit_cast(uint32_t, y), tag1}));
  };
#pragma unroll
  for (int i = 0; i < 8 * ND; ++i) word(i, w.o[D0 + i / 8][2 * (i % 8)], w.o[D0 + i / 8][2 * (i % 8) + 1]);
  word(8 * ND, w.m_run, w.l_run);
}
// Whether the other half was there, and is folded in
template <int D0, int ND, typename T, int KB>
__device__ __forceinline__ bool fold_halves(WaveAttn<T, KB> &w, __amdgpu_buffer_rsrc_t words, int wave, uint64_t number, bool first, float scale_log2e) {
  const uint32_t tag0 = (uint32_t)number, tag1 = (uint32_t)(number >> 32);
  const int at = wave * 17 * 1024 + w.lane * 16;
  u32x4_t v[8 * ND + 1];
  bool there = false;
  for (int looks = kHalfLooks; looks > 0 && !there; --looks) {
    asm volatile("" ::: "memory");  // (the load is made again)
    v[8 * ND] = __builtin_bit_cast(u32x4_t, load_device(words, at + 8 * ND * 1024));
    if (__builtin_amdgcn_ballot_w64(((v[8 * ND][1] ^ tag0) | (v[8 * ND][3] ^ tag1)) != 0) != 0) {
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    asm volatile("" ::: "memory");
    uint32_t differs = 0;
#pragma unroll
    for (int i = 0; i < 8 * ND; ++i) v[i] = __builtin_bit_cast(u32x4_t, load_device(words, at + i * 1024));
#pragma unroll
    for (int i = 0; i < 8 * ND; ++i) differs |= (v[i][1] ^ tag0) | (v[i][3] ^ tag1);
    there = __builtin_amdgcn_ballot_w64(differs != 0) == 0;
  }
  if (!there) return false;
  const float m = __builtin_bit_cast(float, (uint32_t)v[8 * ND][0]), l = __builtin_bit_cast(float, (uint32_t)v[8 * ND][2]);
  const float m_new = fmaxf(w.m_run, m), m_use = (m_new == -INFINITY) ? 0.0f : m_new;
  const float own = fast_exp2((w.m_run - m_use) * scale_log2e), other = fast_exp2((m - m_use) * scale_log2e);
  // (the first half's product is rounded, whichever it is)
  auto sum = [&](float mine, float theirs) {
    return first ? __builtin_fmaf(theirs, other, mine * own) : __builtin_fmaf(mine, own, theirs * other);
  };
  w.l_run = sum(w.l_run, l);
#pragma unroll
  for (int i = 0; i < 8 * ND; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      w.o[D0 + i / 8][2 * (i % 8) + j] = sum(w.o[D0 + i / 8][2 * (i % 8) + j], __builtin_bit_cast(float, (uint32_t)v[i][2 * j]));
  w.m_run = m_new;
  return true;
}

// One global_load_lds_dwordx4: lane l's 16 bytes at `src` land at the wave-uniform LDS address lds_addr + 16*l.
__device__ __forceinline__ void lds_dma(const char *src, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(src), "s"(lds_addr)
               : "m0");
}

// Global -> LDS tile loader without VGPR staging (buffer_load_dwordx4 ... lds: lane l's 16 bytes land at the
// wave-uniform LDS address in M0 + the instruction's offset + 16*l).  One wave instruction fills four 256-byte rows; the
// XOR swizzles are realised on the global side: the lane that owns physical granule pg of row r fetches the logical granule
// that belongs there.  A tile of TN keys is TN/4 instructions; slot s of wave w covers rows 4*(w*kSlots + s) .. +3.
// The lane offsets never change and rows past the end are cut off by the descriptor (they read as zero), so a load costs no
// vector ALU work, and M0 is written for every fourth one only: the instruction's offset moves both addresses, and
// the lane offsets make up for it.  (That nothing else uses M0 in between is checked in the built code, check_m0.py.)  The loads are issued from inline asm: the compiler would order every later LDS
// read behind a transfer it knows about (s_waitcnt vmcnt(0)).  Completion is waited for explicitly before the barrier that
// publishes a stage.
typedef __attribute__((ext_vector_type(4))) uint32_t buffer_t;
template <int NW, int TN, bool NT> struct DirectLoader {
  static constexpr int kSlots = TN / 4 / NW;  // instructions per wave per tile
  static constexpr int kLow = 1024 * ((kSlots < 4 ? kSlots : 4) - 1);
  uint64_t tile_step;                         // bytes to the next tile
  uint32_t whole, last;                       // records of a whole tile and of the cache's last one
  int keys_step;                              // keys to the next tile
  uint32_t lds_wave;                          // LDS byte offset of the wave's first row (wave-uniform)
  uint32_t off_k[kSlots], off_v[kSlots];      // lane offsets within a tile

  // Every step-th tile of n keys
  __device__ __forceinline__ void init(int wave, int lane, int row_bytes, int step, int n) {
    keys_step = TN * step;
    tile_step = (uint64_t)(uint32_t)(TN * row_bytes) * (uint32_t)step;
    whole = (TN - 1) * row_bytes + kRowBytes + kLow;
    last = ((n - 1) & (TN - 1)) * row_bytes + kRowBytes + kLow;
    lds_wave = __builtin_amdgcn_readfirstlane(wave * kSlots * 1024);
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
      const int r = 4 * (wave * kSlots + s) + (lane >> 4), pg = lane & 15;
      const uint32_t at = r * row_bytes + kLow - 1024 * (s & 3);
      off_k[s] = at + ((pg ^ (r & 15)) << 4);
      off_v[s] = at + (((((pg >> 2) ^ (r & 3)) << 2) | (pg & 3)) << 4);
      asm volatile("" : "+v"(off_k[s]), "+v"(off_v[s]));
    }
  }
  // Descriptor of a key tile, kLow bytes early, that walks from tile to tile.  Past the last key it has no
  // bytes: the loads that a workgroup makes ahead of its last steps fetch nothing (the last tile again before; us: 256 tokens of 32
  // heads 5.90 -> 5.84, 512 of 28 8.48 -> 8.40, 1400 22.84 -> 22.47, 2048 38.6 -> 38.1, 100 past 8000 of 40 27.0 -> 26.75).
  struct Stream {
    buffer_t d;
    int left;  // keys from the tile's first one on
  };
  __device__ __forceinline__ uint32_t records(int left) const {
    const uint32_t bytes = left >= TN ? whole : last;
    return left > 0 ? bytes : 0u;
  }
  __device__ __forceinline__ Stream stream(const char *base, int left) const {
    const uint64_t at = (uint64_t)base - kLow;
    return Stream{{(uint32_t)at, (uint32_t)(at >> 32), records(left), 0x00020000u}, left};
  }
  __device__ __forceinline__ void next(Stream &st) const {
    const uint64_t at = (((uint64_t)st.d[1] << 32) | st.d[0]) + tile_step;
    st.left -= keys_step;
    st.d[0] = (uint32_t)at;
    st.d[1] = (uint32_t)(at >> 32);
    st.d[2] = records(st.left);
  }
  // Slots 0 .. kSlots-1 of a tile in order, with no other tile's in between; lds_tile: LDS byte offset of the destination.
  // NT: the tile is read by this workgroup only (a packed chunk of one tile per kv head over a long
  // cache): non-temporal, like the decode kernel's loads (4 tokens over 131072 keys: 106 -> 91 us);
  // tiles that several workgroups read stay ordinary loads (non-temporal costs those 3-10 %).
  template <bool IS_V, int S> __device__ __forceinline__ void issue(const Stream &st, uint32_t lds_tile) const {
    constexpr int at = 1024 * (S % 4);
    if constexpr (at == 0) asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0" : : "s"(lds_wave), "s"(lds_tile + S * 1024) : "m0", "scc");
    const uint32_t off = IS_V ? off_v[S] : off_k[S];
    if constexpr (NT) asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 nt lds" : : "v"(off), "s"(st.d), "n"(at));
    else asm volatile("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 lds" : : "v"(off), "s"(st.d), "n"(at));
  }
  static __device__ __forceinline__ void wait_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
  // All but the last N loads of the wave
  template <int N> static __device__ __forceinline__ void wait_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
};

// ---------------------------------------------------------------------------
// NW waves, 32*NW/KP query rows, two LDS stages of SUB tiles, one barrier per stage.
// Every wave runs S(j+1) = K Q^T, the softmax of tile j and P(j).V(j) as one instruction
// stream (the compiler interleaves the softmax VALU work with the MFMAs); the tile loads
// are spread over that stream.  NW = 4, KP < 4: two workgroups per CU; else one.
// KP = 2: two waves per row block, each on one 32-key half of every 64-key tile; KP = 4: four waves, tiles of
// 128 keys; what they have is merged through LDS at the end.
// ---------------------------------------------------------------------------
template <PrefillKeys KEYS> struct LateOf { using type = PrefillBrief; };
template <> struct LateOf<kRanges> { using type = PrefillLate; };
template <> struct LateOf<kHalves> { using type = PrefillHalves; };

// The rows of a workgroup.  AGAIN: after it has looked for the other half of their keys in vain, over all of them.  True if they are still to be made.
template <typename T, int NW, int KP, bool NT, PrefillKeys KEYS, bool AGAIN = false>
__device__ __forceinline__ bool prefill_rows(addresses_t ea, u32x4_t eb, u32x2_t ec, typename LateOf<KEYS>::type late) {
  constexpr bool SPLIT = KEYS == kRanges;
  const PrefillLate p = late;
  // SUB tiles of 64 keys per stage and per barrier: with one workgroup per CU (NW = 8) a stage
  // holds 128 keys, which halves the number of times the waves are forced in step.
  // LDS: K tiles of both stages [2*SUB][16 KiB], then the V tiles likewise; tile t sits in
  // slot t % (2*SUB) of each region, so every fragment address is a per-lane register plus a
  // constant below 64 KiB.
  constexpr int KB = KP == 1 ? 2 : 1, TN = KP == 4 ? 2 * kTileN : kTileN, TB = TN * kRowBytes;
  constexpr int RB = NW / KP, BM = 32 * RB, PER = TN / 4 / NW, SUB = (NW == 8 && KP < 4) ? 2 : 1, NSLOT = 2 * SUB;
  constexpr int kVRegion = NSLOT * TB;
  constexpr int kWaveKeys = 32 * KB;  // keys of a tile per wave
  constexpr int kSplitKK = 3;  // k-steps of S(j+1) issued beside the row-maximum chain
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const PrefillShared e(ea, eb, ec, AGAIN || KEYS == kHalves);
  const bool pack = SPLIT && e.pack;  // (packed rows exist in split mode only)
  const int rows = pack ? e.m * e.g : e.m;
  int tile, head, split;
  if (!prefill_schedule<AGAIN ? kHalves : KEYS>(e, p, blockIdx.x, (rows + BM - 1) / BM, tile, head, split)) return false;
#ifdef LLMHIP_BENCH
  unsigned long long clk0 = 0, ref0 = 0;
  if (p.clock_probe) {
    clk0 = __builtin_amdgcn_s_memtime();
    ref0 = __builtin_amdgcn_s_memrealtime();
  }
#endif

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int kvh = (int)fast_div(head, e.g_div);
  // Rows of the tile.  Unpacked: rows are tokens of one head.  Packed: row index i stands for token
  // i / g of head kvh*g + i % g; `rows` counts them.  Everything below works on tokens: qtok is this
  // lane's token, tok_lo / tok_hi the first / last token of the wave's 32 rows.
  const int row0 = tile * BM;
  const int rows_end = min(rows, row0 + BM);
  const int rb = wave % RB, kpar = wave / RB;  // row block; which 32 keys of every tile (KP > 1)
  const int kw0 = (KP > 1) ? 32 * kpar : 0;   // first key of the wave's part of a tile
  const int qblk0 = row0 + rb * 32;
  const int l32_ = lane & 31;
  const int qidx = min(qblk0 + l32_, rows - 1);
  const bool row_valid = qblk0 + l32_ < rows;
  int qtok = qidx, qhead = head, tok_lo = qblk0, tok_hi = min(qblk0 + 31, rows - 1);
  int tile_tok_end = rows_end;  // one past the tile's last token
  if (pack) {
    qtok = (int)fast_div(qidx, e.g_div);
    qhead = head + qidx - qtok * e.g;
    tok_lo = (int)fast_div(qblk0, e.g_div);
    tok_hi = (int)fast_div(tok_hi, e.g_div);
    tile_tok_end = (int)fast_div(rows_end - 1, e.g_div) + 1;
  }
  const int n_vis = min(e.n, tile_tok_end + e.offset);  // keys any row of this tile can see
  constexpr int kTileShift = TN == 128 ? 7 : 6;
  static_assert(1 << kTileShift == TN, "");
  const int half = KEYS == kHalves ? ((n_vis + TN - 1) >> kTileShift) >> 1 : 0;  // tiles of the first one
  const int first = SPLIT ? split * p.first_each : KEYS == kHalves && split == 2 ? half : 0, step = SPLIT && p.range_keys == kWholeRange ? p.num_splits : 1;  // of this workgroup's tiles
  int first_keys = n_vis - first * TN;  // keys from its first one on, within its range
  const int range_keys = SPLIT ? p.range_keys : KEYS == kHalves && split == 1 ? half * TN : kWholeRange;
  if (KEYS != kAllKeys) first_keys = min(first_keys, range_keys);
  auto mine = [&](int keys) {  // its tiles that hold one of the first `keys` keys
    int tiles = ((KEYS != kAllKeys ? min(keys - first * TN, range_keys) : keys) + TN - 1) >> kTileShift;
    if (SPLIT && step > 1) tiles = tiles > 0 ? (int)fast_div(tiles + step - 1, p.splits_div) : 0;
    return tiles;
  };
  const uint32_t q_row_bytes = (uint32_t)e.H * kRowBytes;
  const int kv_row_bytes = e.Hkv * kRowBytes;
  const size_t kv_first = (size_t)(uint32_t)(first * TN) * kv_row_bytes + (size_t)kvh * kRowBytes;
  const char *kbase = e.k + kv_first, *vbase = e.v + kv_first;

  WaveAttn<T, KB> w;
  const size_t part_slot = SPLIT ? ((size_t)split * e.m + qtok) * e.H + qhead : 0;
  float *part_o = nullptr, *part_ml = nullptr;
  auto find_partial = [&] {
    part_o = p.ws_o + part_slot * kHeadDim;
    part_ml = p.ws_o + (size_t)p.num_splits * e.m * e.H * kHeadDim + part_slot * 2;
  };
  if (SPLIT && first_keys <= 0) {  // workgroup-uniform: no row of this tile sees a key of this range
    find_partial();
    w.init(lds, lane, kVRegion);
    store_partial(w, part_o, part_ml, row_valid);
    return false;
  }
  // Which of a pair begins first passes its half on: it is under way, and so the other one does not wait for a workgroup that is not.
  [[maybe_unused]] unsigned long long began = 0;
  [[maybe_unused]] int pair = 0;
  if constexpr (KEYS == kHalves) {
    if (split) {
      pair = ((rows + BM - 1) / BM - 1 - tile) * e.H + head;
      if (tid == 0)
        began = __hip_atomic_exchange(reinterpret_cast<unsigned long long *>(late.halves + (size_t)late.pairs * kHalfBytes) + pair,
                                      (unsigned long long)late.number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  // Q.  A fragment load straight into the operand layout touches 32 rows with 32 bytes each, 256 tag look-ups per
  // wave; Q goes through LDS like a K tile instead, fetched once as whole rows, and the first scores wait for it and K
  // tile 0 only (256 tokens, 32 heads, two waves per 64 rows: 7.4 -> 7.0 us; the wait 6.1 -> 5.9).  Its place is behind the K
  // and V tiles, or, where every row has one wave, begins with the V slots that the first stage fills.
  constexpr int kQRegion = KP > 1 ? 2 * NSLOT * TB : kVRegion + SUB * TB;
#pragma unroll
  for (int sl = 0; sl < 8 / KP && !AGAIN; ++sl) {  // (they are still there)
    const int r = 4 * (sl * NW + wave) + (lane >> 4);
    const int idx = min(row0 + r, rows - 1);
    const char *src = e.q + ((lane & 15) ^ (r & 15)) * 16;
    if (pack) {
      const int tok = (int)fast_div(idx, e.g_div);
      src += (uint64_t)(uint32_t)tok * q_row_bytes + (uint32_t)(head + idx - tok * e.g) * kRowBytes;
    } else {
      src += (uint64_t)(uint32_t)idx * q_row_bytes + (uint32_t)head * kRowBytes;
    }
    lds_dma(src, kQRegion + (sl * NW + wave) * 4 * kRowBytes);
  }

  DirectLoader<NW, TN, NT> ld;
  ld.init(wave, lane, kv_row_bytes, step, n_vis);
  // K runs one tile ahead of V: S(j+1) = K(j+1) Q^T is issued together with the softmax of
  // tile j, so K tile t is fetched SUB+1 iterations and V tile t SUB iterations before use.
  using Loader = DirectLoader<NW, TN, NT>;
  typename Loader::Stream kst = ld.stream(kbase, first_keys), vst = ld.stream(vbase, first_keys);
  static_for<0, SUB + 1>([&](auto u_) {
    constexpr int u = decltype(u_)::value;
    static_for<0, PER>([&](auto r) { ld.template issue<false, decltype(r)::value>(kst, u % NSLOT * TB); });
    ld.next(kst);
    if constexpr (u < SUB) {
      static_for<0, PER>([&](auto r) { ld.template issue<true, decltype(r)::value>(vst, kVRegion + u * TB); });
      ld.next(vst);
    }
  });
  const int J = mine(n_vis);
  // tiles in which this wave's keys hold at least one visible key
  const int Jw = (qblk0 < rows) ? max(0, min(J, mine(min(e.n, tok_hi + e.offset + 1) - kw0))) : 0;
  // The late arguments are asked for now, while the loads are under way, not at the place of each one's use
  asm volatile("" : : "s"(p.out));
  float scale = kScaleLog2e;  // (in a register: as a literal 8192 tokens take 0.8 % longer)
  asm volatile("" : "+s"(scale));
  if (SPLIT) asm volatile("" : : "s"(p.ws_o));
  w.init(lds, lane, kVRegion, (KP > 1) ? kpar : 0);
  ld.template wait_but<2 * SUB * PER>();  // Q and K tile 0
  lds_barrier();
  w.load_q_lds(lds, kQRegion + (rb - (KP > 1 ? kpar : 0)) * 32 * kRowBytes);

  f32x16_t sa[KB], sb[KB];  // scores of the current / the next tile, roles alternate
  if (Jw > 0) w.qk(lds, 0, sa);
  // A K load of the first stage lands where tile 0 was just read: no wave may issue it (one without rows would at
  // once) before all have read.
  ld.wait_all();
  lds_barrier();

  auto tile_step = [&](int j, int slot, f32x16_t (&s_cur)[KB], f32x16_t (&s_nxt)[KB]) {
    const int kslot = (slot + SUB + 1) % NSLOT, vslot = (slot + SUB) % NSLOT;  // fetched now
    if (j < Jw) {
      const int key0 = (SPLIT ? j * step + first : KEYS == kHalves ? j + first : j) * TN + kw0;
      if ((key0 + kWaveKeys - 1 > tok_lo + e.offset) || (key0 + kWaveKeys > e.n))
        w.mask(s_cur, key0, qtok, e.offset, e.n);
      // In the 8-wave kernel a burst of loads would stall every wave behind the texture addresser's
      // queue: one load every 8 * KB / PER MFMAs instead.  The 4-wave kernels run where a step is
      // short against a memory round trip, and issue a phase's loads beside its first MFMAs
      // (S=2560: 61.0 -> 59.1 us, S=3072: 76.3 -> 75.0 us; the 8-wave kernel loses 0.7 % that way).
      // (Paired waves, KB == 1, run short sequences, where a step is shorter than a memory round
      // trip: there all loads of a step go out with its first MFMAs.)
      auto k_hook = [&](auto i_) {
        constexpr int i = decltype(i_)::value;
        static_for<0, PER>([&](auto r_) {
          constexpr int r = decltype(r_)::value;
          if constexpr (KB == 1) {
            if constexpr (i == r) ld.template issue<false, r>(kst, kslot * TB);
            if constexpr (PER < 8 && i == PER + r) ld.template issue<true, r>(vst, kVRegion + vslot * TB);
          } else if constexpr (i == (NW == 4 ? r : (8 * KB / PER) * r + 1)) {
            ld.template issue<false, r>(kst, kslot * TB);
          }
        });
      };
      // The MFMAs of S(j+1) overlap the softmax of tile j: the first ones run beside the row
      // maximum chain, the rest -- and the MFMAs of P.V -- beside the exponentials.  (For the
      // wave's last tile the result is not used: one surplus pass instead of a branch that
      // would separate these MFMAs from the instructions they overlap with.)
      const int koff = ((slot + 1) % NSLOT) * TB;
      w.template qk<0, kSplitKK>(lds, koff, s_nxt, k_hook);
      w.row_max(s_cur, scale);
      w.template qk<kSplitKK, 8>(lds, koff, s_nxt, k_hook);
      w.l_run += w.probabilities(s_cur, scale);
      w.pv(slot * TB, [&](auto i_) {
        constexpr int i = decltype(i_)::value;
        static_for<0, PER>([&](auto r_) {
          constexpr int r = decltype(r_)::value;
          if constexpr (KB == 1 ? (PER == 8 && i == r) : i == (NW == 4 ? r : (8 * KB / PER) * r + 1))
            ld.template issue<true, r>(vst, kVRegion + vslot * TB);
        });
      });
    } else {
      static_for<0, PER>([&](auto r) { ld.template issue<false, decltype(r)::value>(kst, kslot * TB); });
      static_for<0, PER>([&](auto r) { ld.template issue<true, decltype(r)::value>(vst, kVRegion + vslot * TB); });
    }
    ld.next(kst);
    ld.next(vst);
  };

  for (int jb = 0; jb < J; jb += NSLOT) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int u = 0; u < SUB; ++u) {
        const int slot = st * SUB + u;  // compile-time after unrolling
        if (slot % 2 == 0)
          tile_step(jb + slot, slot, sa, sb);
        else
          tile_step(jb + slot, slot, sb, sa);
      }
      ld.wait_all();
      lds_barrier();
      if (st == 0 && jb + SUB >= J) break;  // workgroup-uniform: the second stage holds nothing
    }
  }
  // every wave is past the last barrier of the loop: nobody reads the K/V tiles any more
  if (SPLIT) find_partial();
  char *out_blk = p.out + (size_t)qblk0 * q_row_bytes + (size_t)head * kRowBytes;
  auto part_row = [&](int r) {  // where the partial of row r of the wave's goes
    int tok = qblk0 + r, h = head;
    if (pack) {
      const int idx = tok;
      tok = (int)fast_div(idx, e.g_div);
      h = head + idx - tok * e.g;
    }
    return p.ws_o + (((size_t)split * e.m + tok) * e.H + h) * kHeadDim;
  };
  if constexpr (KP > 1) {
    constexpr int kTrade = WaveAttn<T, KB>::trade_bytes(KP), ND = 4 / KP;
    char *rows_lds = lds + rb * kTrade;
    w.template give<KP>(rows_lds, kpar);
    constexpr int kNotes = 2 * NSLOT * TB - 32;
    static_assert(KEYS != kHalves || RB * kTrade + NW * 32 * 64 * ND <= kNotes, "");
    // (told to be in LDS: a read through a generic pointer would wait for the stores of the rows too)
    auto *notes = (volatile __attribute__((address_space(3))) uint32_t *)(lds + kNotes);
    if constexpr (KEYS == kHalves) {
      if (split && tid == 0) notes[0] = began == late.number;  // (the second to begin)
    }
    __syncthreads();
    [[maybe_unused]] bool in_vain = false;
    auto finish = [&](auto part) {
      constexpr int PART = decltype(part)::value;
      w.template take<KP, PART>(rows_lds, scale);
      if constexpr (KEYS == kHalves) {
        if (split) {
          const __amdgpu_buffer_rsrc_t words = byte_buffer(late.halves + (size_t)pair * kHalfBytes, kHalfBytes);
          if (!__builtin_amdgcn_readfirstlane(notes[0])) {
            pass_half<PART * ND, ND>(w, words, wave, late.number);
            return;
          }
          in_vain = !fold_halves<PART * ND, ND>(w, words, wave, late.number, split == 1, scale);
          if (in_vain) return;
        }
      }
      if (SPLIT && rows > kFewRows)
        store_partial_rows<PART * ND, ND>(w, lds + RB * kTrade + wave * (32 * 128 * ND), part_row, part_ml, row_valid, rows - qblk0);
      else if (SPLIT)
        store_partial<PART * ND, ND>(w, part_o, part_ml, row_valid);
      else
        w.template store<PART * ND, ND>(lds + RB * kTrade + wave * (32 * 64 * ND), out_blk, q_row_bytes, e.m - qblk0);
    };
    if (kpar == 0) finish(std::integral_constant<int, 0>());
    if (kpar == 1) finish(std::integral_constant<int, 1>());
    if constexpr (KP == 4) {
      if (kpar == 2) finish(std::integral_constant<int, 2>());
      if (kpar == 3) finish(std::integral_constant<int, 3>());
    }
    if constexpr (KEYS == kHalves) {
      if (split && __builtin_amdgcn_readfirstlane(notes[0])) {  // all waves or none
        if (lane == 0) notes[1 + wave] = in_vain;
        lds_barrier();
        return __builtin_amdgcn_readfirstlane(notes[1] | notes[2] | notes[3] | notes[4]) != 0;
      }
    }
  } else if (SPLIT) {
    if (rows > kFewRows)
      store_partial_rows<0, 4>(w, lds + rb * 32 * 512, part_row, part_ml, row_valid, rows - qblk0);
    else
      store_partial(w, part_o, part_ml, row_valid);
  } else {
    w.store(lds + rb * 32 * kRowBytes, out_blk, q_row_bytes, e.m - qblk0);
  }
#ifdef LLMHIP_BENCH
  if (p.clock_probe && blockIdx.x == 0 && tid == 0) {
    p.clock_probe[0] = __builtin_amdgcn_s_memtime() - clk0;
    p.clock_probe[1] = __builtin_amdgcn_s_memrealtime() - ref0;
  }
#endif
  return false;
}

template <typename T, int NW, int KP, bool NT, PrefillKeys KEYS>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void flash_prefill_kernel(addresses_t ea, u32x4_t eb, u32x2_t ec,
                                                                                  typename LateOf<KEYS>::type late) {
  const bool in_vain = prefill_rows<T, NW, KP, NT, KEYS>(ea, eb, ec, late);
  if constexpr (KEYS == kHalves) {
    if (!in_vain) return;
    lds_barrier();  // (tiles come where the notes are)
    asm volatile("" : "+s"(ea), "+s"(eb), "+s"(ec));  // (nothing is kept for this beside the first way)
    prefill_rows<T, NW, KP, NT, kAllKeys, true>(ea, eb, ec, late);
  }
}

// Folds the key-range partials of the output rows with the log-sum-exp rule.  256 threads handle 8
// (row, head) slots, 32 threads (4 dims each) per slot; grid = ceil(m * H / 8).
// a: partials, their maxima and sums, out, slots per split (m * H); c: splits, scale.
template <typename T>
__global__ __launch_bounds__(256) void prefill_combine_kernel(addresses_t a, u32x2_t c) {
  using E = Elem<T>;
  const float *ws_o = at_address<const float>(a[0]), *ws_ml = at_address<const float>(a[1]);
  char *out = at_address<char>(a[2]);
  const float scale_log2e = __builtin_bit_cast(float, (uint32_t)c[1]);
  const size_t stride = a[3];  // slots per split
  const size_t slot = (size_t)blockIdx.x * 8 + (threadIdx.x >> 5);
  const int d4 = threadIdx.x & 31;
  if (slot >= stride) return;
  // One pass, four key ranges per round: all loads of a round are issued before any is used, and the
  // running reference maximum moves between rounds (a pass for the maximum first would be one memory
  // round trip per key range).
  const int S = c[0];
  float M = -INFINITY, L = 0.0f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < S; s0 += 4) {
    float mv[4], lv[4];
    f32x4_t ov[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t at = (size_t)min(s0 + j, S - 1) * stride + slot;
      mv[j] = ws_ml[at * 2];
      lv[j] = ws_ml[at * 2 + 1];
      ov[j] = *reinterpret_cast<const f32x4_t *>(ws_o + at * kHeadDim + 4 * d4);
    }
    float Mn = M;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s0 + j < S) Mn = fmaxf(Mn, mv[j]);
    const float M_use = (Mn == -INFINITY) ? 0.0f : Mn;
    const float resc = fast_exp2((M - M_use) * scale_log2e);  // 0 on the first round (M = -inf)
    L *= resc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= resc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // exp2(-inf) = 0 for an empty range
      const float wt = (s0 + j < S) ? fast_exp2((mv[j] - M_use) * scale_log2e) : 0.0f;
      L += wt * lv[j];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += wt * ov[j][i];
    }
    M = Mn;
  }
  const float inv = (L > 0.0f) ? 1.0f / L : 0.0f;
  u32x2_t w;
  w[0] = E::pack2(acc[0] * inv, acc[1] * inv);
  w[1] = E::pack2(acc[2] * inv, acc[3] * inv);
  *reinterpret_cast<u32x2_t *>(out + slot * kRowBytes + d4 * 8) = w;
}

// The same fold for few output rows and many key ranges (a short chunk over a very long cache): one
// (row, head) slot per workgroup, its key ranges dealt to 8 groups of 32 threads (group sg takes ranges
// sg, sg + 8, ..., four per round), the groups merged through LDS -- the slots alone would not fill
// the chip and every thread would walk all ranges.  grid = m * H.
template <typename T>
__global__ __launch_bounds__(256) void prefill_combine_wide_kernel(addresses_t a, u32x2_t c) {
  using E = Elem<T>;
  const float *ws_o = at_address<const float>(a[0]), *ws_ml = at_address<const float>(a[1]);
  char *out = at_address<char>(a[2]);
  const float scale_log2e = __builtin_bit_cast(float, (uint32_t)c[1]);
  __shared__ float red_m[8], red_l[8];
  __shared__ f32x4_t red_o[8][32];
  const size_t stride = a[3], slot = blockIdx.x;
  const int sg = threadIdx.x >> 5, d4 = threadIdx.x & 31;
  const int S = c[0];
  float M = -INFINITY, L = 0.0f;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = sg; s0 < S; s0 += 32) {
    float mv[4], lv[4];
    f32x4_t ov[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t at = (size_t)min(s0 + 8 * j, S - 1) * stride + slot;
      mv[j] = ws_ml[at * 2];
      lv[j] = ws_ml[at * 2 + 1];
      ov[j] = *reinterpret_cast<const f32x4_t *>(ws_o + at * kHeadDim + 4 * d4);
    }
    float Mn = M;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (s0 + 8 * j < S) Mn = fmaxf(Mn, mv[j]);
    const float M_use = (Mn == -INFINITY) ? 0.0f : Mn;
    const float resc = fast_exp2((M - M_use) * scale_log2e);
    L *= resc;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= resc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float wt = (s0 + 8 * j < S) ? fast_exp2((mv[j] - M_use) * scale_log2e) : 0.0f;
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
    const float wt = fast_exp2((red_m[g8] - Mt_use) * scale_log2e);  // 0 for a group without ranges (-inf)
    Lt += wt * red_l[g8];
    const f32x4_t o = red_o[g8][d4];
#pragma unroll
    for (int i = 0; i < 4; ++i) tot[i] += wt * o[i];
  }
  const float inv = (Lt > 0.0f) ? 1.0f / Lt : 0.0f;
  u32x2_t w;
  w[0] = E::pack2(tot[0] * inv, tot[1] * inv);
  w[1] = E::pack2(tot[2] * inv, tot[3] * inv);
  *reinterpret_cast<u32x2_t *>(out + slot * kRowBytes + d4 * 8) = w;
}

constexpr int kClusterTiles = 6;

template <typename T, int NW, int KP = 1>
static hipError_t launch_prefill_t(const PrefillParams &p0, hipStream_t stream) {
  PrefillParams p = p0;
  constexpr int BM = 32 * NW / KP;
  constexpr int NT = 64 * NW;
  const int T_ = ((p.pack ? p.m * p.g : p.m) + BM - 1) / BM;
  int grid, list_heads;
  const int S_ = p.num_splits, share = prefill_xcd_share_log2(p.Hkv);
  p.xcd_bits = p.sched_shift = 0;
  p.per_xcd = 0;
  const int T_cut = T_ + p.cut;  // workgroups of a head
  if (p.pack) {
    list_heads = p.Hkv;
    grid = T_ * p.Hkv * S_;
    // Tiles of a kv head read the same keys.  Dealt one by one, T_ of them meet in 1 / (8 / gcd(kv heads, 8)) of the XCDs; where that puts
    // no more than two on an XCD, clusters of up to 6 are dealt instead, so that an L2 serves them (attention and combine, us, one by
    // one / clusters: 14 tokens past 25506 keys of 28 + 4 heads, 2 tiles, 23.9 / 18.5; 17 past 10561 of 12 + 2, 4 tiles, 13.3 / 10.8; 62 past
    // 30822 of 8 + 1, 16 tiles, 26.5 / 22.9; but 5 tiles of 4 kv heads 15.6 / 16.2, 12 26.5 / 27.9, and with 29 to a cluster 1.25 times).
    const int heads_xcds = p.Hkv % 8 == 0 ? 8 : p.Hkv % 4 == 0 ? 4 : p.Hkv % 2 == 0 ? 2 : 1;
    const int clusters = (T_ + kClusterTiles - 1) / kClusterTiles, each = (T_ + clusters - 1) / clusters;
    // (16-bit reciprocals of 1 to 6 are exact below 16384 items of a cluster; over 256 compute units plans have up to 5940)
    if (T_ > 1 && heads_xcds < 8 && T_ * heads_xcds <= 16 && (long long)each * p.Hkv * S_ < 16384) {
      const int last = (T_ - 1) % each + 1;
      p.per_xcd = (grid + 7) / 8;
      grid = 8 * p.per_xcd;
      p.tiles = (uint32_t)(each | last << 8);
      p.each_part = 65536u / each + 1;
      p.last_part = 65536u / last + 1;
      p.per_list = make_fast_div((uint32_t)(each * p.Hkv * S_));
    }
  } else if (share >= 0) {
    p.xcd_bits = 3;
    p.sched_shift = share;
    list_heads = p.H >> (3 - share);
    const int xcds = 1 << share;  // per list
    grid = 8 * ((list_heads * T_cut * S_ + xcds - 1) / xcds);
  } else {
    list_heads = p.H;
    grid = T_cut * p.H * S_;
  }
  // Two workgroups to a CU: the second one that a CU gets runs beside its first one, the heaviest ones' too, so that those
  // places are dealt from the lightest on (us: 700 tokens of 40 heads 13.0 -> 12.5, 1019 of 28 16.7 -> 16.1, of 32 18.6 -> 18.0,
  // 2700 of 12 35.4 -> 33.8).  With 64 rows each not where more are to follow, which would begin behind the light
  // ones and end last (900 of 40, 600 workgroups: 17.2 -> 17.9); with 128, of many more steps, there too (2700 of 28, 616:
  // 62.0 -> 60.2).
  p.second = p.second_end = 0;
  if (NW == 4 && KP < 4 && S_ == 1) {
    const int lists = 1 << p.xcd_bits, len = grid / lists, first = device_compute_units() / lists;
    if (len > first && (KP == 1 || len <= 2 * first + first / 8)) {
      p.second = first;
      p.second_end = len < 2 * first ? len : 2 * first;
    }
  }
  p.list_heads = make_fast_div((uint32_t)list_heads);
  if (!p.per_xcd) p.per_list = make_fast_div((uint32_t)(list_heads * T_));
  p.splits_div = make_fast_div((uint32_t)S_);
  // Key ranges lie side by side, or, where a key's rows together are long, one tile wide through each other, so that the workgroups
  // walk through the cache together: ranges that begin a multiple of MiB apart meet the same memory channels (rope and combine included,
  // us, side by side / through each other: 40 tokens past 16233 keys of 32 kv heads 66.8 / 58.0, past 4013 22.7 / 20.1, 64 past
  // 32174 119.1 / 108.3, 20 past 32216 of 8 40.2 / 34.7; of 4 and 2, 100 past 3943 19.8 / 20.6, 20 past 16318 18.3 / 18.9).
  const bool through = p.Hkv >= 8;
  constexpr int TN = KP == 4 ? 2 * kTileN : kTileN;
  p.first_each = through ? 1 : p.chunk / TN;
  p.range_keys = through ? kWholeRange : p.chunk;
  p.g_div = make_fast_div((uint32_t)p.g);
  const size_t tile_bytes = (NW == 8 || KP == 4 ? 2 : 1) * 4 * kTileBytes, q_bytes = (size_t)BM * kRowBytes;
  const size_t lds_bytes = tile_bytes + (KP > 1 ? q_bytes : q_bytes - tile_bytes / 4);  // (half of the V slots are Q's at first)
  // packed rows, one tile per kv head: every K/V tile is read by one workgroup only (KP == 1 there)
  const bool nt = KP == 1 && p.pack && T_ == 1, cut = S_ > 1;
  const auto whole = flash_prefill_kernel<T, NW, KP, false, kAllKeys>;
  const auto ranges = nt ? flash_prefill_kernel<T, NW, KP, (KP == 1), kRanges> : flash_prefill_kernel<T, NW, KP, false, kRanges>;
  const void *kern = cut ? reinterpret_cast<const void *>(ranges) : reinterpret_cast<const void *>(whole);
  [[maybe_unused]] const auto halves = flash_prefill_kernel<T, 4, 2, false, kHalves>;
  if (p.cut) kern = reinterpret_cast<const void *>(halves);
  // the opt-in for more than 64 KiB of dynamic LDS is per device: once per device and kernel
  static std::atomic<uint64_t> attr_done_all[4];
  std::atomic<uint64_t> &attr_done = attr_done_all[p.cut ? 3 : nt ? 2 : cut ? 1 : 0];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (!(attr_done.load(std::memory_order_acquire) & bit)) {
    e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return e;
    attr_done.fetch_or(bit, std::memory_order_release);
  }
  const PrefillEarly early(p);
  if (cut) {
    e = launch(ranges, dim3(grid), NT, lds_bytes, stream, early.a, early.b, early.c, static_cast<const PrefillLate &>(p));
  } else if (p.cut) {
    PrefillHalves late = {};
    late.out = p.out;
    late.halves = p.halves;
    late.number = p.number;
    late.pairs = p.cut * p.H;
    e = launch(halves, dim3(grid), NT, lds_bytes, stream, early.a, early.b, early.c, late);
  } else {
    PrefillBrief brief;
    brief.out = p.out;
#ifdef LLMHIP_BENCH
    brief.clock_probe = p.clock_probe;
#endif
    e = launch(whole, dim3(grid), NT, lds_bytes, stream, early.a, early.b, early.c, brief);
  }
  if (e != hipSuccess || p.num_splits == 1) return e;
  const size_t slots = (size_t)p.m * p.H;
  const addresses_t a = {address(p.ws_o), address(p.ws_o + (size_t)p.num_splits * slots * kHeadDim), address(p.out), slots};
  const u32x2_t c = {(uint32_t)p.num_splits, __builtin_bit_cast(uint32_t, kScaleLog2e)};
  if (slots <= 2048 && p.num_splits >= 8)
    return launch(prefill_combine_wide_kernel<T>, dim3((unsigned)slots), 256, 0, stream, a, c);
  return launch(prefill_combine_kernel<T>, dim3((unsigned)((slots + 7) / 8)), 256, 0, stream, a, c);
}

// Compute units of the current device (the kernel choice and the split counts aim at them); 256 when
// no device can be asked.
int device_compute_units() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int cus = cached[dev].load(std::memory_order_relaxed);
  if (cus <= 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      cus = 256;
    cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

// ---------------------------------------------------------------------------
// Kernel and key-range split of a call.
// ---------------------------------------------------------------------------
// The workgroup shapes, and what a launch of one costs on this part, in us: `fixed` per workgroup, a step over one
// tile `step_free` on an otherwise empty chip and `step_full` with every CU busy, up to `past_l2` times that once K and V
// outgrow the L2s of the 8 XCDs together (32 to 48 MiB; 32 heads, kQuad64: 1.13 us a step at 2450 keys, 1.6 at 2900).  Fitted
// over 13000 timed launches (204 shapes of 2-32 kv heads, 3-8192 tokens, 0-31000 cached keys, every shape and
// split), and again over 180000 (1800 shapes of 1-32 kv heads, 2-3000 tokens, 200-131072 cached keys).  Kernels have become faster since,
// 0.4-0.5 us of `fixed` and part of a step, and the figures were not fitted again: what that costs stands at the two rules below.
enum PrefillKind { kPair64, kPair128, kRows128, kRows256, kQuad64, kQuad32, kPrefillKinds };
struct PrefillShape {
  int rows, tile, per_cu;  // query rows, keys of a tile, workgroups resident on a CU
  double fixed, step_free, step_full, past_l2;
};
static const PrefillShape kShapes[kPrefillKinds] = {
    {64, 64, 2, 2.42, 0.74, 1.10, 1.5},   // 4 waves, two per row block
    {128, 64, 1, 3.92, 0.73, 0.85, 1.3},  // 8 waves, two per row block
    {128, 64, 2, 2.50, 1.10, 1.62, 1.3},  // 4 waves
    {256, 64, 1, 3.00, 1.12, 1.44, 1.3},  // 8 waves
    {64, 128, 1, 3.25, 1.03, 1.20, 1.5},  // 8 waves, four per row block
    {32, 128, 1, 2.99, 0.81, 1.03, 1.4},  // 4 waves, four per row block
};
struct PrefillPlan {
  PrefillKind kind;
  bool pack;
  int num_splits, chunk;
  int cut = 0, cut_at = 0;  // see prompt_cut
};

// The most scratch a plan may ask for.  Without a bound it grows with the chunk (behind 131072 keys 7151 tokens of 28
// heads 521 MB, 30000 of 40 1248).  By the model below 256 MiB costs at most 2.3 % behind up to 32768 keys and 6 % up
// to 131072; half of it would be felt: 4885 tokens of 28 heads behind 31258 keys take 2122 us with 213 MB and 2570
// within 128 MiB, 4096 of 40 behind 16384 1357 and 1415.
constexpr size_t kMaxPrefillScratch = (size_t)256 << 20;

static size_t partial_bytes(long long splits, int m, long long H) {
  return splits > 1 ? (size_t)splits * m * H * (kHeadDim + 2) * sizeof(float) : 0;
}

// A prompt (no more cached than new tokens) is never split: the fp32 partials would cost more HBM traffic than K and
// V.  Which shape: while the chip is not full, the launch waits for the chain of the waves with the most
// keys, so that as many waves as fit share every row block; once it is, the cheapest step wins.  Lines where the
// measured times cross (H=32 / 28 / 12, bf16, 256 CUs, us, best / runner-up):
//   four waves per 32 rows while one such workgroup per CU is enough, from about 100 keys: 256 tokens 6.7 / 7.0
//   four waves per 64 rows likewise, from about 480 keys: 512 tokens 9.2 / 9.8 (28 heads); with twice as many
//     workgroups as CUs from 1500 keys on: 2048 tokens 24.6 / 28.8 (12 heads)
//   two waves per 64 rows up to 1.3 128-row workgroups per CU: 1019 tokens 17.8 / 19.2 (28), 1400 25.6 / 25.8
//   two waves per 128 rows up to 2 per CU: 1700 tokens 34.0 / 35.3 (28)
//   256 rows from more than 1.5 workgroups per CU on: 3500 tokens 107.8 / 111 (28); 128 rows of one wave each up to there:
//     3000 tokens 81.7 / 85.8, 80.2 / 82.6 (32), 8192 tokens 188 / 202 (12)
// With the kernels of today the choice is 0.6 % slower than the fastest of the six shapes on average over 60 prompts of 24-4096
// tokens and 1-32 kv heads, 2.8 % at the 90th percentile, 11 % at most (1439 of 12 heads, two kv heads, 17.0 / 15.3, four waves per 64 rows).
static PrefillKind prompt_kind(int m, long long n_vis, int H, int cus) {
  auto per_cu = [&](int rows) { return (double)((m + rows - 1) / rows) * H / cus; };
  if (n_vis > 96 && per_cu(32) <= 1.05) return kQuad32;
  if ((n_vis >= 480 && per_cu(64) <= 1.05) || (n_vis >= 1500 && per_cu(64) <= 2.0)) return kQuad64;
  if (per_cu(128) <= 1.3) return kPair64;
  if (per_cu(128) <= 2.0) return kPair128;
  return per_cu(256) > 1.5 ? kRows256 : kRows128;
}

// Where two waves share 64 rows and not every CU has two workgroups, the launch waits for those with the most keys, while others have long
// ended: the longest rows are dealt to two workgroups each (see pass_half), as many as leave places for all workgroups at once, and as many
// as leave those that are not cut longer than a half and what it is passed on in, which takes as long as 6 steps.  Cut ones come behind those that
// are longer than a half and 4 steps (by 2 to 6 the same; before all others 1.05 to 1.15 times as long: the longest rows then begin later and
// beside longer ones).  Attention, us, whole / so: 1019 tokens of 28 + 4 heads (of 16 steps 14) 14.15 / 13.8, 930 13.35 / 13.05, 1088 15.1 / 15.05, 930 of 32
// + 32 13.75 / 13.6, 1480 of 12 + 2 17.1 / 15.35 (another box 14.9 / 14.1, 13.2 / 12.75, 15.9 / 15.4, 15.2 / 13.8, 17.2 / 15.0, before those who look in vain made
// their rows themselves, which costs up to 0.1); with 3 steps for passing a half on 700 of 28 + 4 10.35 / 11.1.
static void prompt_cut(int m, long long n_vis, int g, int Hkv, int cus, int &cut, int &cut_at) {
  constexpr int kPassSteps = 6, kOrderSteps = 4;
  const int share = prefill_xcd_share_log2(Hkv), H = g * Hkv;
  const long long tiles = (m + 63) / 64, longest = (n_vis + kTileN - 1) / kTileN;
  // (a list has the heads of 2^share XCDs)
  const long long places = (share >= 0 ? (2LL * cus / 8 << share) / (H >> (3 - share)) : 2LL * cus / H) - tiles;
  long long most = longest / 2 - kPassSteps;
  if (places < most) most = places;
  if (tiles < most) most = tiles;
  cut = cut_at = 0;
  if (most < 1 || 2 * cus > 1023) return;  // (places are told in 10 bits)
  cut = (int)(most < 63 ? most : 63);
  const long long before = longest - cut - ((longest + 1) / 2 + kOrderSteps) + 1;
  cut_at = before < 0 ? 0 : (int)(before < tiles - cut ? before : tiles - cut);
  if (cut_at > 63) cut_at = 63;
}

// A chunk behind a longer cache makes few workgroups with many keys each: its key range is cut, and with fewer rows than a
// tile has the g query heads of a kv head share a tile (K and V of the kv head are then read once, not g times).
// Taken is the combination of shape, packing and cut that the costs above make cheapest: workgroups in rounds of as
// many as are resident at once, 2.65 us and the traffic of the partials for the combine launch.  Only combinations whose
// partials fit max_bytes are looked at; an unsplit one always does.  Over the 1800 measured shapes the choice was 1.1 %
// slower than the fastest combination on average, 4 % at the 90th percentile; with the kernels of today, over 110 shapes of 2-512
// tokens behind 260-29600 keys, 1.9 % and 5.4 %, 22 % at most (19 tokens behind 22155 keys of 20 + 4 heads 20.6 / 16.9 us, 121 behind 1350 of
// 28 + 4 13.3 / 11.7), and since ranges go through each other and tiles in clusters 2.0 % over 761 shapes, which constants fitted again would
// make 1.3 %.  Among combinations within 4 % of the
// cheapest one that reads K and V once and gives every CU the same number of workgroups is preferred.
// Rows that fit one 256-row tile over a cache larger than the last-level cache are a stream from HBM: that tile's loads are
// non-temporal then, and nothing else was faster (us, it / the best other one: 23 tokens over 68925 keys of 4 kv heads 49.6
// / 54.3, 7 over 127579 of 8 90.9 / 98.8; below 256 MiB of K and V it no longer holds: 38 over 17018 of 8 36.6 / 31.2).
// Against fixed rules (a cut for about one round of workgroups of 128 or 256 rows), us: 3 tokens over 3000 keys 28.9 /
// 9.3, 20 over 600 11.5 / 8.5, 130 over 2000 28.0 / 16.8, 200 over 16001 63.0 / 58.3 (28 heads); 300 over 30000, 40 heads,
// 227 / 175.  (1800 other shapes: 0.68 of the time of the fixed rules on average, 22 of them more than 2 % slower.)
static PrefillPlan chunk_plan(int m, long long n_vis, long long past, int g, int Hkv, int cus, size_t max_bytes) {
  PrefillPlan best = {kPair64, false, 1, kWholeRange};
  double best_us = 1e30;
  const double kv_bytes = 2.0 * n_vis * Hkv * kRowBytes;
  double over = (kv_bytes / (1 << 20) - 32.0) / 16.0;  // how far K and V are past the L2s
  over = over < 0 ? 0 : over > 1 ? 1 : over;
  const bool streamed = kv_bytes > 256 << 20 && g > 1 && (long long)m * g <= kShapes[kRows256].rows &&
                        partial_bytes(2, m, (long long)g * Hkv) <= max_bytes;
  for (int kind = 0; kind < kPrefillKinds; ++kind)
    for (int pack = 0; pack < (g > 1 ? 2 : 1); ++pack) {
      if (streamed && !(kind == kRows256 && pack)) continue;
      const PrefillShape &sh = kShapes[kind];
      const long long rows = pack ? (long long)m * g : m, tiles = (rows + sh.rows - 1) / sh.rows;
      const long long groups = pack ? Hkv : (long long)Hkv * g;
      const double last_rows = ((double)sh.rows * (tiles - 1) * tiles / 2 + rows) / tiles / (pack ? g : 1);
      const double keys = past + last_rows;  // that a tile's last row sees, on average
      for (int s = pack ? 2 : 1; s <= kMaxPrefillSplits; s += s < 16 ? 1 : s < 32 ? 2 : s < 64 ? 4 : 16) {
        if (s > 1 && n_vis / s < 128) break;
        const long long chunk = s > 1 ? ((n_vis + s - 1) / s + 127) / 128 * 128 : n_vis;
        const long long splits = (n_vis + chunk - 1) / chunk;  // no empty trailing range
        if (partial_bytes(splits, m, (long long)g * Hkv) > max_bytes) continue;
        const long long items = tiles * groups * splits, slots = (long long)cus * sh.per_cu;
        double busy = (double)items / cus;
        busy = sh.per_cu == 2 ? busy - 1 : busy * busy;
        busy = busy < 0 ? 0 : busy > 1 ? 1 : busy;
        const double step = (sh.step_free + (sh.step_full - sh.step_free) * busy) * (1.0 + over * (sh.past_l2 - 1.0));
        const double most = (double)((chunk + sh.tile - 1) / sh.tile);
        double mean = keys / (splits * sh.tile) + 0.5;
        if (mean > most) mean = most;
        double us = sh.fixed + step * most;
        if (items > slots) {
          const double rounds = 0.63 * ((items + slots - 1) / slots) + 0.37 * ((double)items / slots);
          const double all = (sh.fixed + step * mean) * rounds;
          if (all > us) us = all;
        }
        us += 1.8;
        if (splits > 1) us += 2.65 + (double)splits * m * g * Hkv * (kHeadDim + 2) * sizeof(float) / 1.9e6;
        if (tiles == 1 && items % cus == 0) us *= 0.96;
        if (us < best_us) {
          best_us = us;
          best = {(PrefillKind)kind, pack != 0, (int)splits, splits > 1 ? (int)chunk : kWholeRange};
        }
      }
    }
  return best;
}

// The last answers are kept per thread: every layer of a model asks for the same chunk (several hundred combinations).
static PrefillPlan plan_prefill(int m, int n, int offset, int g, int Hkv, int cus, size_t max_bytes) {
  const long long n_vis = ((long long)m + offset < n) ? (long long)m + offset : n;  // keys the last row sees
  if (prefill_is_prompt(m, n_vis)) {
    PrefillPlan pl = {prompt_kind(m, n_vis, g * Hkv, cus), false, 1, kWholeRange};
    if (pl.kind == kPair64) prompt_cut(m, n_vis, g, Hkv, cus, pl.cut, pl.cut_at);
    return pl;
  }
  struct Memo {
    int m, n, offset, g, Hkv, cus;
    size_t bytes, max_bytes;  // what the plan takes, what it was allowed
    PrefillPlan plan;
  };
  constexpr int kMemo = 8;
  static thread_local Memo memo[kMemo] = {};
  static thread_local unsigned next = 0;
  for (const Memo &e : memo)  // (the cheapest plan of a larger allowance that fits this one is the cheapest here)
    if (e.m == m && e.n == n && e.offset == offset && e.g == g && e.Hkv == Hkv && e.cus == cus &&
        e.bytes <= max_bytes && max_bytes <= e.max_bytes)
      return e.plan;
  const PrefillPlan pl = chunk_plan(m, n_vis, n_vis - m, g, Hkv, cus, max_bytes);
  memo[next++ % kMemo] = Memo{m, n, offset, g, Hkv, cus, partial_bytes(pl.num_splits, m, (long long)g * Hkv), max_bytes, pl};
  return pl;
}

size_t flash_prefill_workspace_bytes(int m, int n, int offset, int group_size, int kv_head_num) {
  const PrefillPlan pl = plan_prefill(m, n, offset, group_size, kv_head_num, device_compute_units(), kMaxPrefillScratch);
  return partial_bytes(pl.num_splits, m, (long long)group_size * kv_head_num);
}

static size_t halves_bytes(long long pairs) { return pairs * (kHalfBytes + sizeof(uint64_t)); }
size_t flash_prefill_halves_bytes(int m, int n, int offset, int group_size, int kv_head_num) {
  const PrefillPlan pl = plan_prefill(m, n, offset, group_size, kv_head_num, device_compute_units(), 0);
  return halves_bytes((long long)pl.cut * group_size * kv_head_num);
}

// Where a call may not do with less: a chunk behind at least 2048 keys and 8 times its own length whose unsplit form would
// leave more than half of the chip idle.  The size is that of one round of workgroups with whole tiles of 128 or 256
// rows.  This is what callers under graph capture were promised; it does not move with the plan above, so that a
// better plan never turns a call away that ran before.
size_t flash_prefill_least_workspace_bytes(int m, int n, int offset, int group_size, int kv_head_num) {
  const long long n_vis = ((long long)m + offset < n) ? (long long)m + offset : n;
  const long long cus = device_compute_units(), H = (long long)group_size * kv_head_num;
  if (n_vis < 8LL * m || n_vis < 2048 || 2 * ((m + 255LL) / 256) * H >= 3 * cus) return 0;
  const bool pack = group_size > 1 && m < 128;
  const long long rows = pack ? (long long)m * group_size : m, groups = pack ? kv_head_num : H;
  const int tile = rows >= 192 ? 256 : 128;
  const long long wgs = (rows + tile - 1) / tile * groups;
  long long splits = (tile == 256 ? cus : 2 * cus) / wgs;
  if (splits > n_vis / 1024) splits = n_vis / 1024;
  const long long most = wgs <= 2 ? kMaxPrefillSplits : kMaxPrefillSplits / 2;
  if (splits > most) splits = most;
  if (splits <= 1) return 0;
  const long long chunk = ((n_vis + splits - 1) / splits + 127) / 128 * 128;
  return partial_bytes((n_vis + chunk - 1) / chunk, m, H);
}

template <typename T> static hipError_t launch_prefill(const PrefillParams &p, PrefillKind kind, hipStream_t stream) {
  switch (kind) {
    case kPair64: return launch_prefill_t<T, 4, 2>(p, stream);
    case kPair128: return launch_prefill_t<T, 8, 2>(p, stream);
    case kRows128: return launch_prefill_t<T, 4, 1>(p, stream);
    case kRows256: return launch_prefill_t<T, 8, 1>(p, stream);
    case kQuad64: return launch_prefill_t<T, 8, 4>(p, stream);
    default: return launch_prefill_t<T, 4, 4>(p, stream);
  }
}

#ifdef LLMHIP_BENCH
hipError_t launch_flash_prefill(void *out, const void *q, const void *k, const void *v, int m,
                                int n, int offset, int group_size, int kv_head_num, int dt,
                                hipStream_t stream, void *workspace, size_t workspace_bytes, void *clock_probe) {
  PrefillParams p;
  p.clock_probe = static_cast<unsigned long long *>(clock_probe);
#else
hipError_t launch_flash_prefill(void *out, const void *q, const void *k, const void *v, int m,
                                int n, int offset, int group_size, int kv_head_num, int dt,
                                hipStream_t stream, void *workspace, size_t workspace_bytes) {
  PrefillParams p;
#endif
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = static_cast<char *>(out);
  p.m = m;
  p.n = n;
  p.offset = offset;
  p.g = group_size;
  p.Hkv = kv_head_num;
  p.H = group_size * kv_head_num;
  if (workspace_bytes > kMaxPrefillScratch) workspace_bytes = kMaxPrefillScratch;
  const PrefillPlan pl =
      plan_prefill(m, n, offset, group_size, kv_head_num, device_compute_units(), workspace ? workspace_bytes : 0);
  p.cut = p.cut_at = 0;
  if (pl.cut && workspace && halves_bytes((long long)pl.cut * p.H) <= workspace_bytes && !may_be_capturing(stream)) {
    p.cut = pl.cut;
    p.cut_at = pl.cut_at;
    p.halves = static_cast<char *>(workspace);
    p.number = launch_number();
  }
  p.pack = pl.pack ? 1 : 0;
  p.num_splits = pl.num_splits;
  p.chunk = pl.chunk;
  p.ws_o = static_cast<float *>(workspace);
  return dt == kDtFloat16 ? launch_prefill<_Float16>(p, pl.kind, stream) : launch_prefill<__bf16>(p, pl.kind, stream);
}

}  // namespace LLMHIP_NS
