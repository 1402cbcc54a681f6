// Projection of many rows: out[m][n] = lhs[m][k] . W[n][k]^T + bias, fp32 accumulation, one rounding, for calls whose
// tiles fit the chip in one round (matmul_tile_takes); a launch that needs more is left to hipBLASLt.
//
// A workgroup computes one tile of 32*MT lhs rows x 32*NT features over all of k in stages of KS * 64 k (KS 128-byte
// lines of every operand row).  Lines travel global -> LDS without registers, STAGES of them in flight or in use; a
// fragment load straight into the operand layout, 16 rows by 64 bytes, ran at a third of the rate.
// Four waves, one per SIMD, take a quadrant each.  A wave issues one instruction every 4-5 cycles and an MFMA takes
// 16, so that two others fit between two MFMAs: the loop is written as slots, one MFMA each with the fragment reads (one; two
// in tiles of up to 96 x 96) and line loads that go out before it, and a line load is one instruction (constant lane
// offsets, the LDS address in M0 for four of them at a time).  One barrier a stage, where the last fragments of this
// stage have come back: it frees the stage's place and publishes the next one.  The loads of a stage are spread over the slots
// behind it, at most one to a slot where a stage has one line: the last 40 of 56 of 128 x 224, half of them in tiles of up to 128 x
// 96.  A CU takes in 64 bytes per cycle and no more (128 x 224: 704 cycles of loads beside 896 of MFMAs), and the fewer slots
// share them the longer the loads hold the wave up (3584 x 3584, 2048 rows, over 28 and over 40 slots: loop 41.3, 39.0 us).
//   Eight waves, two for each quadrant on alternate halves of k, hide more latency but trade their sums through LDS
// at the end and issue more: 3584 x 3584, 2048 rows 54.9 us, this kernel 46.2; 4096 x 4096 67.6 / 59.3; 1536 x 1536,
// 2048 rows 17.5 / 13.7; 512 x 3584, 2048 rows 14.8 / 13.6.  mfma_32x32x16, with half the operand reads, is no
// faster (4096 x 4096 62.3 / 57.9), the power it saves being small.
//   Small tiles are bound by the barrier and the LDS latency of a stage, and take several lines per stage (32 x 32, four
// lines instead of two: 512 x 3584, 400 rows 8.5 -> 7.8 us; 1536 x 1536, 100 rows 5.4 -> 4.9).  There the barrier comes so late that
// the loads go out in a burst behind it: 32 x 32 all eight in the last of 8 slots, 64 x 32 (two lines) six in the last two of 8.
// Where the time of a launch goes, by clock stamps in a copy of the kernel, us: 128 x 224 tile, k = 3584: 2.6 until the first
// lines are in, 56 stages of 0.67, 2.3 for the store (of pieces of 64 bytes into the L2s, before rows past them), the rest launch.
// A stage takes 1120 cycles at 1.68 GHz: the clock is what the power leaves (half of the chip: 1090 cycles at 2.2 GHz; without the line loads 1.9 GHz).
//
// A lane's accumulators are four features of one lhs row; W rows are dealt to LDS so that two neighbouring blocks make
// them eight, and a store 16 bytes.  The bias goes to LDS ahead of the first lines: read from memory at the end it
// was one round trip more per pair of blocks (epilogue 6.2 us in the kernel of eight waves).
//
// Rows of the operands lie k elements apart, often a multiple of 4 KiB: workgroups that walk k in step would ask few
// memory channels for everything.  Each XCD starts at another eighth of k, neighbouring tiles of W rows a line apart
// (4096 x 4096, 1024 rows: 40 -> 36.6 us; 3584 x 3584, 2048 rows, W from HBM: 51.8 -> 49.5, kernel of eight waves).
//   A CU draws no more than 30 to 45 GB/s from beyond its XCD's L2, however much it has under way.  Tiles of the same W rows that
// take the lines in one order leave all of that to the one that is ahead, and the others wait with it (3584 x 3584, 256 rows: 31 GB/s of
// W to a tile of 64 rows, and as long with 112 workgroups as with 224).  So lines go in groups, and each of up to 4 such tiles
// begins at another place of a group: the first to ask for a line is a different one each time, and the rest find it in the L2 a moment later
// (us, one order / so, W from HBM: 3584 x 3584, 64 rows 10.4 / 9.0, 256 18.2 / 13.9, 512 24.1 / 20.2, 1024 30.2 / 27.2, 2048 44.0 / 43.0;
// 4096 x 4096, 256 rows 20.2 / 15.3; 5120 x 5120, 768 rows 47.9 / 43.7; what leaves the L2s downwards stays within
// 5 %: 256 rows 39.9 / 41.8 MiB, 2048 131.4 / 129.4).
// With W in the last-level cache it costs 2 to 6 % (3584 x 3584, 256 rows 11.5 / 12.2, 1024 24.5 / 25.0), and more the larger group and tile are, the lines of
// a group being in the L2 longer: hence groups of 8, 4 and 2 (2048 rows by groups of 8 43.8).  Where lhs is the larger operand there is nothing to gain (512 x 3584,
// 2048 rows 11.6 / 12.6 by groups of 8).  Half or a quarter of k apart instead, the small ones are as fast, but what the L2 has to keep outgrows it (1024 rows 36.0).
//   Stages under way: as few as hold 64 to 100 KiB, but for 96 x 64.  More of them are no faster anywhere, and begin with a longer burst (5 / 9 stages of a
// 64 x 64 tile, us: 512 x 3584, 2048 rows 12.6 / 13.1, 3584 x 3584, 256 rows 14.15 / 14.55; 3 / 4 of 32 x 32, 512 x 3584, 512 rows 7.1 / 7.35;
// 3 / 5 of 96 x 128, 3584 x 3584, 768 rows 24.0 / 24.9; one line to a stage less and four stages of 64 x 32: 256 x 1536, 2048 rows 5.65 / 5.45).
//
// bf16, us, hipBLASLt / here, back-to-back calls, W walked through 800 MB (hipBLASLt takes the host 10-13 us a call, which is
// what its small sizes show): 3584 x 3584: 64 rows 13.7 / 9.4, 128 rows 22.5 / 11.5, 256 rows 20.1 / 14.1, 768 rows 32.2 / 23.9,
// 2048 rows 55.9 / 44.1; 512 x 3584: 100 rows 13.4 / 6.7, 2048 rows 19.3 / 12.4; 1536 x 1536: 128 rows 9.7 / 4.8; 5120 x 5120: 100
// rows 27.6 / 24.7, 1280 rows 76.1 / 55.3.
#include <atomic>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace LLMHIP_NS {

namespace {

constexpr int kTileThreads = 256;
constexpr int kLineK = 64;             // k of a 128-byte line of an operand row
constexpr int kStageRow = 2 * kLineK;  // its bytes
constexpr int kBiasBytes = 4 * 512;    // LDS: bias of each wave's features
constexpr int kBandRows = 4;           // m tiles of a band
constexpr int kMostPieces = 8;         // of k
constexpr int kWordsBytes = 2 * 16 * kTileThreads;  // of a piece's sums
#ifdef LLMHIP_BENCH
constexpr uint32_t kLooks = 0;  // (the measurement library's copy: a workgroup that adds up takes no words for new, and makes all sums by itself)
#else
constexpr uint32_t kLooks = 2000;      // 0.7 us each or more: what a launch takes, many times over
#endif

// LDS offset of logical 16-byte granule g of a staged row
__device__ __forceinline__ int stage_off(int row, int g) { return row * kStageRow + ((g ^ ((row >> 1) & 7)) << 4); }

template <int N> __device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "i"(N) : "memory");
}

// global_load_lds_dwordx4, OFF (0, 1024, 2048 or 3072) added to the global address and to the LDS address in M0, which
// nothing but the assembly of this kernel uses (checked in the built code, check_m0.py)
template <int OFF> __device__ __forceinline__ void line_load(uint32_t voff, const char *base) {
  if constexpr (OFF == 0) asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base));
  else asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" : : "v"(voff), "s"(base), "n"(OFF));
}

// What the workgroups of a tile whose k is cut pass on (PIECES): fetched from memory while the first lines are under way.
struct TilePieces {
  char *words;   // [tile][piece][half of a lane's four][thread], 16 bytes each: two sums, beside either half of the launch's number
  uint64_t number;
  uint32_t looks;
};
struct NoPieces {};

template <typename T, int MT, int NT, int KS, int STAGES, bool PIECES>
__global__ __launch_bounds__(kTileThreads, 2) void matmul_tile_kernel(addresses_t a_, u32x4_t size, u32x2_t divisors,
                                                                      std::conditional_t<PIECES, TilePieces, NoPieces> late) {
  using E = Elem<T>;
  static_assert(!PIECES || MT * NT == 1);
  const char *x = at_address<const char>(a_[0]), *w = at_address<const char>(a_[1]);
  const float *bias = at_address<const float>(a_[2]);
  uint16_t *out = at_address<uint16_t>(a_[3]);
  const int m = size[0], n = size[1], k = size[2] & 0x1fffffu, pieces = PIECES ? (int)(size[2] >> 21) : 1;
  constexpr int BM = 32 * MT, BN = 32 * NT;
  constexpr int kLineBytes = (BM + BN) * kStageRow, kStageBytes = KS * kLineBytes;
  constexpr int L = MT + NT;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int i = lane & 15, cg = lane >> 4;

  // Workgroups are dealt round-robin to the 8 XCDs: each takes a run of tiles, and runs go through bands of up to four
  // m tiles, so that the tiles of an XCD share rows of both operands in its L2.
  // (divisors and size[3]: factors and shifts of the divisions by the tiles of a band and by the m tiles of a full band; with pieces, from bit 10
  // on, 2^16 over the tiles, rounded up)
  const int m_tiles = (m + BM - 1) / BM, n_tiles = (n + BN - 1) / BN, gm = min(m_tiles, kBandRows);
  const FastDiv by_band = {(uint32_t)(gm * n_tiles), divisors[0], size[3] & 31u}, by_rows = {(uint32_t)gm, divisors[1], size[3] >> 5 & 31u};
  const int tiles = m_tiles * n_tiles, total = tiles * pieces, xcd = blockIdx.x & 7, each = total >> 3, rest = total & 7;
  int t = xcd * each + min(xcd, rest) + (int)(blockIdx.x >> 3), piece = 0;
  if (PIECES) {  // the slow index: an XCD reads one or two of them, and those of the last piece, which wait, come behind the others of their XCD
    piece = (int)((uint32_t)t * (size[3] >> 10) >> 16);
    t -= piece * tiles;
  }
  const int band = (int)fast_div(t, by_band), rem = t - band * gm * n_tiles;
  const int rows_here = min(gm, m_tiles - band * gm);
  const int tn = rows_here == gm ? (int)fast_div(rem, by_rows) : rem / rows_here;
  const int in_band = rem - tn * rows_here, m0 = (band * gm + in_band) * BM, n0 = tn * BN;
  const int wm = wave & 1, wn = wave >> 1;
  const int col0 = n0 + wn * (BN / 2);

  // Bias of the wave's features to LDS of its own (any fp32 address, so four bytes a lane)
  const uint32_t bias_at = STAGES * kStageBytes + wave * 512;
  if (bias) {
#pragma unroll
    for (int h = 0; h < (16 * NT + 63) / 64; ++h) {
      const float *src = bias + min(col0 + 64 * h + lane, n - 1);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(src), "s"(bias_at + 256 * h) : "m0");
    }
  }

  // Line loads of a wave: NT of 8 W rows each, then MT of 8 lhs rows, either run contiguous in LDS.  Staged W row
  // 32b + 16c + 4q + j of a half (c: block of a pair) holds feature 32b + 8q + 4c + j.  Rows past the end: the last one.
  const uint32_t row_bytes = 2 * (uint32_t)k;
  uint32_t voff[L];
#pragma unroll
  for (int s = 0; s < L; ++s) {
    const bool is_w = s < NT;
    const int nth = is_w ? s : s - NT, row = 8 * (is_w ? wave * NT + nth : wave * MT + nth) + (lane >> 3);
    int r = row;
    if (is_w) {
      const int half = row >= BN / 2 ? BN / 2 : 0, in = row - half, blk = in >> 4;
      if (blk < (NT & ~1)) r = half + (in & ~31) + 8 * ((in >> 2) & 3) + 4 * (blk & 1) + (in & 3);
    }
    r = min(r, is_w ? n - n0 - 1 : m - m0 - 1);
    voff[s] = (uint32_t)r * row_bytes + (((lane & 7) ^ ((row >> 1) & 7)) << 4) + 3072 - 1024 * (nth & 3);
  }
  const char *wbase = w + n0 * (size_t)row_bytes - 3072, *xbase = x + m0 * (size_t)row_bytes - 3072;
  const uint32_t wdst = __builtin_amdgcn_readfirstlane(wave * NT * 1024);
  const uint32_t xdst = __builtin_amdgcn_readfirstlane(BN * kStageRow + wave * MT * 1024);
  auto issue = [&](auto s_, const char *wk, const char *xk, uint32_t slot) {
    constexpr int s = decltype(s_)::value;
    constexpr bool is_w = s < NT;
    constexpr int nth = is_w ? s : s - NT;
    if constexpr (nth % 4 == 0)
      asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0" : : "s"(slot + (is_w ? wdst : xdst)), "n"(nth * 1024) : "m0", "scc");
    line_load<1024 * (nth % 4)>(voff[s], is_w ? wk : xk);
  };
  const int all_lines = k / kLineK;
  int w_addr[2], x_addr[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    w_addr[h] = stage_off(wn * (BN / 2) + i, 4 * h + cg);
    x_addr[h] = stage_off(BN + wm * (BM / 2) + i, 4 * h + cg);
  }
  f32x4_t acc[MT][NT];
  u32x4_t wf[2][NT], xf[2][MT];
  constexpr int NR = MT + NT, NM = MT * NT;
  auto read = [&](auto r_, int h, uint32_t at) {  // in the order of use
    constexpr int r = decltype(r_)::value;
    if constexpr (r == 0) wf[h][0] = lds_read_b128(lds, w_addr[h] + at);
    else if constexpr (r <= MT) xf[h][r - 1] = lds_read_b128(lds, x_addr[h] + at + (r - 1) * 16 * kStageRow);
    else wf[h][r - MT] = lds_read_b128(lds, w_addr[h] + at + (r - MT) * 16 * kStageRow);
  };
  constexpr int R1 = NR + 4 > NM ? 2 : 1;               // fragment reads of a slot
  constexpr int READ = (NR + R1 - 1) / R1 + 5;          // by this slot the reads of a phase have come back
  constexpr int PH = 2 * KS, BS = (PH - 2) * NM + (READ < NM ? READ : NM), DS = PH * NM - BS, NL = KS * L;
  using True = std::true_type;
  using False = std::false_type;
  [[maybe_unused]] bool alone = false;
  for (;;) {  // (once, unless a workgroup that has waited in vain for the sums of others makes them itself)
    // The order of the lines: each XCD begins at another eighth, and where W is the larger operand, in every group of 8, of 4 (tiles from 96 x 64 on) or
    // of 2 (from 128 x 160 on, and what divides k) each tile of those that share W rows at another place.  Not where a quarter of the last one is padding:
    // begun ahead of the others it stays there, and fetches for them.  Of a piece each tile begins elsewhere.
    int lines = all_lines;
    uint32_t from = 0, end = row_bytes, pos, turn = 0;
    if constexpr (PIECES) {
      const int first = piece * all_lines / pieces;
      lines = (piece + 1) * all_lines / pieces - first;
      from = (uint32_t)first * kStageRow;
      end = from + (uint32_t)lines * kStageRow;
      pos = from + ((uint32_t)t * (size[3] >> 10) * (uint32_t)lines >> 16) * kStageRow;
    } else {
      const bool padded = m_tiles <= kBandRows && 4 * (m - (m_tiles - 1) * BM) <= 3 * BM;
      pos = (((uint32_t)(xcd * lines) >> 3) + ((padded ? t : tn) & 3)) * kStageRow;
      if (pos >= row_bytes) pos = 0;
      constexpr int kGroup = L <= 4 ? 8 : L <= 8 ? 4 : 2;
      const int group = min(lines & -lines, kGroup);
      turn = padded || n < m ? 0u : (uint32_t)(group == 2 ? in_band & 1 : in_band * group >> (rows_here == 2 ? 1 : 2)) * kStageRow;
    }
    const int stages = (lines + KS - 1) / KS, last_lines = lines - (stages - 1) * KS;
    uint32_t kpos = pos ^ turn;
    auto advance = [&]() {
      pos = pos + kStageRow == end ? from : pos + kStageRow;
      kpos = pos ^ turn;
    };
#pragma unroll
    for (int s = 0; s < STAGES * KS; ++s) {
      static_for<0, L>([&](auto l) { issue(l, wbase + kpos, xbase + kpos, s * kLineBytes); });
      advance();
    }

#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < NT; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    uint32_t slot = 0;
    // Fragments of 32 k (half a line) are read while the MFMAs of the 32 before run.
    wait_loads<L * KS * (STAGES - 1)>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    static_for<0, NR>([&](auto r) { read(r, 0, 0); });
    // One stage.  LEFT: stages under way beyond the next one; LOAD: fetch another; NEXT: there is a next one.
    auto stage = [&](auto left, auto load, auto next_) {
      constexpr int LEFT = decltype(left)::value;
      constexpr bool LOAD = decltype(load)::value, NEXT = decltype(next_)::value;
      const uint32_t fetch = slot, next = slot + kStageBytes == STAGES * kStageBytes ? 0 : slot + kStageBytes;
      static_for<0, PH * NM>([&](auto j_) {
        constexpr int j = decltype(j_)::value, h = j / NM, q = j % NM;
        if (KS > 1 && !NEXT && h >= 2 && h / 2 >= last_lines) return;  // (the last stage may hold surplus lines)
        if constexpr (j == BS && NEXT) {
          wait_loads<L * KS * LEFT>();
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        static_for<0, R1>([&](auto r_) {
          constexpr int r = q * R1 + decltype(r_)::value;
          if constexpr (r < NR && (h < PH - 1 || NEXT))
            read(std::integral_constant<int, r>(), (h + 1) & 1, h == PH - 1 ? next : slot + (h + 1) / 2 * kLineBytes);
        });
        if constexpr (LOAD && j >= BS) {  // load l in slot BS + l * DS / NL
          constexpr int first = ((j - BS) * NL + DS - 1) / DS, end = ((j + 1 - BS) * NL + DS - 1) / DS;
          static_for<first, end>([&](auto l_) {
            constexpr int l = decltype(l_)::value;
            issue(std::integral_constant<int, l % L>(), wbase + kpos, xbase + kpos, fetch + l / L * kLineBytes);
            if (l % L == L - 1) advance();
          });
        }
        __builtin_amdgcn_sched_barrier(0);
        acc[q % MT][q / MT] = E::mfma16(wf[h & 1][q / MT], xf[h & 1][q % MT], acc[q % MT][q / MT]);
        __builtin_amdgcn_sched_barrier(0);
      });
      slot = next;
    };
    for (int s = STAGES; s < stages; ++s) stage(std::integral_constant<int, STAGES - 2>(), True(), True());
    static_for<0, STAGES>([&](auto u_) {
      constexpr int u = decltype(u_)::value, left = STAGES - 2 - u;
      if (stages - STAGES + u < 0) return;  // k of fewer stages than are kept
      stage(std::integral_constant<int, (left > 0 ? left : 0)>(), False(), std::integral_constant<bool, (u < STAGES - 1)>());
    });
    wait_loads<0>();  // (k of one stage: the surplus ones are still under way, and LDS is given up at the end)
    if constexpr (!PIECES) {
      break;
    } else {
      // The last piece's workgroup adds up: its own sums, then those of pieces 0, 1, ...  Every word of theirs goes past the XCD's L2 beside half
      // of the launch's number, and is looked at until the number is there.  They wait for nothing, and come before it in the order of
      // their XCD; launches of two streams can hold each other's workgroups up all the same, and so a look in vain has an end.
      f32x4_t &own = acc[0][0];
      const __amdgpu_buffer_rsrc_t words = byte_buffer(late.words + (size_t)t * pieces * kWordsBytes, (uint32_t)pieces * kWordsBytes);
      const uint32_t tag0 = (uint32_t)late.number, tag1 = (uint32_t)(late.number >> 32);
      if (!alone) {
        if (piece < pieces - 1) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            store_device(words, piece * kWordsBytes + h * (kWordsBytes / 2) + tid * 16,
                         __builtin_bit_cast(f32x4_t, u32x4_t{__builtin_bit_cast(uint32_t, (float)own[2 * h]), tag0,
                                                             __builtin_bit_cast(uint32_t, (float)own[2 * h + 1]), tag1}));
          return;
        }
        u32x4_t v[kMostPieces - 1][2];
        bool there;
        int looks = (int)late.looks;
        do {
          asm volatile("" ::: "memory");  // (the loads are made again)
          uint32_t differs = 0;
#pragma unroll
          for (int o = 0; o < kMostPieces - 1; ++o)
#pragma unroll
            for (int h = 0; h < 2; ++h)  // (past the others: past the buffer, and zero)
              v[o][h] = __builtin_bit_cast(u32x4_t, load_device(words, o < pieces - 1 ? o * kWordsBytes + h * (kWordsBytes / 2) + tid * 16 : 0x7fffff00));
#pragma unroll
          for (int o = 0; o < kMostPieces - 1; ++o)
#pragma unroll
            for (int h = 0; h < 2; ++h) differs |= o < pieces - 1 ? (v[o][h][1] ^ tag0) | (v[o][h][3] ^ tag1) : 0u;
          there = kLooks != 0 && __builtin_amdgcn_ballot_w64(differs != 0) == 0;
        } while (!there && --looks > 0);
#pragma unroll
        for (int o = 0; o < kMostPieces - 1; ++o)
          if (o < pieces - 1)
            own += f32x4_t{__builtin_bit_cast(float, (uint32_t)v[o][0][0]), __builtin_bit_cast(float, (uint32_t)v[o][0][2]),
                           __builtin_bit_cast(float, (uint32_t)v[o][1][0]), __builtin_bit_cast(float, (uint32_t)v[o][1][2])};
        volatile uint32_t *gave_up = reinterpret_cast<volatile uint32_t *>(lds + STAGES * kStageBytes + kBiasBytes);
        if (lane == 0) gave_up[wave] = !there;
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(gave_up[0] | gave_up[1] | gave_up[2] | gave_up[3]) == 0) break;
        alone = true;  // all pieces in the same order, the sum so far in the last one's place among the words
      } else {
        const int place = (pieces - 1) * kWordsBytes + tid * 16;
        if (piece != pieces - 1) own = load_device(words, place) + own;
        if (piece == pieces - 2) break;
        store_device(words, place, own);
        piece = piece == pieces - 1 ? 0 : piece + 1;
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // (nobody reads the lines of the piece before any more)
    }
  }
  if constexpr (MT * NT <= 2) {  // (two barriers and a way through LDS take longer there: 512 x 2048, 24 rows 4.56 / 4.70)
    const int row0 = m0 + wm * (BM / 2);
#pragma unroll
    for (int b = 0; b < NT; b += 2) {
      const bool two = b + 1 < NT;
      const int c = 16 * b + (two ? 8 : 4) * cg, col = col0 + c;
      f32x4_t b0 = {0.f, 0.f, 0.f, 0.f}, b1 = b0;
      if (bias) {
        b0 = *reinterpret_cast<const f32x4_t *>(lds + bias_at + 4 * c);
        if (two) b1 = *reinterpret_cast<const f32x4_t *>(lds + bias_at + 4 * c + 16);
      }
#pragma unroll
      for (int a = 0; a < MT; ++a) {
        const int row = row0 + 16 * a + i;
        const f32x4_t u = acc[a][b] + b0;
        uint16_t *o = out + (size_t)row * n + col;
        if (two) {
          const f32x4_t v = acc[a][b + 1 < NT ? b + 1 : b] + b1;
          if (row < m && col < n)
            *reinterpret_cast<u32x4_t *>(o) = u32x4_t{E::pack2(u[0], u[1]), E::pack2(u[2], u[3]), E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
        } else if (row < m && col < n) {
          *reinterpret_cast<u32x2_t *>(o) = u32x2_t{E::pack2(u[0], u[1]), E::pack2(u[2], u[3])};
        }
      }
    }
    return;
  }
  // The tile leaves as whole rows, by way of the lines' place (rows 16 bytes apart from a multiple of the banks), and past the L2, where they are whole
  // sectors: lines that are left there are written back at the end of the launch.  (Block of Qwen2.5-7B, 2048 tokens, us, pieces of 64 bytes and
  // ordinary stores / rows / rows past the L2: 174.5 / 173.8 / 170.6; 3584 x 3584, 2048 rows 43.05 / 42.65 / 41.9, 1536 x 1536 12.05 / 12.0 / 11.6.)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  constexpr int kRow = 2 * BN + 16;
  static_assert(BM * kRow <= STAGES * kStageBytes, "");
#pragma unroll
  for (int b = 0; b < NT; b += 2) {
    const bool two = b + 1 < NT;
    const int c = 16 * b + (two ? 8 : 4) * cg;
    f32x4_t b0 = {0.f, 0.f, 0.f, 0.f}, b1 = b0;
    if (bias) {
      b0 = *reinterpret_cast<const f32x4_t *>(lds + bias_at + 4 * c);
      if (two) b1 = *reinterpret_cast<const f32x4_t *>(lds + bias_at + 4 * c + 16);
    }
#pragma unroll
    for (int a = 0; a < MT; ++a) {
      char *at = lds + (wm * (BM / 2) + 16 * a + i) * kRow + (wn * (BN / 2) + c) * 2;
      const f32x4_t u = acc[a][b] + b0;
      if (two) {
        const f32x4_t v = acc[a][b + 1 < NT ? b + 1 : b] + b1;
        *reinterpret_cast<u32x4_t *>(at) = u32x4_t{E::pack2(u[0], u[1]), E::pack2(u[2], u[3]), E::pack2(v[0], v[1]), E::pack2(v[2], v[3])};
      } else {
        *reinterpret_cast<u32x2_t *>(at) = u32x2_t{E::pack2(u[0], u[1]), E::pack2(u[2], u[3])};
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  constexpr int kPieces = BN / 8;  // of a row
  const bool sectors = (a_[3] & 63) == 0 && n % 32 == 0;
#pragma unroll
  for (int j = 0; j < (BM * kPieces + kTileThreads - 1) / kTileThreads; ++j) {
    const int piece = tid + j * kTileThreads, r = piece / kPieces, c = piece - r * kPieces;
    if (r < BM && m0 + r < m && n0 + 8 * c < n) {
      const u32x4_t v = lds_read_b128(lds, r * kRow + 16 * c);
      uint16_t *o = out + (size_t)(m0 + r) * n + n0 + 8 * c;
      if (sectors) store_device_b128(o, v);
      else *reinterpret_cast<u32x4_t *>(o) = v;
    }
  }
}

struct TileCall {
  addresses_t a;  // lhs, W, bias, out
  int m, n, k;
  int pieces = 1;
  TilePieces late = {};
};

template <typename T, int MT, int NT, int KS, int STAGES, bool PIECES = false> hipError_t launch_tile(const TileCall &c, hipStream_t stream) {
  const int m_tiles = (c.m + 32 * MT - 1) / (32 * MT), n_tiles = (c.n + 32 * NT - 1) / (32 * NT);
  const int gm = m_tiles < kBandRows ? m_tiles : kBandRows;
  const FastDiv band = make_fast_div((uint32_t)(gm * n_tiles)), band_rows = make_fast_div((uint32_t)gm);
  constexpr int lds_bytes = STAGES * KS * 32 * (MT + NT) * kStageRow + kBiasBytes + (PIECES ? 16 : 0);
  static_assert(lds_bytes > 64 * 1024 && lds_bytes <= 160 * 1024, "");
  const auto kern = matmul_tile_kernel<T, MT, NT, KS, STAGES, PIECES>;
  std::conditional_t<PIECES, TilePieces, NoPieces> late;
  if constexpr (PIECES) late = c.late;
  static std::atomic<uint64_t> attr_done{0};  // more than 64 KiB of dynamic LDS is an opt-in per device and kernel
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (!(attr_done.load(std::memory_order_acquire) & bit)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return e;
    attr_done.fetch_or(bit, std::memory_order_release);
  }
  const uint32_t tiles = (uint32_t)(m_tiles * n_tiles);
  return launch(kern, dim3(tiles * c.pieces), kTileThreads, lds_bytes, stream, c.a,
                u32x4_t{(uint32_t)c.m, (uint32_t)c.n, (uint32_t)c.k | (uint32_t)c.pieces << 21,
                        band.l | band_rows.l << 5 | (65536u / tiles + 1) << 10},
                u32x2_t{band.m, band_rows.m}, late);
}

// Lhs rows, features, lines of a stage and stages of the tiles; see tile_kind for their order
#define LLMHIP_TILES(TILE)                                                                                            \
  TILE(1, 1, 4, 3) TILE(1, 1, 4, 4) TILE(2, 1, 2, 4) TILE(1, 2, 2, 5) TILE(2, 2, 1, 5) TILE(3, 2, 1, 5) TILE(2, 3, 1, 4) TILE(4, 2, 1, 4) \
  TILE(3, 3, 1, 4) TILE(3, 4, 1, 3) TILE(4, 3, 1, 4) TILE(4, 4, 1, 4) TILE(4, 5, 1, 4) TILE(4, 6, 1, 3) TILE(5, 5, 1, 3) \
  TILE(4, 7, 1, 3) TILE(5, 6, 1, 3) TILE(4, 8, 1, 3)
struct Tile {
  int m, n;
};
constexpr Tile kTiles[] = {
#define LLMHIP_TILE(MT, NT, KS, STAGES) {32 * MT, 32 * NT},
    LLMHIP_TILES(LLMHIP_TILE)
#undef LLMHIP_TILE
};
constexpr int kTileKinds = sizeof(kTiles) / sizeof(kTiles[0]), kDeep = 1, kTall = 2, kWide = 3;  // 32 x 32 with more stages, 64 x 32, 32 x 64
static_assert(kTiles[kTall].m == 2 * kTiles[kTall].n && kTiles[kWide].n == 2 * kTiles[kWide].m, "");

#ifndef LLMHIP_BENCH
template <typename T> hipError_t launch_kind(const TileCall &c, int kind, hipStream_t stream) {
  using Launch = hipError_t (*)(const TileCall &, hipStream_t);
  static constexpr Launch launch[] = {
#define LLMHIP_TILE(MT, NT, KS, STAGES) launch_tile<T, MT, NT, KS, STAGES>,
      LLMHIP_TILES(LLMHIP_TILE)
#undef LLMHIP_TILE
  };
  return launch[kind](c, stream);
}
#endif

// The smallest tile that needs no more workgroups than there are CUs: the chain of a workgroup is the shortest then.
// Over 270 sizes (16 weights of 256-11008 rows and k of 1536-18944, 17-4096 lhs rows, W from HBM) it takes 0.80 of hipBLASLt's
// time on average, before the lines went in turns.  Taken though slower, so that no such call needs hipBLASLt's handle and 64 MiB workspace (which a stream under
// capture cannot create): few rows over k = 8192, which hipBLASLt cuts (us, hipBLASLt / here: 1024 x 8192, 17 rows 11.8 / 15.4,
// 64 rows 13.8 / 17.5; 2048 x 8192, 24 rows 14.0 / 18.3; 4096 x 8192, 17 rows 17.2 / 17.2, 32 rows 18.3 / 20.3; not so 1536 x
// 8960, 17 rows 28.2 / 19.0, 3584 x 18944, 32 rows 109.6 / 48.4; 64 rows of 1024 x 8192 15.1 by now; 5120 x 5120, 64 rows 21.5 / 18.9, 4096 x 11008, 680 rows
// 80.5 / 71.3).  More than one round is not: 5120 x 5120, 2048 rows 100.5 / 101.4 with 128 x 160 tiles, 3584 x 3584, 2048 rows 54.4 /
// 54.5 with 128 x 128.
//   Of 64 x 32 and 32 x 64 the second where W is much the larger operand and next to nothing is padding: up to 4 tiles then share its rows,
// and not two (us, 64 x 32 / 32 x 64: 3584 x 3584, 128 rows 12.5 / 11.7, 5120 x 5120, 64 rows 23.1 / 19.0, with 320 workgroups; but
// 512 x 3584, 768 rows 9.5 / 9.9, 1536 x 1536, 256 rows 5.85 / 6.05, 3584 x 3584, 96 rows 11.4 / 12.5).
//   32 x 32 with a stage more where W rows are fetched by one tile alone, or by one that is ahead of another, and many CUs do so: the longer way
// to HBM wants more under way (3 / 4 stages: 3584 x 3584, 17 rows 9.4 / 9.25, 40 9.0 / 8.6; 4096 x 4096, 40 rows 9.55 / 9.1; 512 x 3584, 32 rows 6.3 / 6.5).
int tile_kind(int m, int n, int k) {
  const long long cus = device_compute_units();
  auto count = [&](int kind) {
    const Tile &t = kTiles[kind];
    return (long long)((m + t.m - 1) / t.m) * ((n + t.n - 1) / t.n);
  };
  if (count(0) <= cus) return m <= 56 && 4 * count(0) >= cus && 4 * ((m - 1) % 32 + 1) <= (m <= 32 ? 128 : 96) ? kDeep : 0;
  for (int kind = kTall; kind < kTileKinds; ++kind)
    if (count(kind) <= cus)
      return kind == kTall && n >= 16LL * m && count(kWide) <= cus && (m - 1) % 64 >= 56 ? kWide : kind;
  return -1;
}

}  // namespace

// k in whole stages; offsets inside a tile are 32 bits.
bool matmul_tile_takes(int m, int n, int k) {
  return k % kLineK == 0 && k <= 1 << 20 && tile_kind(m, n, k) >= 0;
}

// Few tiles of 32 x 32 over k of some thousands wait for a chain of 48 or more lines, and for the 30 to 45 GB/s that a CU gets from beyond its L2,
// while most CUs have nothing to do: k is cut into as many pieces as give every CU a workgroup, of at least 12 lines.  A piece's sums
// go past the L2 with tags and are added up by the workgroup of the last one: 2.2 us, a third of it the way there (us, whole / in
// pieces, W from HBM, then in the last-level cache: 1024 x 5120, 16 rows 9.5 / 6.6, 8.2 / 5.9, 32 14.2 / 7.0, 8.3 / 6.0, 64 12.05 / 7.8,
// 8.45 / 6.5, 128 10.9 / 9.8, 8.5 / 7.4; 512 x 3584, 9 rows 5.05 / 4.95, 4.8 / 4.9, 32 6.5 / 5.1, 64 6.3 / 5.4, 128 6.3 / 6.0; 3584 x 3584, 32 rows
// 10.9 / 9.0, 6.75 / 6.4; 4096 x 4096, 32 rows 11.45 / 9.4; but 8 rows, for which W is read in shares, 1024 x 5120 5.9 / 6.35, two pieces of
// fewer than 24 rows, where a part whose way past the L2s is 1 us longer gains nothing from HBM and loses from the cache, 3584 x 3584,
// 17 rows 9.25 / 9.25, 6.65 / 8.5 (32 there 10.8 / 9.7, 7.0 / 8.5; blocks of 30 and 32 rows gain 6 and 18 %), and k below
// 3072, 512 x 2048 4.4 / 4.6, 1536 x 1536 5.2 / 5.15, 3.75 / 4.7).  One line to a stage less and five stages: 3 to 10 % ahead of two or three of four
// lines.  Tiles that are larger have too much to pass on (64 x 128 over half of 3584: 18.5 us, of them 3.5).  The line at k = 6144 is not a
// measured one (whole, 1024 x 8192, 17 rows 15.4 us, hipBLASLt 11.8): from there on a call gives the same bits eager and captured, which below it does not.
int matmul_tile_pieces(int m, int n, int k) {
  const long long cus = device_compute_units(), tiles = (long long)((m + 31) / 32) * ((n + 31) / 32);
  if (m <= 8 || k % kLineK != 0 || k < 3072 || k >= 6144 || 2 * tiles > cus || tiles * cus >= 65536) return 1;
  const long long by_cus = cus / tiles, by_lines = k / kLineK / 12, pieces = by_cus < by_lines ? by_cus : by_lines;
  if (pieces == 2 && m < 24) return 1;
  return (int)(pieces < kMostPieces ? pieces : kMostPieces);
}
int matmul_tile_size(int m, int n, int k) {
  return matmul_tile_takes(m, n, k) ? kTiles[tile_kind(m, n, k)].m << 16 | kTiles[tile_kind(m, n, k)].n : 0;
}
size_t matmul_pieces_bytes(int m, int n, int pieces) { return (size_t)((m + 31) / 32) * ((n + 31) / 32) * pieces * kWordsBytes; }

hipError_t launch_matmul_tile(void *out, const void *lhs, const void *weight, const float *bias, int m, int n, int k,
                              int dt, hipStream_t stream, int pieces, void *workspace) {
  TileCall c = {{address(lhs), address(weight), address(bias), address(out)}, m, n, k};
  if (pieces > 1) {
    c.pieces = pieces;
    c.late = {static_cast<char *>(workspace), launch_number(), kLooks};
    return dt == kDtFloat16 ? launch_tile<_Float16, 1, 1, 2, 5, true>(c, stream) : launch_tile<__bf16, 1, 1, 2, 5, true>(c, stream);
  }
#ifdef LLMHIP_BENCH
  return hipErrorInvalidValue;
#else
  const int kind = tile_kind(m, n, k);
  return dt == kDtFloat16 ? launch_kind<_Float16>(c, kind, stream) : launch_kind<__bf16>(c, kind, stream);
#endif
}

}  // namespace LLMHIP_NS
