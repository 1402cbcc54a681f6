// Projection of many rows: out[m][n] = lhs[m][k] . W[n][k]^T + bias, fp32 accumulation, one rounding, for calls whose
// tiles fit the chip in one round (matmul_tile_takes); a launch that needs more is left to hipBLASLt.
//
// A workgroup computes one tile of 32*MT lhs rows x 32*NT features over all of k in stages of KS * 64 k (KS 128-byte
// lines of every operand row).  Lines travel global -> LDS without registers, STAGES of them in flight or in use; a
// fragment load straight into the operand layout, 16 rows by 64 bytes, ran at a third of the rate (512 x
// 3584, 2048 rows: 29.9 us against 14.3).  Eight waves: four quadrants of the tile, each shared by two waves that take 32 k
// of every line, so that a SIMD always has two waves; their sums are traded through LDS at the end.  The fragments of
// the next stage are read beside the MFMAs of this one, and loads and fragment reads are dealt out among the MFMAs
// one by one: issued in a burst they held the matrix unit up (3584 x 3584, 2048 rows, W from HBM: 53.2 -> 50.4 us).
// Where the time of a launch goes, by clock stamps in a copy of the kernel, us: 128 x 224 tile, k = 3584: 3.0 until the first
// lines are in, 56 stages of 0.69, 6.2 for the trade of the sums and the store, the rest launch.  A stage is 28 MFMAs of
// 16x16x32 for each of a SIMD's two waves, 0.52 at the 1.72 GHz that they leave; with zeros for lhs the clock stays at
// 2.28 GHz and a stage takes 0.51.  Small tiles are bound by the rate at which one CU takes lines in, 90-120 KB/us, and
// the barrier and LDS latency of a stage: 64 x 64 1.5, 56 of 0.175, 1.3; 32 x 32 1.1, 56 lines of 0.07 where their MFMAs take
// 0.02, 0.4 (two lines a stage: 512 x 3584, 100 rows 8.0 -> 7.4; larger tiles gain nothing by it).
//
// Rows of the operands lie k elements apart, often a multiple of 4 KiB: workgroups that walk k in step would ask few
// memory channels for everything.  Each XCD starts at another eighth of k, neighbouring tiles a stage apart
// (4096 x 4096, 1024 rows: 40 -> 36.6 us; 3584 x 3584, 2048 rows, W from HBM: 51.8 -> 49.5).
//
// bf16, us, hipBLASLt (without its 10 us of host time) / here, W from HBM: 3584 x 3584: 64 rows 13.2 / 11.0, 128 rows
// 21.6 / 15.0, 256 rows 19.8 / 18.6, 768 rows 33.1 / 29.4, 2048 rows 52.3 / 49.6; 512 x 3584: 100 rows 11.1 / 7.5,
// 2048 rows 17.7 / 14.4; 1536 x 1536: 128 rows 7.5 / 5.3; 5120 x 5120: 100 rows 24.3 / 22.1, 1280 rows 74.4 / 69.1.
#include <atomic>

#include "common.hpp"
#include "kernels.hpp"

namespace llmhip {

namespace {

constexpr int kTileWaves = 8;
constexpr int kLineK = 64;             // k of a 128-byte line of an operand row
constexpr int kStageRow = 2 * kLineK;  // its bytes

struct TileParams {
  const char *x, *w;
  const float *bias;
  uint16_t *out;
  int m, n, k;
  int m_tiles, n_tiles;
  FastDiv band, band_rows;  // tiles of a band, m tiles of a full band
};

// LDS offset of logical 16-byte granule g of a staged row
__device__ __forceinline__ int stage_off(int row, int g) { return row * kStageRow + ((g ^ ((row >> 1) & 7)) << 4); }

template <int N> __device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "i"(N) : "memory");
}

template <typename T, int MT, int NT, int KS, int STAGES>
__global__ __launch_bounds__(64 * kTileWaves, 2) void matmul_tile_kernel(TileParams p) {
  using E = Elem<T>;
  constexpr int BM = 32 * MT, BN = 32 * NT, NW = kTileWaves, F = MT * NT, HALF = (F + 1) / 2;
  constexpr int kLineBytes = (BM + BN) * kStageRow;       // one line of every row: W rows, then lhs rows
  constexpr int kStageBytes = KS * kLineBytes;
  constexpr int kInstr = (BM + BN) / 8;                   // an instruction fetches 8 rows
  constexpr int L = (kInstr + NW - 1) / NW;               // of a wave per line
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int i = lane & 15, cg = lane >> 4;

  // Workgroups are dealt round-robin to the 8 XCDs: each takes a run of tiles, and runs go through bands of up to four
  // m tiles, so that the tiles of an XCD share rows of both operands in its L2.
  const int total = p.m_tiles * p.n_tiles, xcd = blockIdx.x & 7, each = total >> 3, rest = total & 7;
  const int t = xcd * each + min(xcd, rest) + (int)(blockIdx.x >> 3);
  const int band = (int)fast_div(t, p.band), rem = t - band * (int)p.band.d, gm = (int)p.band_rows.d;
  const int rows_here = min(gm, p.m_tiles - band * gm);
  const int tn = rows_here == gm ? (int)fast_div(rem, p.band_rows) : rem / rows_here;
  const int m0 = (band * gm + rem - tn * rows_here) * BM, n0 = tn * BN;

  const size_t row_bytes = 2 * (size_t)p.k;
  const char *base[L];
  uint32_t voff[L], dst[L];
#pragma unroll
  for (int s = 0; s < L; ++s) {
    const int q = min(s * NW + wave, kInstr - 1);  // (a wave without an instruction of its own repeats the last)
    const int row = 8 * q + (lane >> 3);
    const bool is_w = 8 * q < BN;
    const int r = is_w ? min(row, p.n - n0 - 1) : min(row - BN, p.m - m0 - 1);  // rows past the end: the last one
    base[s] = is_w ? p.w + n0 * row_bytes : p.x + m0 * row_bytes;
    voff[s] = (uint32_t)r * (uint32_t)row_bytes + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    dst[s] = __builtin_amdgcn_readfirstlane(q * 8 * kStageRow);
  }
  auto issue = [&](int s, int stage, uint32_t slot) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff[s]), "s"(base[s] + (size_t)stage * kStageRow), "s"(slot + dst[s])
                 : "m0");
  };

  const int wm = wave & 1, wn = (wave >> 1) & 1, kg = wave >> 2;
  const int w_addr = stage_off(wn * (BN / 2) + i, 4 * kg + cg), x_addr = stage_off(BN + wm * (BM / 2) + i, 4 * kg + cg);
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // The fragments of stage s+1 are read while the MFMAs of stage s run, so that the place of stage s is free for
  // stage s + STAGES as soon as every wave has come to the barrier.
  const int lines = p.k / kLineK;
  int kpos = (int)((unsigned)(xcd * lines / 8 + (t & 3)) % (unsigned)lines);
  auto issue_line = [&](uint32_t place) {
#pragma unroll
    for (int l = 0; l < L; ++l) issue(l, kpos, place);
    kpos = kpos + 1 == lines ? 0 : kpos + 1;
  };
#pragma unroll
  for (int s = 0; s < STAGES * KS; ++s) issue_line(s * kLineBytes);
  uint32_t slot = 0;
  u32x4_t w0[KS][NT], x0[KS][MT], w1[KS][NT], x1[KS][MT];
  auto step = [&](int line, const u32x4_t (&wf)[KS][NT], const u32x4_t (&xf)[KS][MT], u32x4_t (&wnext)[KS][NT],
                  u32x4_t (&xnext)[KS][MT]) {
    wait_loads<L * KS * (STAGES - 2)>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const uint32_t fetch = slot;
    slot = slot + kStageBytes == STAGES * kStageBytes ? 0 : slot + kStageBytes;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const bool have = KS == 1 || line + u < lines;  // (the last stage may hold surplus lines)
#pragma unroll
      for (int b = 0; b < (NT > L ? NT : L); ++b) {
        if (b < L) issue(b, kpos, fetch + u * kLineBytes);
        if (b < NT) wnext[u][b] = lds_read_b128(lds, w_addr + slot + u * kLineBytes + b * 16 * kStageRow);
#pragma unroll
        for (int a = b; a < MT; a += NT)
          xnext[u][a] = lds_read_b128(lds, x_addr + slot + u * kLineBytes + a * 16 * kStageRow);
        __builtin_amdgcn_sched_barrier(0);
        if (b < NT && have) {
#pragma unroll
          for (int a = 0; a < MT; ++a) acc[a][b] = E::mfma16(wf[u][b], xf[u][a], acc[a][b]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      kpos = kpos + 1 == lines ? 0 : kpos + 1;
    }
  };
  wait_loads<L * KS * (STAGES - 1)>();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int u = 0; u < KS; ++u) {
#pragma unroll
    for (int a = 0; a < MT; ++a) x0[u][a] = lds_read_b128(lds, x_addr + u * kLineBytes + a * 16 * kStageRow);
#pragma unroll
    for (int b = 0; b < NT; ++b) w0[u][b] = lds_read_b128(lds, w_addr + u * kLineBytes + b * 16 * kStageRow);
  }
  for (int line = 0; line < lines; line += 2 * KS) {
    step(line, w0, x0, w1, x1);
    if (line + KS < lines) step(line + KS, w1, x1, w0, x0);
  }

  wait_loads<0>();  // the loads past the last stage (k from its start again) still aim at the places written next
  // The two waves of a quadrant trade halves of their sums, and each rounds and stores the half it keeps.
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  f32x4_t *pieces = reinterpret_cast<f32x4_t *>(lds) + lane;
#pragma unroll
  for (int f = 0; f < F; ++f)
    if ((f >= HALF) == (kg == 0)) pieces[((wave & 3) * F + f) * 64] = acc[f / NT][f % NT];
  __syncthreads();
#pragma unroll
  for (int f = 0; f < F; ++f) {
    if ((f >= HALF) == (kg == 0)) continue;  // (wave-uniform)
    const int row = m0 + wm * (BM / 2) + (f / NT) * 16 + i, col = n0 + wn * (BN / 2) + (f % NT) * 16 + 4 * cg;
    f32x4_t sum = acc[f / NT][f % NT] + pieces[((wave & 3) * F + f) * 64];
    if (row >= p.m || col >= p.n) continue;
    if (p.bias) {
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += p.bias[col + j];
    }
    *reinterpret_cast<u32x2_t *>(p.out + (size_t)row * p.n + col) = u32x2_t{E::pack2(sum[0], sum[1]), E::pack2(sum[2], sum[3])};
  }
}

template <typename T, int MT, int NT, int KS, int STAGES> hipError_t launch_tile(TileParams &p, hipStream_t stream) {
  p.m_tiles = (p.m + 32 * MT - 1) / (32 * MT);
  p.n_tiles = (p.n + 32 * NT - 1) / (32 * NT);
  const int gm = p.m_tiles < 4 ? p.m_tiles : 4;
  p.band = make_fast_div((uint32_t)(gm * p.n_tiles));
  p.band_rows = make_fast_div((uint32_t)gm);
  constexpr int stage_bytes = STAGES * KS * 32 * (MT + NT) * kStageRow, piece_bytes = 4 * MT * NT * 1024;
  constexpr int lds_bytes = stage_bytes > piece_bytes ? stage_bytes : piece_bytes;
  static_assert(lds_bytes <= 160 * 1024, "");
  void (*kern)(TileParams) = matmul_tile_kernel<T, MT, NT, KS, STAGES>;
  if (lds_bytes > 64 * 1024) {  // an opt-in per device and kernel
    static std::atomic<uint64_t> attr_done{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(attr_done.load(std::memory_order_acquire) & bit)) {
      e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
      if (e != hipSuccess) return e;
      attr_done.fetch_or(bit, std::memory_order_release);
    }
  }
  hipLaunchKernelGGL(kern, dim3(p.m_tiles * p.n_tiles), dim3(64 * kTileWaves), lds_bytes, stream, p);
  return hipGetLastError();
}

template <typename T> hipError_t launch_kind(TileParams &p, int kind, hipStream_t stream) {
  switch (kind) {
    case 0: return launch_tile<T, 1, 1, 2, 4>(p, stream);
    case 1: return launch_tile<T, 2, 1, 1, 6>(p, stream);
    case 2: return launch_tile<T, 2, 2, 1, 6>(p, stream);
    case 3: return launch_tile<T, 3, 2, 1, 5>(p, stream);
    case 4: return launch_tile<T, 4, 2, 1, 4>(p, stream);
    case 5: return launch_tile<T, 3, 3, 1, 4>(p, stream);
    case 6: return launch_tile<T, 3, 4, 1, 4>(p, stream);
    case 7: return launch_tile<T, 4, 4, 1, 4>(p, stream);
    case 8: return launch_tile<T, 4, 5, 1, 4>(p, stream);
    case 9: return launch_tile<T, 4, 6, 1, 3>(p, stream);
    case 10: return launch_tile<T, 4, 7, 1, 3>(p, stream);
    default: return launch_tile<T, 4, 8, 1, 3>(p, stream);
  }
}

// The smallest tile that needs no more workgroups than there are CUs: the chain of a workgroup is the shortest then.
// (Twelve tiles rather than eight fill the round better; us, hipBLASLt / here: 3584 x 3584, 320 rows 22.8 / 19.7, 768 rows
// 33.1 / 29.4, 1280 rows 43.3 / 39.2; 5120 x 5120, 900 rows 62.6 / 56.9.  128 x 96 and 64 x 96 are slower than 96 x 128 and
// 96 x 64: 640 rows 31.3 / 28.6, 200 rows of 5120 30.4 / 28.2.)
// From 96 x 64 on hipBLASLt, which cuts k too, is the faster one where that leaves a fifth of the CUs idle: 5120 x 5120, 640
// rows (78 % busy) 51.5 us against 53.7, 768 rows (94 %) 53.3 / 53.2, 900 rows (100 %) 62.6 / 56.9.  Not so up to k = 2048,
// where the start of a workgroup weighs more: 1536 x 1536, 768 rows (56 %) 12.4 / 11.2.  And from 128 x 192 on where rows are a
// multiple of 4 KiB apart: 4096 x 4096, 1280 rows 46.6 / 47.6, 1500 rows 49.7 / 53.7, against 3584 x 3584, 1500 rows 44.2 /
// 42.7, 2048 rows 52.4 / 50.7; 8192 x 8192, 2000 rows 175 / 182.
// hipBLASLt's time is no smooth function of the rows, so that the two cross more often than these lines say.  Left to it
// though tiles would be faster: 3584 x 3584, 257-288 rows 29.5 / 23.1, 577-672 32.0 / 29.6, 865-896 35.5 / 34.0; 4096 x 4096,
// 513-576 rows 35.3 / 32.7; 1024 x 5120, 1025-1152 rows 28.3 / 26.6.  Taken though slower: 3584 x 3584, 784-864 rows 29.2 /
// 31.5; 5120 x 5120, 64-80 rows 21.7 / 24.2, 257-272 30.9 / 33.2, 528-560 41.6 / 45.0; 1024 and 2048 x 8192, 17-32 rows
// 11.7-16.2 / 18-22 (a quarter of the CUs, rows a multiple of 4 KiB apart).
int tile_kind(int m, int n, int k) {
  static const struct { int m, n; } tiles[] = {{32, 32},  {64, 32},   {64, 64},   {96, 64},   {128, 64},  {96, 96},
                                               {96, 128}, {128, 128}, {128, 160}, {128, 192}, {128, 224}, {128, 256}};
  const long long cus = device_compute_units();
  for (int kind = 0; kind < 12; ++kind) {
    const long long count = (long long)((m + tiles[kind].m - 1) / tiles[kind].m) * ((n + tiles[kind].n - 1) / tiles[kind].n);
    if (count > cus) continue;
    if (kind >= 3 && k > 2048 && 5 * count <= 4 * cus) return -1;
    if (kind >= 9 && k % 2048 == 0) return -1;
    return kind;
  }
  return -1;
}

}  // namespace

// k in whole stages; offsets inside a tile are 32 bits.
bool matmul_tile_takes(int m, int n, int k) {
  return k % kLineK == 0 && k <= 1 << 20 && tile_kind(m, n, k) >= 0;
}

hipError_t launch_matmul_tile(void *out, const void *lhs, const void *weight, const float *bias, int m, int n, int k,
                              int dt, hipStream_t stream) {
  TileParams p;
  p.x = static_cast<const char *>(lhs);
  p.w = static_cast<const char *>(weight);
  p.bias = bias;
  p.out = static_cast<uint16_t *>(out);
  p.m = m;
  p.n = n;
  p.k = k;
  const int kind = tile_kind(m, n, k);
  return dt == kDtFloat16 ? launch_kind<_Float16>(p, kind, stream) : launch_kind<__bf16>(p, kind, stream);
}

}  // namespace llmhip
