// Projection of few rows (one generated token, a handful of tokens): out[m][n] = lhs[m][k] . W[n][k]^T + bias,
// fp32 accumulation, one rounding, m <= 16 (from 9 rows on only where W has few rows: the tiled kernel is faster
// beyond, lines and figures in matmul_common).
//
// Bound by reading W once.  W is dealt out in equal shares of whole rows (at most 16) to one workgroup per
// CU, two or more rounds of them for a wide n: a CU cannot have more than its 32 KiB of first-level cache
// in flight (about 30 GB/s), so a matrix is only read at full speed if every CU has the same share of it --
// with 16 rows per workgroup 512 x 3584 ran on 32 CUs in 6.0 us, with 2 rows on all 256 it took 4.2 (3.35 now).
// The eight waves of a workgroup deal k out among themselves, and the partial sums meet in LDS.
//
// mfma_f32_16x16x32 takes 16 rows of 32 k; read that way every load instruction would touch half a
// cache line of 16 rows.  With at most 8 lhs rows the operand rows are instead 8 rows of W at two
// neighbouring k slices (KS = 2) and the operand columns the lhs rows at the same two slices: a load covers
// whole 128-byte lines of 8 rows, of the result the two diagonal blocks are wanted.  3584 x 3584, one
// row: 6.2 us from HBM (non-temporal loads) against 6.8 with KS = 1; KS = 4 is no better.  For 9..16
// rows KS = 1, and ordinary loads, because the second half of a line is asked for by the next instruction.
//
// Where a workgroup has at most 8 W rows (TW = 1; 2 with more) it is not the stream but one wave's chain that counts: all
// loads of a wave go out before its first MFMA, as many units B as its share of k has, up to 12 (one lhs row, W from HBM, us,
// four units at a time and a second, empty group of rows / this: 512 x 3584 4.13 / 3.68, 1024 x 5120 5.45 / 4.65, 256 x 1536
// 2.97 / 2.82, 2048 x 11008, in several rounds of 8, 11.45 / 10.62).  With more rows the stream is what counts, and four units of
// two groups are what a CU can have under way (3584 x 3584, two / four / six / eight 7.07 / 6.25 / 6.67 / 6.28).
//
// Over a k of more than 12 units there are several passes, and the lhs, which every workgroup reads whole, comes with each: eight
// units at a time with few rows, four with many (us, eight / four: one row of 1536 x 8960 6.93 / 7.46, 512 x 18944 9.19 / 10.93; 5 rows of
// 1024 x 8192 6.78 / 6.94; 4 rows of 2048 x 8960 9.67 / 8.83, 6 of 2048 x 13824 14.46 / 13.00, 8 of 1536 x 8960 9.83 / 9.19).  The line is a
// product of lhs rows and W rows per workgroup, from 280 sizes of 1-8 rows, 512-2048 W rows, k of 6160-18944: 20, or 32 with 14 to 16
// units (two passes with little left over: 4 rows of 2048 x 7168 7.35 / 7.57, of 2048 x 6160, 13 units, 7.62 / 7.17).
//
// EXACT: k is a multiple of 512, so that every wave has the same units, and nothing is asked for or left out under a mask: a
// mask and a branch to each load were 190 of the 270 instructions before the first MFMA, and a wave issues one in 4-5 cycles (us, with
// masks and the bias fetched at the end / this: 512 x 3584 3.50 / 3.35, 3584 x 3584 6.03 / 5.90, 1024 x 5120 4.48 / 4.32, 5120 x 5120, two
// passes of five units, 11.05 / 10.05, 18944 x 3584 23.0 / 21.2, 1536 x 1536 3.13 / 2.99; eight rows 4096 x 4096 8.16 / 7.93).  Not
// where it takes more passes than two, nor two of more than five units: they end and begin all at once (1024 x 8192, two of eight
// 5.68 / 5.90; 4096 x 7168, two of seven 10.87 / 11.45; 4096 x 6144, two of six 9.65 / 10.32, 8 rows 11.39 / 11.53, 8192 x 6144 17.0 / 17.4,
// three of four 9.74 / 9.91; 4096 x 10240, four of five 15.2 / 15.9).  As one pass takes up to eight units, two passes are a k of 5120.
#include "common.hpp"
#include "kernels.hpp"

namespace llmhip {

namespace {

constexpr int kSkinnyWaves = 8;

// KS k-slices per MFMA: operand row (column) index i stands for W (lhs) row i % (16/KS) at slice
// i / (16/KS).  TW groups of 16/KS W rows; B units of 32*KS k per wave and pass.  rows: W rows of a workgroup, at most 16.
// a: lhs, W, bias, out; size: m, n, k, rows.
template <typename T, int KS, int TW, int B, bool EXACT>
__global__ __launch_bounds__(64 * kSkinnyWaves, 4) void matmul_skinny_kernel(addresses_t a, u32x4_t size) {
  using E = Elem<T>;
  const uint16_t *x = at_address<const uint16_t>(a[0]), *w = at_address<const uint16_t>(a[1]);
  const float *bias = at_address<const float>(a[2]);
  uint16_t *out = at_address<uint16_t>(a[3]);
  const int m = size[0], n = size[1], k = size[2], row_share = size[3];
  constexpr int NW = kSkinnyWaves, R = 16 / KS, UK = 32 * KS;
  __shared__ __attribute__((aligned(16))) float red[NW * TW * 256];  // [wave][group of R rows][lane] of f32x4
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int i = lane & 15, cg = lane >> 4, r = i % R;
  const int n0 = blockIdx.x * row_share;
  const int rows = min(row_share, n - n0);
  const int koff = 32 * (i / R) + 8 * cg;
  f32x4_t acc[TW];
#pragma unroll
  for (int t = 0; t < TW; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // The result that this thread will write: feature n0 + f of lhs row `row`.  Its bias is asked for beside the operands, not when the
  // sum is there.
  const int f = tid & 15, row = tid >> 4;
  const bool writes = f < rows && row < m;
  float bias_here = 0.0f;
  if constexpr (EXACT) {
    // What rows past the share or past m hold reaches no result: they read the last (first) one again.
    const char *wb = reinterpret_cast<const char *>(w + (size_t)n0 * k + wave * UK), *xb = reinterpret_cast<const char *>(x + wave * UK);
    uint32_t wo[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) wo[t] = 2 * ((uint32_t)min(t * R + r, rows - 1) * k + koff);
    const uint32_t xo = 2 * ((uint32_t)(r < m ? r : 0) * k + koff);
    constexpr int kPass = 2 * NW * UK * B;
    for (int left = 2 * k; left > 0; left -= kPass, wb += kPass, xb += kPass) {
      u32x4_t wf[B][TW], xf[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int t = 0; t < TW; ++t) wf[b][t] = global_load_b128_nt(wb + b * (2 * NW * UK) + wo[t]);
        xf[b] = global_load_b128(xb + b * (2 * NW * UK) + xo);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (bias && writes && left == 2 * k) bias_here = bias[n0 + f];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int t = 0; t < TW; ++t) acc[t] = E::mfma16(wf[b][t], xf[b], acc[t]);
    }
  } else {
    if (bias && writes) bias_here = bias[n0 + f];
    const uint16_t *wp[TW];
#pragma unroll
    for (int t = 0; t < TW; ++t) wp[t] = w + (size_t)(n0 + min(t * R + r, rows - 1)) * k + koff;
    const bool xv = r < m;
    const uint16_t *xp = x + (size_t)(xv ? r : 0) * k + koff;
    const int units = (k + UK - 1) / UK;
    const u32x4_t zero = {0u, 0u, 0u, 0u};
    for (int u0 = wave; u0 < units; u0 += NW * B) {
      u32x4_t wf[B][TW], xf[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int kk = (u0 + b * NW) * UK;
        const bool in = kk + koff < k;  // k is a multiple of 16, a fragment 8 long
#pragma unroll
        for (int t = 0; t < TW; ++t) {
          wf[b][t] = zero;
          if (in && t * R + r < rows) wf[b][t] = KS > 1 ? global_load_b128_nt(wp[t] + kk) : global_load_b128(wp[t] + kk);
        }
        xf[b] = zero;
        if (in && xv) xf[b] = global_load_b128(xp + kk);
      }
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int t = 0; t < TW; ++t) acc[t] = E::mfma16(wf[b][t], xf[b], acc[t]);
    }
  }
  f32x4_t *slots = reinterpret_cast<f32x4_t *>(red);
#pragma unroll
  for (int t = 0; t < TW; ++t) slots[(wave * TW + t) * 64 + lane] = acc[t];
  __syncthreads();
  if (!writes) return;
  float sum = 0.0f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int ar = s * R + f % R, col = s * R + row;
    const float *src = red + ((f / R) * 64 + (ar >> 2) * 16 + col) * 4 + (ar & 3);
#pragma unroll
    for (int v = 0; v < NW; ++v) sum += src[v * TW * 256];
  }
  if (bias) sum += bias_here;
  out[(size_t)row * n + n0 + f] = E::round(sum);
}

using SkinnyKernel = void (*)(addresses_t, u32x4_t);
// The EXACT kernel of so many units a pass; none beyond what a wave has registers for.
template <typename T, int TW, int B = TW == 1 ? 12 : 8> SkinnyKernel exact_kernel(int units) {
  if (units == B) return matmul_skinny_kernel<T, 2, TW, B, true>;
  if constexpr (B > 1) return exact_kernel<T, TW, B - 1>(units);
  return nullptr;
}
constexpr int kTwoPassUnits = 5;  // of a pass, where there are two

template <typename T> SkinnyKernel kernel_of(int m, int k, int rows) {
  if (m > 8) return matmul_skinny_kernel<T, 1, 1, 8, false>;
  const int round = 64 * kSkinnyWaves, units = (k + round - 1) / round;  // of a wave
  if (k % round == 0) {
    if (const SkinnyKernel one = rows <= 8 ? exact_kernel<T, 1>(units) : exact_kernel<T, 2>(units)) return one;
    if (rows > 8 && units % 2 == 0 && units / 2 <= kTwoPassUnits) return exact_kernel<T, 2>(units / 2);
  }
  if (rows > 8) return matmul_skinny_kernel<T, 2, 2, 4, false>;
  if (units <= 4) return matmul_skinny_kernel<T, 2, 1, 4, false>;
  if (units <= 8) return matmul_skinny_kernel<T, 2, 1, 8, false>;
  if (units <= 12) return matmul_skinny_kernel<T, 2, 1, 12, false>;
  // Several passes: of eight units while a workgroup has few results, a little longer where two passes hold nearly all of k
  return m * rows <= (units >= 14 && units <= 16 ? 32 : 20) ? matmul_skinny_kernel<T, 2, 1, 8, false> : matmul_skinny_kernel<T, 2, 1, 4, false>;
}

}  // namespace

hipError_t launch_matmul_skinny(void *out, const void *lhs, const void *weight, const float *bias, int m, int n,
                                int k, int dt, hipStream_t stream) {
  const int cus = device_compute_units();
  const int rounds = (n + 16 * cus - 1) / (16 * cus);
  const int rows = (n + rounds * cus - 1) / (rounds * cus);
  const SkinnyKernel kern = dt == kDtFloat16 ? kernel_of<_Float16>(m, k, rows) : kernel_of<__bf16>(m, k, rows);
  return launch(kern, dim3((n + rows - 1) / rows), 64 * kSkinnyWaves, 0, stream,
                addresses_t{address(lhs), address(weight), address(bias), address(out)},
                u32x4_t{(uint32_t)m, (uint32_t)n, (uint32_t)k, (uint32_t)rows});
}

}  // namespace llmhip
