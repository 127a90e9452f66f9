// RMSNorm+linear, gated MLP and linear(+residual) on the matrix-product
// kernel: the choice of tile and K splits, the row pass of RMSNorm for many
// rows, and the launches.
#include "gemm.h"

#include "gemm_kernel.h"

namespace yr {
namespace gm {

// ---------------------------------------------------------------- RMSNorm row pass
// rs[row] = rsqrt(mean(x[row]^2) + eps) and, with a gamma, xg = x * gamma
// rounded to the storage type (the operand the fused kernels form in LDS).
// One workgroup per row, 16-byte accesses; bound by its two streams.
template <int DT>
__global__ __launch_bounds__(256) void norm_rows_kernel(const uint16_t* x, const uint16_t* gamma, uint16_t* xg,
                                                        float* rs, int K, float eps) {
  const uint16_t* xr = x + (size_t)blockIdx.x * K;
  uint16_t* gr = xg + (size_t)blockIdx.x * K;
  float ss = 0.f;
  for (int k = threadIdx.x * 8; k < K; k += 256 * 8) {
    const uint4 v = ldg16(xr + k);
    ss = sumsq8<DT>(v, ss);
    if (gamma) stg16(gr + k, scale8<DT>(v, ldg16(gamma + k)));
  }
  ss = wave_sum(ss);
  __shared__ float part[4];
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = ss;
  __syncthreads();
  if (threadIdx.x == 0) rs[blockIdx.x] = rsqrtf((part[0] + part[1] + part[2] + part[3]) / (float)K + eps);
}

// ---------------------------------------------------------------- plan
struct Plan {
  int cfg, splits, tm, tn;
  bool pass;  // RMSNorm row pass first
};

struct CfgShape {
  int bm, bn, per_cu;
};
constexpr CfgShape kCfg[kNumCfg] = {{32, 64, 2},   {32, 128, 2},  {64, 128, 1}, {128, 128, 1},
                                    {128, 192, 1}, {128, 256, 1}, {256, 256, 1}};
constexpr int kCus = 256;
// RMSNorm: the tiles of up to 64 rows scale x in LDS; up to 64 rows that is
// always the faster way, beyond 256 rows never, between them the cheaper by
// the model below (71 rows, K 2992, N 3728: 14.9 us against 18.7 with the row
// pass; 174 rows, K 2928, N 14280: 58.4 against 31.9).  The row pass counts
// with what such a call takes beyond the model's time for its product (741
// shapes of 65..315 rows, least squares): 6.3 us and its two streams of x at a
// rate that holds the product model's own error at these sizes.
constexpr int kNormLdsAlways = 64, kNormLdsMax = 256;
constexpr float kRowPassUs = 6.3f, kRowPassTbs = 1.1f;
constexpr int kPanelRows = 8192;   // rows per launch
// A stream keeps the largest workspace it has needed, so scratch is bounded:
// the row pass's copy of x (fewer rows per launch where K is long) and the
// records of the K splits (one per CU of the largest tile).
// Records past 64 MiB were no gain either (1654 rows, RMSNorm 6648 x 11848: 379
// us with two splits of 256 x 256 tiles, 318 without; 1730 rows, gated 14192 x
// 3376: 403 with four, 280 without).
constexpr size_t kPassBytes = 128u << 20, kSplitBytes = 64u << 20;

// Microseconds of one 64-k chunk of a tile, alone on its CU and with as many
// workgroups per CU as fit, its factor for K x N weights, and the terms around
// it: start, memory TB/s, a K split's merge (fixed, per 64 KB of records, per
// split) and the slowdown of a full chip.  The model only ranks.  Linear and
// gated are fitted to calls that repeat their weights, which partly stay in the
// cache; where the weights come from HBM the plan is on average 3.9 % (linear,
// 1176 shapes of 2..2048 rows, K and N 720..14264) and 4.0 % (gated, 2007)
// slower than the fastest, 18 and 17 % at the 95th percentile, 45 % at worst.
struct Cost {
  float chunk[kNumCfg], chunk_full[kNumCfg], kn[kNumCfg];
  float start, tbs, merge0, merge_rec, merge_split, load;
};
constexpr Cost kCostLinear = {{0.139f, 0.308f, 0.366f, 0.426f, 0.507f, 0.612f, 0.846f},
                        {0.321f, 0.617f, 0.366f, 0.426f, 0.507f, 0.612f, 0.846f},
                        {1.101f, 0.853f, 0.965f, 1.140f, 1.159f, 1.135f, 1.099f},
                        1.84f, 7.71f, 1.33f, 0.760f, 0.150f, 0.312f};
constexpr Cost kCostGated = {{0.f, 0.328f, 0.401f, 0.464f, 0.f, 0.772f, 1.330f},  // 0: no tile of the gated MLP
                        {0.f, 0.645f, 0.401f, 0.464f, 0.f, 0.772f, 1.330f},
                        {0.f, 1.012f, 0.973f, 1.234f, 0.f, 1.095f, 0.992f},
                        1.67f, 6.88f, 1.25f, 0.666f, 0.147f, 0.176f};
// RMSNorm in LDS is fitted to weights that come from HBM, as those of a model's
// layers do (2410 shapes of 2..315 rows, every tile and split count): 1.0 % on
// average, 5 % at the 95th percentile, 27 % at worst (5.8, 25 and 65 % with one
// memory rate for all tiles: it left a quarter of the chip idle where one more
// split fills it.  8 rows, 4096 x 4096 K x N: 3 splits 12.7 us, 4 12.2; the same
// weights again 11.2 and 10.7).
constexpr Cost kCostNorm = {{0.252f, 0.370f, 0.497f},
                        {0.374f, 0.370f, 0.497f},
                        {1.073f, 1.002f, 0.956f},
                        3.624f, 7.08f, 1.135f, 0.499f, 0.156f, 0.329f};
// its memory rate by layout (N x K, K x N) and tile, and what uneven rounds of
// the chip add to the memory time (with less than a workgroup per CU, and more)
constexpr float kNormTbs[2][3] = {{5.609f, 5.669f, 4.600f}, {5.643f, 6.344f, 4.912f}};
constexpr float kNormFew = 0.458f, kNormUneven = 0.665f;

// Scratch after the tickets: row factors and scaled x of the row pass, then
// the records of the K splits.
static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
static size_t pass_bytes(const Plan& p, int M, int K) {
  return p.pass ? align256((size_t)M * 4) + align256((size_t)M * K * 2) : 0;
}
static size_t split_bytes(int cfg, long tiles, int splits, bool lds_norm) {
  const CfgShape& s = kCfg[cfg];
  // one float4 more per thread where a normalising tile also adds row sums
  const size_t rec = (size_t)s.bm * s.bn * 4 + (lds_norm ? 512 * 16 : 0);
  return splits > 1 ? (size_t)tiles * splits * rec : 0;
}

// The best plan of one kind (`pass`: RMSNorm with its row pass) and its time;
// `staged`: of the tiles that load through registers, with at most `most`
// bytes of records.
static Plan best_plan(int M, int K, int N, int epi, bool nkl, bool pass, float* time, bool staged = false,
                      size_t most = 0) {
  Plan best = {};
  best.pass = pass;
  const bool lds_norm = epi == EPI_RMSNORM && !pass;
  const Cost& c = lds_norm ? kCostNorm : epi == EPI_GATED ? kCostGated : kCostLinear;
  const int nmat = epi == EPI_GATED ? 2 : 1, chunks = (K + KS - 1) / KS;
  const float mbytes = 2e-6f * ((float)nmat * K * N + (float)M * K + (float)M * N);
  const int least = lds_norm ? 3 : 5;  // chunks per split (a deep pipeline has to fill)
  float best_t = 3e38f;
  for (int f = 0; f < kNumCfg; f++) {
    const CfgShape& s = kCfg[f];
    if (epi == EPI_GATED && (f == C32x64 || f == C128x192)) continue;
    if (lds_norm && f > C64x128) break;
    if (pass && f <= C64x128) continue;
    if (staged && f != C32x128 && f != C64x128) continue;
    if (s.bm > 32 && s.bm >= 2 * M && !pass) break;  // a smaller tile holds every row
    if ((size_t)K * 2 * (M < s.bm ? M : s.bm) >= kOob) break;  // 32-bit offsets within a tile's rows of x
    const int tm = (M + s.bm - 1) / s.bm, tn = (N + s.bn / nmat - 1) / (s.bn / nmat);
    const long tiles = (long)tm * tn;
    // two workgroups per CU need two times their LDS: the normalising 32 x
    // 128 tile holds a fourth stage instead
    const int per_cu = lds_norm && f == C32x128 ? 1 : s.per_cu;
    const float kf = nkl ? 1.f : c.kn[f];
    for (int sp = 1; sp <= kMaxSplits; sp++) {
      // no empty split, and no more workgroups than a second round of the chip holds
      if (sp > 1 && (chunks < least * sp || tiles * sp > 4 * kCus || tiles > kMaxTickets)) break;
      const int per = (chunks + sp - 1) / sp;
      if ((chunks + per - 1) / per != sp) continue;
      if (split_bytes(f, tiles, sp, lds_norm) > (staged ? most : kSplitBytes)) continue;
      const long wg = tiles * sp, cap = (long)kCus * per_cu, rounds = wg / cap, rest = wg % cap;
      float t = rounds * (per_cu > 1 ? c.chunk_full[f] : c.chunk[f]);
      if (rest) t += rest <= kCus ? c.chunk[f] : c.chunk_full[f];
      t *= per * kf * (1.f + c.load * (wg < kCus ? (float)wg / kCus : 1.f));
      float mem = mbytes / c.tbs;
      if (lds_norm) {
        const float uneven = (float)((wg + kCus - 1) / kCus * kCus) / wg - 1.f;  // the fullest CU over the average
        mem = mbytes / kNormTbs[nkl ? 0 : 1][f] * (1.f + (wg < kCus ? kNormFew : kNormUneven) * uneven);
      }
      t = c.start + (t > mem ? t : mem);
      const float rec = s.bm * s.bn * 4.f;  // bytes of a split's record
      if (sp > 1) t += c.merge0 + sp * (c.merge_rec * rec / 65536 + c.merge_split) + 2e-6f * wg * rec / c.tbs;
      if (t < best_t) {
        best_t = t;
        best.cfg = f;
        best.splits = sp;
        best.tm = tm;
        best.tn = tn;
      }
    }
  }
  *time = best_t + (pass ? kRowPassUs + 4e-6f * M * K / kRowPassTbs : 0.f);
  return best;
}

static Plan make_plan(int M, int K, int N, int epi, bool nkl) {
  float t0 = 0.f, t1 = 0.f;
  if (epi != EPI_RMSNORM || M <= kNormLdsAlways || (size_t)M * K * 2 > kPassBytes)
    return best_plan(M, K, N, epi, nkl, false, &t0);
  const Plan p = best_plan(M, K, N, epi, nkl, true, &t1);
  if (M > kNormLdsMax) return p;
  const Plan q = best_plan(M, K, N, epi, nkl, false, &t0);
  return t0 < t1 ? q : p;
}

static size_t plan_bytes(const Plan& p, int M, int K, int epi) {
  const size_t more =
      pass_bytes(p, M, K) + split_bytes(p.cfg, (long)p.tm * p.tn, p.splits, epi == EPI_RMSNORM && !p.pass);
  return more ? kTicketBytes + more : 0;
}

// Operands through registers: no row pass, and no more scratch than the plan
// for aligned operands has, since the workspace query knows no addresses.
static Plan make_staged_plan(int M, int K, int N, int epi, bool nkl) {
  float t;
  const size_t have = plan_bytes(make_plan(M, K, N, epi, nkl), M, K, epi);
  return best_plan(M, K, N, epi, nkl, false, &t, true, have ? have - kTicketBytes : 0);
}

// A plan depends on the sizes alone; a thread keeps the last ones it made
// (the workspace query and the call ask for the same one).
static Plan plan(int M, int K, int N, int epi, bool nkl, bool staged = false) {
  struct Entry {
    int M, K, N, how;
    Plan p;
  };
  constexpr int kEntries = 64;
  static thread_local Entry kept[kEntries] = {};
  const int how = 1 + epi * 2 + (nkl ? 1 : 0) + (staged ? 8 : 0);
  Entry& e = kept[((uint32_t)M * 31 + (uint32_t)K * 7 + (uint32_t)N / 8 + how) % kEntries];
  if (e.M != M || e.K != K || e.N != N || e.how != how)
    e = {M, K, N, how, staged ? make_staged_plan(M, K, N, epi, nkl) : make_plan(M, K, N, epi, nkl)};
  return e.p;
}

// Column panels: a tile's W rows (N x K) are reached by 32-bit offsets, so K
// beyond 2^32 bytes / 256 rows takes fewer columns at a time.
static int panel_cols(int K, int N, bool nkl) {
  if (!nkl || (size_t)K * 2 * 256 < kOob) return N;
  const int n = (int)(kOob / (2 * (size_t)K)) & ~7;
  return n < 8 ? 8 : n < N ? n : N;
}

// Rows per launch.  RMSNorm: as many as the row pass's copy of x may have, in
// even panels of whole 256-row tiles (beyond K = 262144 not even one tile's
// rows may, and the tiles scale x themselves).
static int panel_rows(int M, int K, int epi) {
  if (epi != EPI_RMSNORM) return kPanelRows;
  int most = (int)(kPassBytes / (2 * (size_t)K)) / 256 * 256;
  most = most < 256 ? 256 : most < kPanelRows ? most : kPanelRows;
  const int panels = (M + most - 1) / most;
  return ((M + panels - 1) / panels + 255) / 256 * 256;
}

size_t workspace(int M, int K, int N, int epi, bool nkl) {
  const int cols = panel_cols(K, N, nkl), most = panel_rows(M, K, epi);
  size_t need = 0;
  // whole panels are alike: the first one and the remainder
  for (int rows : {M < most ? M : most, M % most})
    for (int nc : {cols, N % cols})
      if (rows > 0 && nc > 0) {
        const size_t b = plan_bytes(plan(rows, K, nc, epi, nkl), rows, K, epi);
        if (b > need) need = b;
      }
  return need;
}

void describe(int M, int K, int N, int epi, bool nkl, bool staged, int* plan6) {
  const int cols = panel_cols(K, N, nkl);
  const int most = panel_rows(M, K, epi);
  const Plan p = plan(M < most ? M : most, K, N < cols ? N : cols, epi, nkl, staged);
  const int d[6] = {YR_PLAN_PRODUCT, kCfg[p.cfg].bm, kCfg[p.cfg].bn, p.splits, p.pass, staged};
  for (int i = 0; i < 6; i++) plan6[i] = d[i];
}

int run(const Call& c, void* ws, hipStream_t st, const char* name) {
  const int cols = panel_cols(c.K, c.N, c.nkl), most = panel_rows(c.M, c.K, c.epi);
  // K and N are multiples of 8, so every row and panel keeps the alignment
  const bool staged =
      (((uintptr_t)c.x | (uintptr_t)c.gamma | (uintptr_t)c.w0 | (uintptr_t)c.w1) & 15) != 0;
  for (int m0 = 0; m0 < c.M; m0 += most)
    for (int n0 = 0; n0 < c.N; n0 += cols) {
      Args a = {};
      a.M = c.M - m0 < most ? c.M - m0 : most;
      a.K = c.K;
      a.N = c.N - n0 < cols ? c.N - n0 : cols;
      a.ldo = c.N;
      const Plan p = plan(a.M, a.K, a.N, c.epi, c.nkl, staged);
      a.x = c.x + (size_t)m0 * c.K;
      a.gamma = c.gamma;
      a.w0 = c.w0 + (size_t)n0 * c.K;  // n0 > 0 only for N x K weights
      a.w1 = c.w1 ? c.w1 + (size_t)n0 * c.K : nullptr;
      const size_t at = (size_t)m0 * c.N + n0;
      a.residual = c.residual ? c.residual + at : nullptr;
      a.out = c.out + at;
      a.eps = c.eps;
      a.splits = p.splits;
      a.tm = p.tm;
      a.tn = p.tn;
      char* scratch = ws ? (char*)ws + kTicketBytes : nullptr;
      a.tickets = (uint32_t*)ws;
      if (p.pass) {
        float* rs = (float*)scratch;
        uint16_t* xg = (uint16_t*)(scratch + align256((size_t)a.M * 4));
        if (c.dtype == YR_DTYPE_F16)
          hipLaunchKernelGGL(norm_rows_kernel<DT_F16>, dim3(a.M), dim3(256), 0, st, a.x, c.gamma, xg, rs, c.K, c.eps);
        else
          hipLaunchKernelGGL(norm_rows_kernel<DT_BF16>, dim3(a.M), dim3(256), 0, st, a.x, c.gamma, xg, rs, c.K, c.eps);
        YR_CHECK_LAUNCH(name);
        a.rs = rs;
        if (c.gamma) a.x = xg;
      }
      a.partial = (float*)(scratch + pass_bytes(p, a.M, a.K));
      if (c.epi == EPI_GATED) launch<EPI_GATED>(p.cfg, c.dtype, c.nkl, staged, a, st);
      else if (c.epi == EPI_RMSNORM) launch<EPI_RMSNORM>(p.cfg, c.dtype, c.nkl, staged, a, st);
      else launch<EPI_LINEAR>(p.cfg, c.dtype, c.nkl, staged, a, st);
      YR_CHECK_LAUNCH(name);
    }
  return YR_OK;
}

}  // namespace gm
}  // namespace yr
