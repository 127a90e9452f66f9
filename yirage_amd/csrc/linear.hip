// RMSNorm+linear, gated MLP and linear(+residual): the C entry points, their
// checks, and the one-row kernel for N x K weights.  Everything else runs on
// the matrix-product kernel (gemm.hip).
//
// One-row kernel (W[N][K], torch Linear.weight):
//  * A workgroup takes 32 output rows of W over a K slice of 2048; a lane owns
//    4 16-byte pieces of the slice and keeps x's in registers; a wave walks 4
//    rows of W at a time, 16 loads per lane in flight, v_dot2_f32_{f16,bf16}.
//  * K slices of a tile meet through fp32 records: the last workgroup to
//    arrive (atomic ticket) sums them in slice order.  Deterministic.
// Its start is short: no LDS stages to fill and, up to K = 2048, no merge.  It
// is latency-bound there, 4-9 us a launch (rule and figures at one_row()).
#include <stdarg.h>
#include <stdio.h>

#include "gemm.h"
#include "yr_common.h"

namespace yr {

enum : int { EPI_LINEAR = 0, EPI_RMSNORM = 1, EPI_GATED = 2 };
constexpr uint32_t kOob = 0xfffffff0u;  // no buffer reaches this offset

struct GemvArgs {
  const uint16_t* x;        // [B][K]
  const uint16_t* gamma;    // [K] or null
  const uint16_t* w0;       // weights (W or W1)
  const uint16_t* w1;       // W3 for the gated MLP
  const uint16_t* residual; // [B][N] or null
  uint16_t* out;            // [B][N]
  float* partial;           // [tiles][S][rec]
  uint32_t* tickets;        // [tiles]
  int B, K, N, S;           // S: number of K slices
  float eps;
};

constexpr int NK_WAVES = 8;
constexpr int NK_THREADS = NK_WAVES * kWave;
constexpr int NK_C = 4;        // 16-byte pieces per lane and row
constexpr int NK_TROWS = 32;   // output rows per workgroup
constexpr int NK_SLICE = kWave * 8 * NK_C;

template <int DT, int NMAT, int EPI>
__global__ __launch_bounds__(NK_THREADS) void gemv_nk_kernel(GemvArgs a) {
  constexpr int C = NK_C, TROWS = NK_TROWS;
  constexpr int REC = round_up4(NMAT * TROWS + 1);  // row sums, and x's sum of squares
  __shared__ float red[REC], sum[REC];
  __shared__ float ssl[NK_WAVES];

  const int tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  const int tile = blockIdx.x, split = blockIdx.y;
  const int n_base = tile * TROWS;
  const int k0 = split * NK_SLICE;

  // this lane's pieces of x (gamma applied), kept in registers
  uint32_t xr[C][4];
  float ss_part = 0.f;
#pragma unroll
  for (int c = 0; c < C; c++) {
    const int k = k0 + (lane + kWave * c) * 8;
    const bool kok = k < a.K;
    uint4 gv = make_uint4(0, 0, 0, 0), xv = make_uint4(0, 0, 0, 0);
    if constexpr (EPI == EPI_RMSNORM)
      if (a.gamma && kok) gv = ldg16(a.gamma + k);
    if (kok) xv = ldg16(a.x + k);
    const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, xw[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float lo = lo16<DT>(xw[j]), hi = hi16<DT>(xw[j]);
      if (wave == 0) ss_part += lo * lo + hi * hi;
      uint32_t p = xw[j];
      if constexpr (EPI == EPI_RMSNORM)
        if (a.gamma) p = pack2<DT>(lo * lo16<DT>(gw[j]), hi * hi16<DT>(gw[j]));
      xr[c][j] = p;
    }
  }
  if constexpr (EPI == EPI_RMSNORM) {
    const float s = wave_sum(ss_part);
    if (lane == 0) ssl[wave] = s;
  }

  // rows of this wave: wave, wave + 8, ..., 4 at a time
  constexpr int RPWV = TROWS / NK_WAVES;
  constexpr int RU = RPWV < 4 ? RPWV : 4;
#pragma unroll 1
  for (int r0 = 0; r0 < RPWV; r0 += RU) {
    uint4 w[NMAT][RU][C];
#pragma unroll
    for (int m = 0; m < NMAT; m++) {
      const uint16_t* W = m == 0 ? a.w0 : a.w1;
#pragma unroll
      for (int u = 0; u < RU; u++) {
        const int n = n_base + wave + NK_WAVES * (r0 + u);
#pragma unroll
        for (int c = 0; c < C; c++) {
          const int k = k0 + (lane + kWave * c) * 8;
          if (n < a.N && k < a.K) w[m][u][c] = ldg16(W + (size_t)n * a.K + k);
          else w[m][u][c] = make_uint4(0, 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < NMAT; m++)
#pragma unroll
      for (int u = 0; u < RU; u++) {
        float s = 0.f;
#pragma unroll
        for (int c = 0; c < C; c++) {
          s = dot2<DT>(w[m][u][c].x, xr[c][0], s);
          s = dot2<DT>(w[m][u][c].y, xr[c][1], s);
          s = dot2<DT>(w[m][u][c].z, xr[c][2], s);
          s = dot2<DT>(w[m][u][c].w, xr[c][3], s);
        }
        s = wave_sum(s);
        if (lane == 0) red[m * TROWS + wave + NK_WAVES * (r0 + u)] = s;
      }
  }
  __syncthreads();
  if (tid == 0) red[NMAT * TROWS] = EPI == EPI_RMSNORM ? ssl[0] : 0.f;
  __syncthreads();

  const float* fin = red;
  if (a.S > 1) {
    put_record(a.partial + ((size_t)tile * a.S + split) * REC, red, REC);
    if (!arrive_last(&a.tickets[tile], a.S)) return;
    sum_records(a.partial + (size_t)tile * a.S * REC, a.S, REC, sum);
    __syncthreads();
    fin = sum;
  }
  for (int rl = tid; rl < TROWS; rl += NK_THREADS) {
    const int n = n_base + rl;
    if (n >= a.N) continue;
    float v = fin[rl];
    if constexpr (EPI == EPI_RMSNORM) v *= rsqrtf(fin[NMAT * TROWS] / (float)a.K + a.eps);
    else if constexpr (EPI == EPI_GATED) v = silu(v) * fin[TROWS + rl];
    if (a.residual) v += ld_elem<DT>(a.residual[n]);
    a.out[n] = (uint16_t)st_elem<DT>(v);
  }
}

// ---------------------------------------------------------------- host side
// One row of x on N x K weights: the one-row kernel while its short start
// counts, i.e. while one K slice holds K (no merge; without a norm to wait for,
// as long as the tiles do not pass the chip) and up to 32 MiB of weights; the
// gated MLP, whose weights are two, only with one slice.  us, one-row kernel /
// product kernel, weights from HBM (in the cache):
//   RMSNorm 2048 x 14336 (K x N) 15.6 / 17.2 (13.1 / 12.3), 4096 x 1024 8.9 /
//           9.3 (7.3 / 8.9), 4096 x 4096 12.7 / 11.9 (8.7 / 10.8), 4096 x 6144
//           16.2 / 16.1 (14.8 / 14.2)
//   linear  2048 x 8192 9.5 / 11.0 (4.7 / 6.6), 2048 x 12288 12.6 / 12.9 (8.1 /
//           9.5), 4096 x 4096 11.1 / 10.6 (6.9 / 7.7), 4096 x 6144 14.9 / 15.5
//           (13.2 / 11.4), 14336 x 4096 26.5 / 24.4 (22.1 / 19.9)
//   gated   2048 x 4096 11.1 / 11.8 (6.5 / 9.3), 2048 x 8192 15.9 / 20.5 (13.4 /
//           12.0), 2048 x 12288 24.2 / 22.3 (19.8 / 16.1), 3072 x 2048 12.1 /
//           11.5 (8.9 / 7.7)
// Over 573 shapes the rule is slower than the better of the two by 0.3 %
// (RMSNorm), 2.2 % (linear) and 3.5 % (gated) on weights from HBM.
constexpr int kLongK = 1 << 26;  // 32 rows of x reach 4 GiB

static bool one_row(int B, int K, int N, int layout, int epi) {
  if (B != 1 || layout != YR_W_NK) return false;
  if (K >= kLongK) return true;  // the product kernel cuts K in 16 at most, this one in any number of slices
  if (K <= NK_SLICE) return epi == EPI_RMSNORM || N <= 8192;
  return epi != EPI_GATED && (long long)K * N <= 1ll << 24;
}

static size_t gemv_workspace(int K, int N, int nmat) {
  const size_t tiles = (N + NK_TROWS - 1) / NK_TROWS, slices = (K + NK_SLICE - 1) / NK_SLICE;
  return slices > 1 ? kTicketBytes + tiles * slices * round_up4(nmat * NK_TROWS + 1) * sizeof(float) : 0;
}

// K a kernel takes: the product kernel reaches the (up to 32) rows of x of its
// smallest tile by 32-bit offsets, 2..16 rows on N x K weights end at 2^26, and
// the one-row kernel at the K slices that its grid can hold.
static bool k_fits(int B, int K, int layout) {
  if (layout == YR_W_NK && B == 1) return K <= 65535ll * NK_SLICE;
  if (layout == YR_W_NK && B <= 16 && K >= kLongK) return false;
  return (size_t)K * 2 * (B < 32 ? B : 32) < kOob;
}
static bool ws_ok(int B, int K, int N, int layout) { return B > 0 && K > 0 && N > 0 && k_fits(B, K, layout); }

static size_t ws_for(int B, int K, int N, int layout, int epi) {
  if (!ws_ok(B, K, N, layout)) return 0;
  if (one_row(B, K, N, layout, epi)) return gemv_workspace(K, N, epi == EPI_GATED ? 2 : 1);
  const size_t w = gm::workspace(B, K, N, epi, layout == YR_W_NK);
  // K x N calls hold the ticket region at least, whether or not K is split
  return layout == YR_W_KN && w < kTicketBytes ? kTicketBytes : w;
}

// The launch of a call (yr_hip_fused_plan).
bool linear_plan(int epi, int B, int K, int N, int layout, bool aligned, int* plan6) {
  if (!ws_ok(B, K, N, layout) || K % 8 || N % 8) return false;
  if (one_row(B, K, N, layout, epi)) {
    const int d[6] = {YR_PLAN_ONE_ROW, 1, NK_TROWS, (K + NK_SLICE - 1) / NK_SLICE, 0, 0};
    for (int i = 0; i < 6; i++) plan6[i] = d[i];
  } else {
    gm::describe(B, K, N, epi, layout == YR_W_NK, !aligned, plan6);
  }
  return true;
}

template <int NMAT, int EPI>
static int run_linear(GemvArgs a, int dtype, int layout, void* ws, size_t ws_bytes, hipStream_t st,
                      const char* name) {
  if (a.B <= 0 || a.K <= 0 || a.N <= 0) return fail(YR_E_INVALID, "%s: empty shape", name);
  if (a.K % 8 || a.N % 8) return fail(YR_E_INVALID, "%s: K and N must be multiples of 8 (K=%d N=%d)", name, a.K, a.N);
  if (dtype != YR_DTYPE_F16 && dtype != YR_DTYPE_BF16) return fail(YR_E_INVALID, "%s: dtype must be f16/bf16", name);
  if (layout != YR_W_KN && layout != YR_W_NK) return fail(YR_E_INVALID, "%s: bad weight layout", name);
  if (!a.x || !a.w0 || !a.out || (NMAT == 2 && !a.w1)) return fail(YR_E_INVALID, "%s: null pointer", name);
  const size_t need = ws_for(a.B, a.K, a.N, layout, EPI);
  if (need > ws_bytes || (need && !ws))
    return fail(YR_E_WORKSPACE, "%s: workspace %zu < required %zu", name, ws_bytes, need);
  if (layout == YR_W_KN ? (a.N + 63) / 64 > kMaxTickets : (a.N + 31) / 32 > kMaxTickets)
    return fail(YR_E_INVALID, "%s: N=%d too large", name, a.N);
  // 32-bit buffer offsets: K x N operands as a whole; N x K ones are reached
  // tile by tile, but more than 16 rows were never taken past 4 GiB
  const size_t xrows = layout == YR_W_KN || a.B < 128 ? a.B : 128;
  if ((layout == YR_W_KN || a.B > 16) && ((size_t)a.K * a.N * 2 >= kOob || xrows * a.K * 2 >= kOob))
    return fail(YR_E_INVALID, "%s: operands must be < 4 GiB (32-bit buffer offsets)", name);
  if (!k_fits(a.B, a.K, layout)) return fail(YR_E_INVALID, "%s: K=%d too large", name, a.K);
  if (!one_row(a.B, a.K, a.N, layout, EPI)) {
    const gm::Call c = {a.x, a.gamma, a.w0, a.w1, a.residual, a.out, a.B, a.K, a.N, dtype, EPI, layout == YR_W_NK,
                        a.eps};
    return gm::run(c, ws, st, name);
  }
  a.S = (a.K + NK_SLICE - 1) / NK_SLICE;
  a.tickets = (uint32_t*)ws;
  a.partial = a.S > 1 ? (float*)((char*)ws + kTicketBytes) : nullptr;
  const dim3 grid((a.N + NK_TROWS - 1) / NK_TROWS, a.S);
  if (dtype == YR_DTYPE_F16)
    hipLaunchKernelGGL((gemv_nk_kernel<DT_F16, NMAT, EPI>), grid, dim3(NK_THREADS), 0, st, a);
  else
    hipLaunchKernelGGL((gemv_nk_kernel<DT_BF16, NMAT, EPI>), grid, dim3(NK_THREADS), 0, st, a);
  YR_CHECK_LAUNCH(name);
  return YR_OK;
}

}  // namespace yr

using namespace yr;

extern "C" {

size_t yr_hip_rmsnorm_linear_workspace(int batch, int k, int n, int dtype, int w_layout) {
  (void)dtype;
  return ws_for(batch, k, n, w_layout, EPI_RMSNORM);
}

size_t yr_hip_gated_mlp_workspace(int batch, int k, int n, int dtype, int w_layout) {
  (void)dtype;
  return ws_for(batch, k, n, w_layout, EPI_GATED);
}

size_t yr_hip_linear_workspace(int batch, int k, int n, int dtype, int w_layout) {
  (void)dtype;
  return ws_for(batch, k, n, w_layout, EPI_LINEAR);
}

int yr_hip_rmsnorm_linear(const void* x, const void* gamma, const void* w, void* out, int batch, int k,
                          int n, int dtype, int w_layout, float eps, void* workspace,
                          size_t workspace_bytes, void* stream) {
  GemvArgs a = {};
  a.x = (const uint16_t*)x;
  a.gamma = (const uint16_t*)gamma;
  a.w0 = (const uint16_t*)w;
  a.out = (uint16_t*)out;
  a.B = batch; a.K = k; a.N = n; a.eps = eps;
  return run_linear<1, EPI_RMSNORM>(a, dtype, w_layout, workspace, workspace_bytes, (hipStream_t)stream,
                                   "yr_hip_rmsnorm_linear");
}

int yr_hip_gated_mlp(const void* x, const void* w1, const void* w3, void* out, int batch, int k, int n,
                     int dtype, int w_layout, void* workspace, size_t workspace_bytes, void* stream) {
  GemvArgs a = {};
  a.x = (const uint16_t*)x;
  a.w0 = (const uint16_t*)w1;
  a.w1 = (const uint16_t*)w3;
  a.out = (uint16_t*)out;
  a.B = batch; a.K = k; a.N = n;
  return run_linear<2, EPI_GATED>(a, dtype, w_layout, workspace, workspace_bytes, (hipStream_t)stream,
                                 "yr_hip_gated_mlp");
}

int yr_hip_linear(const void* x, const void* w, const void* residual, void* out, int batch, int k,
                  int n, int dtype, int w_layout, void* workspace, size_t workspace_bytes,
                  void* stream) {
  GemvArgs a = {};
  a.x = (const uint16_t*)x;
  a.w0 = (const uint16_t*)w;
  a.residual = (const uint16_t*)residual;
  a.out = (uint16_t*)out;
  a.B = batch; a.K = k; a.N = n;
  return run_linear<1, EPI_LINEAR>(a, dtype, w_layout, workspace, workspace_bytes, (hipStream_t)stream,
                                  "yr_hip_linear");
}

}  // extern "C"
