// Instances of the matrix-product kernel, one epilogue per source file.
#pragma once
#include "gemm.h"
#include "gemm_kernel.h"

namespace yr {
namespace gm {

template <int DT, int EPI, bool NKL, int BM, int BN, int WM, int WN, int NST, bool DMA = true>
static void go(const Args& a, hipStream_t st) {
  hipLaunchKernelGGL((gemm_kernel<DT, EPI, NKL, BM, BN, WM, WN, NST, DMA>), dim3(a.tm * a.tn * a.splits),
                     dim3(64 * WM * WN), 0, st, a);
}

// The tiles of up to 64 rows scale x in LDS when they normalise, the others
// take x already scaled; 192 columns do not halve into two matrices of whole
// LDS rows.  Stages: what 160 KB of LDS hold, two workgroups per CU for the
// two narrowest tiles.  An unsplit 128 x 128 tile of the K x N gated MLP takes
// 4 waves of 128 rows each: W comes back by transposing reads, at two thirds
// of the rate of plain ones, and is then read once instead of by two waves
// (128 rows, 2 x 4096 x 14336: 57.0 us against 59.4; with K splits the merge
// wants the 8 waves, 120 rows, 2 x 3000 x 5000: 22.4 against 23.6).
template <int DT, int EPI, bool NKL>
static void go_cfg(int cfg, const Args& a, hipStream_t st) {
  constexpr int E = EPI == EPI_RMSNORM ? EPI_RMSNORM_LDS : EPI;
  switch (cfg) {
    case C32x64:
      if constexpr (EPI != EPI_GATED) go<DT, E, NKL, 32, 64, 1, 4, 5>(a, st);
      break;
    case C32x128: go<DT, E, NKL, 32, 128, 1, 4, EPI == EPI_RMSNORM ? 4 : 3>(a, st); break;
    case C64x128: go<DT, E, NKL, 64, 128, 2, 4, 6>(a, st); break;
    case C128x128:
      if constexpr (EPI == EPI_GATED && !NKL) {
        if (a.splits == 1) {
          go<DT, EPI, NKL, 128, 128, 1, 4, 4>(a, st);
          break;
        }
      }
      go<DT, EPI, NKL, 128, 128, 2, 4, 4>(a, st);
      break;
    case C128x192:
      if constexpr (EPI != EPI_GATED) go<DT, EPI, NKL, 128, 192, 2, 4, 3>(a, st);
      break;
    case C128x256: go<DT, EPI, NKL, 128, 256, 2, 4, 3>(a, st); break;
    case C256x256: go<DT, EPI, NKL, 256, 256, 2, 4, 2>(a, st); break;
  }
}

// Operands that are not 16-byte aligned: two tiles, both of which also scale x
// themselves; the loads through registers want a stage more than direct ones.
// One chunk per workgroup in flight bounds them: 8 rows, 4096 x 4096 20 us
// (12 aligned), 128 rows, 4096 x 14336 51 us (29), 2048 rows, 4096 x 4096 186
// us (61).
template <int DT, int EPI, bool NKL>
static void go_staged(int cfg, const Args& a, hipStream_t st) {
  constexpr int E = EPI == EPI_RMSNORM ? EPI_RMSNORM_LDS : EPI;
  if (cfg == C32x128) go<DT, E, NKL, 32, 128, 1, 4, EPI == EPI_RMSNORM ? 4 : 3, false>(a, st);
  else go<DT, E, NKL, 64, 128, 2, 4, 6, false>(a, st);
}

template <int EPI>
void launch(int cfg, int dtype, bool nkl, bool staged, const Args& a, hipStream_t st) {
  auto run = [&](auto dt, auto nk) {
    constexpr int DT = decltype(dt)::value;
    constexpr bool NKL = decltype(nk)::value;
    if (staged) go_staged<DT, EPI, NKL>(cfg, a, st);
    else go_cfg<DT, EPI, NKL>(cfg, a, st);
  };
  auto with = [&](auto dt) { nkl ? run(dt, std::true_type{}) : run(dt, std::false_type{}); };
  if (dtype == YR_DTYPE_F16) with(std::integral_constant<int, DT_F16>{});
  else with(std::integral_constant<int, DT_BF16>{});
}

}  // namespace gm
}  // namespace yr
