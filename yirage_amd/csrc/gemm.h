// Host side of the matrix-product kernel (gemm_kernel.h): which tile and how
// many K splits a shape gets, and the launches.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace yr {

// The launch of a call of linear.hip (yr_hip_fused_plan); false if refused.
bool linear_plan(int epi, int B, int K, int N, int layout, bool aligned, int* plan6);

namespace gm {

struct Args;

// One call: out = epilogue(x [M][K] @ W), every pointer checked by the caller
// (EPI_LINEAR / EPI_RMSNORM / EPI_GATED of gemm_kernel.h; K, N multiples of 8).
struct Call {
  const uint16_t *x, *gamma, *w0, *w1, *residual;
  uint16_t* out;
  int M, K, N, dtype, epi;
  bool nkl;
  float eps;
};

// Scratch bytes of a call (tickets first, see kTicketBytes); 0 if none.  The
// same for operands that are not 16-byte aligned.
size_t workspace(int M, int K, int N, int epi, bool nkl);
int run(const Call& c, void* ws, hipStream_t st, const char* name);
// {YR_PLAN_PRODUCT, tile rows, tile columns, K splits, row pass, operands
// through registers} of the first launch of a call
void describe(int M, int K, int N, int epi, bool nkl, bool staged, int* plan6);

// One launch of tile `cfg` (kCfg) with a.splits K splits, `staged` with the
// operands through registers; defined per epilogue so that the instances
// compile in parallel.
template <int EPI>
void launch(int cfg, int dtype, bool nkl, bool staged, const Args& a, hipStream_t st);

// Tiles, smallest first.  BM x BN output (columns of all matrices), waves
// along rows x columns, LDS stages, workgroups per CU.
enum Cfg { C32x64, C32x128, C64x128, C128x128, C128x192, C128x256, C256x256, kNumCfg };

}  // namespace gm
}  // namespace yr
