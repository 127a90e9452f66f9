// The matrix-product kernel behind RMSNorm+linear, gated MLP and
// linear(+residual), any number of rows, W in [K][N] or [N][K] layout.
//
// One workgroup computes a BM x BN tile of the output (for the gated MLP BN/2
// columns of each of W1 and W3) over one K split.  K advances in chunks of 64
// through NST LDS stages that direct buffer -> LDS loads fill (no registers),
// NST - 1 chunks ahead of the matrix cores.  The product is formed transposed
// (A = W, B = x), so a lane of the accumulator holds four consecutive output
// columns of one row and stores them with one 8-byte store.
//
// Software pipeline: a chunk is two 32-k halves.  While the MFMAs of one half
// run, the fragments of the next half come in from LDS, a few reads before
// each group of MFMAs (the order is pinned: left to itself the compiler puts
// the reads in one burst and the MFMAs behind one wait, 1.06 against 1.24
// PFLOP/s on the 2048-row gated MLP).  The workgroup's one barrier per chunk
// sits between the halves: the second half's operands are in registers by
// then, so every wave has a half's MFMAs to issue while it crosses the
// barrier, and the stage just read is refilled right after it, one load
// between MFMA groups (8 loads in a row stall the wave on the load queue).
//
// Rows of the LDS images are permuted in 16-byte chunks, on the global side
// of the loads (the LDS image of one load instruction is contiguous), so that
// fragment reads are free of bank conflicts: 128-byte rows (x, and W in
// N x K) by row % 8, K x N rows of 128 or 64 columns by w_swz.
//
// Direct loads need 16-byte aligned operands.  Without DMA (x, gamma or W at
// another address) the same pieces pass through registers: the loads of a
// chunk are issued where the direct ones are, and written to the stage one
// chunk later, behind the next barrier.
#pragma once
#include <type_traits>

#include "yr_common.h"

namespace yr {
namespace gm {

// EPI_RMSNORM: x is already x * gamma and rs holds the row factors (a pass
// before the product).  EPI_RMSNORM_LDS: raw x; every chunk of it is squared,
// summed and scaled by gamma in LDS, in place, two chunks before its use
// (tiles of few rows: one or two 16-byte pieces per thread and chunk).
enum : int { EPI_LINEAR = 0, EPI_RMSNORM = 1, EPI_GATED = 2, EPI_RMSNORM_LDS = 3 };

struct Args {
  const uint16_t* x;         // [M][K]
  const uint16_t* gamma;     // [K] or null (EPI_RMSNORM_LDS)
  const float* rs;           // [M] (EPI_RMSNORM)
  const uint16_t* w0;        // W, or W1
  const uint16_t* w1;        // W3 (gated)
  const uint16_t* residual;  // [M][ldo] or null
  uint16_t* out;             // [M][ldo]
  float* partial;            // K-split records [tile][split][...]
  uint32_t* tickets;         // [tile], zero at rest
  float eps;
  int M, K, N;
  int ldo;                   // row stride of out and residual (elements)
  int splits, tm, tn;        // K splits per tile; row and column tiles
};

constexpr int KS = 64;                   // k per chunk
constexpr int kMaxSplits = 16;           // K splits of a tile
constexpr uint32_t kOob = 0xfffffff0u;   // offset that is out of range for every buffer
constexpr int kSc1 = 16;                 // buffer cache policy: sc1 (agent-scope coherence)
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

// 16 bytes per lane from a buffer straight into LDS (lane l's data lands at
// lds + 16 l, lds wave-uniform); an offset past the buffer writes zeros.
// Issued as inline assembly: the compiler then inserts no waits of its own
// for these loads (it cannot tell which LDS stage one writes and would wait
// for all of them before any LDS read); the kernel orders them itself
// (s_waitcnt vmcnt and a barrier before a stage is read, a barrier after the
// last read of a stage before it is refilled).  The s_nop is the wait state
// that a load reading M0 needs after a scalar write of it: the compiler
// inserts none inside inline assembly.
__device__ __forceinline__ void bload_lds16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %2, %3 offen lds"
               :
               : "v"(off), "s"(__builtin_amdgcn_readfirstlane(lds)), "s"(r), "s"(__builtin_amdgcn_readfirstlane(soff))
               : "memory", "m0");
}

// At most N of this wave's vector-memory operations and none of its LDS
// operations pending, then the workgroup's barrier (gfx9 encoding of
// s_waitcnt: vmcnt bits 3:0 and 15:14, lgkmcnt 11:8, expcnt 6:4 at its maximum)
template <int N>
__device__ __forceinline__ void wait_and_sync() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// chunk permutation of K x N rows of SW columns: the rows one 32-lane
// transposing read touches (8g + e, and + 4, e < 4, g < 2) get distinct
// 32-byte chunk pairs; rows r and r + 4 (and r + 32) share it
template <int SW>
__device__ __forceinline__ int w_swz(int r) {
  return SW == 128 ? ((r & 3) | (((r >> 3) & 1) << 2)) << 1 : (((r >> 1) & 1) | (((r >> 3) & 1) << 1)) << 1;
}

__device__ __forceinline__ uint4 lds_rd(const char* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ uint2 lds_tr(const char* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(const_cast<char*>(p))));
}

// x * gamma, element-wise on 8 packed values, rounded to the storage type
// (the normalised activation the reference feeds its matmul).  f16: the packed
// product rounds once, as the exact fp32 product of two halves does.
template <int DT>
__device__ __forceinline__ uint4 scale8(uint4 x, uint4 g) {
  const uint32_t xv[4] = {x.x, x.y, x.z, x.w}, gv[4] = {g.x, g.y, g.z, g.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if constexpr (DT == DT_F16)
      o[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, xv[i]) * __builtin_bit_cast(half2v, gv[i]));
    else
      o[i] = pack2<DT>(lo16<DT>(xv[i]) * lo16<DT>(gv[i]), hi16<DT>(xv[i]) * hi16<DT>(gv[i]));
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// s + the squares of 8 packed values, fp32
template <int DT>
__device__ __forceinline__ float sumsq8(uint4 x, float s) {
  s = dot2<DT>(x.x, x.x, s);
  s = dot2<DT>(x.y, x.y, s);
  s = dot2<DT>(x.z, x.z, s);
  return dot2<DT>(x.w, x.w, s);
}

// WM x WN waves; wave (wm, wn) owns rows wm BM / WM .. of the tile and
// BN / WN columns (for the gated MLP the same BN / WN / 2 columns of both
// matrices, so its lanes hold both factors of an output).
template <int DT, int EPI, bool NKL, int BM, int BN, int WM, int WN, int NST, bool DMA>
__global__ __launch_bounds__(64 * WM * WN) void gemm_kernel(Args a) {
  constexpr bool NORM = EPI == EPI_RMSNORM_LDS;
  constexpr int NW = WM * WN, NMAT = EPI == EPI_GATED ? 2 : 1, BNM = BN / NMAT;
  constexpr int XB = BM * KS * 2, WB = BN * KS * 2, MB = BNM * KS * 2;  // bytes per stage: x, W, one matrix
  constexpr int GB = NORM ? 1024 : 0;                                   // gamma
  constexpr int NX = XB / 1024 / NW, NWL = WB / 1024 / NW;              // 1 KB loads per wave and chunk
  constexpr int LPW = NX + NWL + (NORM ? 1 : 0);
  constexpr int NBM = MB / 1024;
  static_assert(XB % (1024 * NW) == 0 && MB % (1024 * NW) == 0, "whole loads per wave");
  constexpr int MI = BM / WM / 16, NJ = BN / WN / 16, NJM = NJ / NMAT;  // MFMA blocks per wave
  constexpr int SW = BNM % 128 == 0 ? 128 : 64;                         // K x N: columns of a sub-tile
  static_assert(BNM % SW == 0 && NST >= (NORM ? 3 : 2) + (DMA ? 0 : 1) && (NST - 1) * LPW < 64, "stages");
  constexpr int NP = NORM ? BM * 8 / (64 * NW) : 1;                     // 16-byte pieces of x per thread and chunk
  static_assert(!NORM || (NP >= 1 && BM * 8 % (64 * NW) == 0), "whole pieces per thread");
  __shared__ __attribute__((aligned(16))) char lds[NST * (XB + WB + GB)];  // x stages, W stages, gamma stages

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous range of
  // (tile, split), tiles in groups of 8 row tiles by columns, so the
  // workgroups of an XCD share x rows and W columns in its L2.
  const int G = gridDim.x, q8 = G / 8, r8 = G % 8, xcd = blockIdx.x % 8;
  const int v = xcd * q8 + (xcd < r8 ? xcd : r8) + blockIdx.x / 8;
  const int t = v / a.splits, sp = v % a.splits;
  const int grp = t / (8 * a.tn), gt = t - grp * 8 * a.tn, grows = min(a.tm - grp * 8, 8);
  const int m0 = (grp * 8 + gt % grows) * BM, n0 = gt / grows * BNM;
  const int kper = ((a.K + a.splits - 1) / a.splits + KS - 1) / KS * KS;  // k per split (whole chunks)
  const int kbeg = sp * kper, kend = min(a.K, kbeg + kper);
  const int nch = kend > kbeg ? (kend - kbeg + KS - 1) / KS : 0;

  // Rows of x past M, and columns of W past N, repeat the last one: their
  // products go to outputs that are never stored.  k past the split is read
  // as zero on both sides.  The buffers start at the tile's first row (x, and
  // W in N x K layout), so 32-bit offsets reach any M and N.
  const int mrows = min(a.M - m0, BM), ncols = min(a.N - n0, BNM);
  const __amdgpu_buffer_rsrc_t rx = rsrc(a.x + (size_t)m0 * a.K, (uint32_t)((size_t)mrows * a.K * 2));
  const size_t wbase = NKL ? (size_t)n0 * a.K : 0;
  const uint32_t wbytes = NKL ? (uint32_t)((size_t)ncols * a.K * 2) : (uint32_t)((size_t)a.K * a.N * 2);
  const __amdgpu_buffer_rsrc_t rw0 = rsrc(a.w0 + wbase, wbytes);
  const __amdgpu_buffer_rsrc_t rw1 = rsrc((NMAT == 2 ? a.w1 : a.w0) + wbase, wbytes);
  const __amdgpu_buffer_rsrc_t rg = rsrc(NORM ? a.gamma : nullptr, NORM && a.gamma ? (uint32_t)(a.K * 2) : 0u);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)(&lds[0]);

  // load i of this wave fills 1 KB block wave + NW i of the x (W) stage: 8
  // rows of 128 bytes, or 512 / SW rows of SW columns
  uint32_t xo[NX], wo[NWL];
  const int prow = lane >> 3, pchunk = (lane & 7) ^ prow;
#pragma unroll
  for (int i = 0; i < NX; i++)
    xo[i] = (uint32_t)(((size_t)min(8 * (wave + NW * i) + prow, mrows - 1) * a.K + kbeg + 8 * pchunk) * 2);
  constexpr int CPR = SW / 8, RPB = 64 / CPR, BPS = KS / RPB;
#pragma unroll
  for (int i = 0; i < NWL; i++) {
    const int jb = (wave + NW * i) % NBM;
    if constexpr (NKL) {
      wo[i] = (uint32_t)(((size_t)min(8 * jb + prow, ncols - 1) * a.K + kbeg + 8 * pchunk) * 2);
    } else {
      const int sub = jb / BPS, row = RPB * (jb % BPS) + lane / CPR;
      const int src = (lane % CPR) ^ w_swz<SW>(row);
      wo[i] = (uint32_t)(((size_t)(kbeg + row) * a.N + min(n0 + sub * SW + 8 * src, a.N - 8)) * 2);
    }
  }
  const uint32_t wstep = NKL ? KS * 2 : (uint32_t)(KS * a.N * 2);
  const uint32_t xd = lds0 + 1024 * wave, wd = lds0 + NST * XB + 1024 * wave, gd = lds0 + NST * (XB + WB);
  // load p of chunk ci (a whole one) into stage s
  auto load1 = [&](int p, int ci, int s) __attribute__((always_inline)) {
    if (p < NX) bload_lds16(rx, xo[p], (uint32_t)ci * (KS * 2), xd + s * XB + 1024 * NW * p);
    else if (p < NX + NWL)
      bload_lds16(p - NX < NBM / NW ? rw0 : rw1, wo[p - NX], (uint32_t)ci * wstep, wd + s * WB + 1024 * NW * (p - NX));
    else bload_lds16(rg, lane < 8 ? (uint32_t)((kbeg + ci * KS + 8 * lane) * 2) : kOob, 0, gd + s * GB);
  };
  // every load of chunk ci, which may be partial or past the end
  auto issue = [&](int ci, int s) __attribute__((always_inline)) {
    if (ci >= nch) return;
    const int krel = kend - kbeg - ci * KS;
    if (krel >= KS) {
#pragma unroll
      for (int p = 0; p < LPW; p++) load1(p, ci, s);
    } else {
#pragma unroll
      for (int i = 0; i < NX; i++)
        bload_lds16(rx, 8 * pchunk < krel ? xo[i] + (uint32_t)ci * (KS * 2) : kOob, 0, xd + s * XB + 1024 * NW * i);
#pragma unroll
      for (int i = 0; i < NWL; i++) {
        const int k = NKL ? 8 * pchunk : RPB * (((wave + NW * i) % NBM) % BPS) + lane / CPR;
        bload_lds16(i < NBM / NW ? rw0 : rw1, k < krel ? wo[i] + (uint32_t)ci * wstep : kOob, 0,
                    wd + s * WB + 1024 * NW * i);
      }
      if constexpr (NORM)
        bload_lds16(rg, 8 * lane < krel ? (uint32_t)((kbeg + ci * KS + 8 * lane) * 2) : kOob, 0, gd + s * GB);
    }
  };

  // without DMA: the pieces of chunk ci into registers (global loads, any
  // address), and from there into stage s
  uint4 held[DMA ? 1 : LPW];
  auto hold = [&](int ci) __attribute__((always_inline)) {
    const int krel = kend - kbeg - ci * KS;
    const uint4 zero = make_uint4(0, 0, 0, 0);
    if (krel <= 0) return;
#pragma unroll
    for (int p = 0; p < LPW; p++) {
      const char* base;
      uint32_t off;
      int k;
      if (p < NX) {
        base = reinterpret_cast<const char*>(a.x + (size_t)m0 * a.K);
        off = xo[p < NX ? p : 0] + (uint32_t)ci * (KS * 2);
        k = 8 * pchunk;
      } else if (p < NX + NWL) {
        const int i = p - NX;
        base = reinterpret_cast<const char*>((i < NBM / NW ? a.w0 : a.w1) + wbase);
        off = wo[i] + (uint32_t)ci * wstep;
        k = NKL ? 8 * pchunk : RPB * (((wave + NW * i) % NBM) % BPS) + lane / CPR;
      } else {
        base = reinterpret_cast<const char*>(a.gamma);
        off = (uint32_t)((kbeg + ci * KS + 8 * lane) * 2);
        k = lane < 8 && a.gamma ? 8 * lane : KS;
      }
      held[DMA ? 0 : p] = k < min(krel, KS) ? ldg16(base + off) : zero;
    }
  };
  auto put_held = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < LPW; p++) {
      const uint32_t d = p < NX        ? xd + s * XB + 1024 * NW * p
                         : p < NX + NWL ? wd + s * WB + 1024 * NW * (p - NX)
                                        : gd + s * GB;
      *reinterpret_cast<uint4*>(lds + (d - lds0) + 16 * lane) = held[DMA ? 0 : p];
    }
  };

  // fragments: lane l holds row (column) l % 16 of a block, k 8 (l / 16) ..
  // +7 of the half; W in K x N comes back by transposing reads
  const int wm = wave % WM, wn = wave / WM, g = lane >> 4, l15 = lane & 15;
  uint32_t xa[2], wa[NKL ? 2 : NJM];
#pragma unroll
  for (int ks = 0; ks < 2; ks++) {
    const uint32_t c = 16 * ((4 * ks + g) ^ (l15 & 7));
    xa[ks] = (wm * (BM / WM) + l15) * 128 + c;
    if constexpr (NKL) wa[ks] = NST * XB + (wn * NJM * 16 + l15) * 128 + c;
  }
  if constexpr (!NKL) {
    const int e = l15 >> 2, q = l15 & 3, r0 = 8 * g + e;
#pragma unroll
    for (int j = 0; j < NJM; j++) {
      const int jn = (wn * NJM + j) * 16, c = (jn % SW) / 8 + (q >> 1);
      wa[j] = NST * XB + jn / SW * SW * KS * 2 + r0 * SW * 2 + ((c ^ w_swz<SW>(r0)) << 4) + (q & 1) * 8;
    }
  }
  auto rd_w = [&](int j, int ks, int s) __attribute__((always_inline)) -> uint4 {
    const uint32_t off = s * WB + j / NJM * MB;
    if constexpr (NKL) {
      return lds_rd(lds + wa[ks] + off + j % NJM * 2048);
    } else {
      const char* p = lds + wa[j % NJM] + off + ks * 32 * SW * 2;
      const uint2 lo = lds_tr(p), hi = lds_tr(p + 4 * SW * 2);
      return make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
  };
  auto rd_x = [&](int i, int ks, int s) __attribute__((always_inline)) {
    return lds_rd(lds + xa[ks] + s * XB + i * 2048);
  };

  f32x4 acc[NJ][MI];
#pragma unroll
  for (int j = 0; j < NJ; j++)
#pragma unroll
    for (int i = 0; i < MI; i++) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // RMSNorm in LDS: thread t's piece p is physical chunk t % 8 of row t / 8 + 8 NW p
  float ss[NP];  // sums of squares (this thread's k)
  uint4 px[NP], pg;
#pragma unroll
  for (int p = 0; p < NP; p++) ss[p] = 0.f;
  auto norm_rd = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++) px[p] = lds_rd(lds + s * XB + (tid + 64 * NW * p) * 16);
    pg = lds_rd(lds + NST * (XB + WB) + s * GB + 16 * pchunk);
  };
  auto norm_wr = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      ss[p] = sumsq8<DT>(px[p], ss[p]);
      if (a.gamma) *reinterpret_cast<uint4*>(lds + s * XB + (tid + 64 * NW * p) * 16) = scale8<DT>(px[p], pg);
    }
  };

  struct Frag {
    uint4 w[NJ], x[MI];
  };
  Frag f0, f1;
  // One half: MFMAs from `c`, group i = row block i; the next half's
  // fragments (half ks of stage s) into `n` over the first groups; with LD
  // the loads of chunk lci into stage ls, spread over all groups.
  constexpr int NRD = NJ + MI, NG = MI > 1 ? MI - 1 : 1;
  auto half = [&](const Frag& c, Frag& n, int ks, int s, auto ldc, int lci, int ls) __attribute__((always_inline)) {
    constexpr bool LD = decltype(ldc)::value;
#pragma unroll
    for (int i = 0; i < MI; i++) {
#pragma unroll
      for (int r = 0; r < NRD; r++)
        if (r >= i * NRD / NG && r < (i + 1) * NRD / NG) {
          if (r < NJ) n.w[r] = rd_w(r, ks, s);
          else n.x[r - NJ] = rd_x(r - NJ, ks, s);
        }
      if constexpr (LD) {
#pragma unroll
        for (int p = 0; p < LPW; p++)
          if (p >= i * LPW / MI && p < (i + 1) * LPW / MI) load1(p, lci, ls);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int j = 0; j < NJ; j++) acc[j][i] = mfma16<DT>(c.w[j], c.x[i], acc[j][i]);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Chunk ci in stage s.  The wait lets the loads of chunks ci + 2 .. pend
  // (RMSNorm in LDS: ci + 3 .., as chunk ci + 2 is read here and written back
  // scaled before the next barrier, which is the one its first use waits for);
  // near the end fewer are in flight and it waits for all.  (Past the last
  // chunk the reads find stale LDS, which no MFMA uses.)
  constexpr int AHEAD = NORM ? 2 : 1;
  auto chunk = [&](int ci, auto sc, auto ldc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value, s1 = (s + 1) % NST, s2 = (s + 2) % NST;
    constexpr bool LD = decltype(ldc)::value;
    half(f0, f1, 1, s, std::false_type{}, 0, 0);
    if constexpr (NORM)
      if (ci > 0 && (LD || ci + 1 < nch)) norm_wr(s1);  // chunks 0 and 1 were scaled before the loop
    if (LD || ci + NST <= nch) wait_and_sync<(NST - 1 - AHEAD) * LPW>();
    else wait_and_sync<0>();
    if constexpr (NORM)
      if (LD || ci + 2 < nch) norm_rd(s2);
    if constexpr (!DMA) {  // chunk ci - 1 + NST has come in since the last barrier
      if (ci > 0 && ci - 1 + NST < nch) put_held((s + NST - 1) % NST);
      hold(ci + NST);
    } else if constexpr (!LD) {
      issue(ci + NST, s);
    }
    half(f1, f0, 0, s1, ldc, ci + NST, s);
  };
  auto round = [&](int ci, auto self, auto sc, auto ldc) __attribute__((always_inline)) {
    constexpr int s = decltype(sc)::value;
    if (decltype(ldc)::value || ci + s < nch) chunk(ci + s, sc, ldc);
    if constexpr (s + 1 < NST) self(ci, self, std::integral_constant<int, s + 1>{}, ldc);
  };
#pragma unroll
  for (int c = 0; c < NST; c++) {
    if constexpr (DMA) {
      issue(c, c);
    } else if (c < nch) {
      hold(c);
      put_held(c);
    }
  }
  if (nch >= NST) wait_and_sync<(NST - AHEAD) * LPW>();
  else wait_and_sync<0>();
  if constexpr (NORM) {
    if (nch > 0) {
      norm_rd(0);
      norm_wr(0);
    }
    if (nch > 1) {
      norm_rd(1);
      norm_wr(1);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < NJ; j++) f0.w[j] = rd_w(j, 0, 0);
#pragma unroll
  for (int i = 0; i < MI; i++) f0.x[i] = rd_x(i, 0, 0);
  int ci = 0;
  const int nwhole = (kend - kbeg) / KS;
  for (; DMA && ci + 2 * NST <= nwhole; ci += NST) round(ci, round, std::integral_constant<int, 0>{}, std::true_type{});
  for (; ci < nch; ci += NST) round(ci, round, std::integral_constant<int, 0>{}, std::false_type{});

  // RMSNorm in LDS: a row's sum is with the 8 lanes of its pieces
  float* rss = reinterpret_cast<float*>(lds + NST * (XB + WB));  // [BM] row sums (the gamma stages are free)
  if constexpr (NORM) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < NP; p++) {
#pragma unroll
      for (int o = 4; o > 0; o >>= 1) ss[p] += __shfl_xor(ss[p], o, kWave);
      if ((tid & 7) == 0) rss[(tid + 64 * NW * p) >> 3] = ss[p];
    }
    __syncthreads();
  }

  // K splits: every split stores its accumulators in fragment order (1 KB per
  // wave and store) and arrives on the tile's ticket; the last adds all the
  // records in split order (its own among them), so results do not depend
  // on timing.  128-bit sc1 accesses: agent scope, and free to pipeline.
  if (a.splits > 1) {
    constexpr int NV = NJ * MI, NT = 64 * NW, NVR = NV + (NORM ? 1 : 0);  // one more for the row sums
    static_assert(BM <= NT, "one thread per row sum");
    const __amdgpu_buffer_rsrc_t rp =
        rsrc(a.partial + (size_t)t * a.splits * NVR * NT * 4, (uint32_t)(a.splits * NVR * NT * 16));
    f32x4* av = &acc[0][0];
    auto off = [&](int s2, int w) __attribute__((always_inline)) { return (uint32_t)((s2 * NVR + w) * NT + tid) * 16; };
#pragma unroll
    for (int w = 0; w < NV; w++)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(yr_u32x4, av[w]), rp, off(sp, w), 0, kSc1);
    if constexpr (NORM)
      if (tid < BM) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(rss[tid]), rp, off(sp, NV), 0, kSc1);
    if (!arrive_last(&a.tickets[t], a.splits)) return;
    auto rec = [&](int s2, int w) __attribute__((always_inline)) {
      return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, off(s2, w), 0, kSc1));
    };
    // every split's row sum first, in flight beside the records
    float rs[NORM ? kMaxSplits : 1];
    if constexpr (NORM) {
#pragma unroll
      for (int s2 = 0; s2 < kMaxSplits; s2++)
        rs[s2] = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(rp, tid < BM ? off(s2, NV) : kOob, 0, kSc1));
    }
    // VG float4s of SU splits in flight (offsets past the records read zeros):
    // one split at a time, every record was a memory round trip of its own
    constexpr int VG = NV % 4 == 0 ? 4 : NV % 2 == 0 ? 2 : 1, SU = 4;
#pragma unroll
    for (int v0 = 0; v0 < NV; v0 += VG) {
      f32x4 sum[VG];
#pragma unroll
      for (int w = 0; w < VG; w++) sum[w] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < a.splits; s0 += SU) {
        f32x4 ld[SU][VG];
#pragma unroll
        for (int u = 0; u < SU; u++)
#pragma unroll
          for (int w = 0; w < VG; w++) ld[u][w] = rec(s0 + u, v0 + w);
#pragma unroll
        for (int u = 0; u < SU; u++)
#pragma unroll
          for (int w = 0; w < VG; w++) sum[w] += ld[u][w];
      }
#pragma unroll
      for (int w = 0; w < VG; w++) av[v0 + w] = sum[w];
    }
    if constexpr (NORM) {
      if (tid < BM) {
        float sum = 0.f;
#pragma unroll
        for (int s2 = 0; s2 < kMaxSplits; s2++) sum += rs[s2];
        rss[tid] = sum;
      }
      __syncthreads();
    }
  }

  // accumulator block (j, i): row 16 i + l15, columns 16 j + 4 g .. +3
#pragma unroll
  for (int i = 0; i < MI; i++) {
    const int m = m0 + wm * (BM / WM) + 16 * i + l15;
    if (m >= a.M) continue;
    float scale = 1.f;
    if constexpr (EPI == EPI_RMSNORM) scale = gptr(a.rs)[m];
    if constexpr (NORM) scale = rsqrtf(rss[m - m0] / (float)a.K + a.eps);
#pragma unroll
    for (int j = 0; j < NJM; j++) {
      const int n = n0 + (wn * NJM + j) * 16 + 4 * g;
      if (n >= a.N) continue;
      float o[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        o[q] = acc[j][i][q];
        if constexpr (EPI == EPI_RMSNORM || NORM) o[q] *= scale;
        if constexpr (EPI == EPI_GATED) o[q] = silu(o[q]) * acc[NJM + j][i][q];
      }
      const size_t at = (size_t)m * a.ldo + n;
      if (a.residual) {
        const u32x2 r = *(const YR_G u32x2*)(a.residual + at);
        o[0] += lo16<DT>(r[0]);
        o[1] += hi16<DT>(r[0]);
        o[2] += lo16<DT>(r[1]);
        o[3] += hi16<DT>(r[1]);
      }
      *(YR_G u32x2*)(a.out + at) = u32x2{pack2<DT>(o[0], o[1]), pack2<DT>(o[2], o[3])};
    }
  }
}

}  // namespace gm
}  // namespace yr
