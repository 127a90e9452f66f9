// Attention on the operands a kernel graph holds, without packing them first:
//   O[g] = softmax(scale * Q[g] K[g]) V[g],
// Q [G][M][d], K [G][d][L] (rows are head dims), V [G][L][d], d = 64 or 128.
//
// The same transposed flash attention as the prefill kernel (S^T = K Q^T,
// O^T += V^T P^T on MFMA 16x16x32, P straight from the accumulators), with
//   * K read as it lies: a [d][64 tokens] tile in LDS comes back as the A
//     operand (tokens x d) by transposing reads, like V's;
//   * the tokens of a group split over workgroups, so that a few query rows
//     over a long sequence fill the chip; the last workgroup to arrive merges;
//   * a tile for few rows (16 or 32) whose other waves take other tokens.
// A workgroup is RW row waves (16 RB query rows each) x KW token waves.  K / V
// tiles of 64 tokens are double buffered by direct global -> LDS loads.
#include <type_traits>

#include "yr_common.h"
#include "attn_device.h"
#include "attn_launch.h"

namespace yr {
namespace ga {

constexpr int KT = 64;  // tokens per tile

struct Args {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  long long q_bs, k_bs, v_bs, o_bs;  // group strides (elements)
  long long q_ld, k_ld, v_ld, o_ld;  // strides of query rows, head dims, tokens, output rows
  float* partial;                    // [G][nqb][splits]: O [QR][D], then (m, l) [QR][2]
  uint32_t* tickets;                 // [G][nqb]
  int G, M, L, nqb, splits, chunk, nwg;
  float scale_log2;
};

// Bound by LDS reads and the softmax between them where many rows share a
// tile, by the split merge for few.  16 groups of 256 rows, 4096 tokens, d =
// 64, f16: 17.6 us (4.3 GFLOP), against 126 us for packing Q, K, V to d = 128
// and the prefill kernel on 64 workgroups.
template <int DT, int D, int RW, int KW, int RB>
__global__ __launch_bounds__(64 * RW * KW, 2) void graph_attn_kernel(Args a) {
  constexpr int W = RW * KW, QR = 16 * RW * RB, NB = KT / KW / 16, NDT = D / 16, NS = D / 32;
  // one stage: the K tile [D][KT] (128-byte rows), then the V tile [KT][D].
  // 16-byte chunks are permuted in pairs by row, so that the 8 rows x 32 bytes
  // which two 16-lane groups of a transposing read touch lie in 8 different
  // 32-byte bank columns (checked over all rows and tiles).  Two objects: reads
  // of one stage then do not wait for the loads that fill the other.
  __shared__ __attribute__((aligned(16))) uint16_t st0[2 * KT * D], st1[2 * KT * D];
  __shared__ float2 s_ml[RW * RB][kWave];

  // workgroup i runs on XCD i % 8; consecutive items (the query blocks of one
  // token range first) stay on one XCD and share its L2
  const int id = blockIdx.x;
  const int w = a.nwg % 8 == 0 ? (id % 8) * (a.nwg / 8) + id / 8 : id;
  const int qb = w % a.nqb, split = w / a.nqb % a.splits, g = w / a.nqb / a.splits;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int rw = wv % RW, kw = wv / RW;
  const int col = lane % 16, grp = lane / 16, e = col / 4, q4 = 4 * (col % 4);
  const int c0 = split * a.chunk, c1 = min(a.L, c0 + a.chunk);
  const int ntile = (c1 - c0 + KT - 1) / KT;
  const uint16_t* kg = a.k + g * a.k_bs;
  const uint16_t* vg = a.v + g * a.v_bs;

  // K fragment of token block n, step s: rows 32 s + 8 grp + e (and + 4)
  uint32_t koff[NB];
#pragma unroll
  for (int n = 0; n < NB; n++)
    koff[n] = (8 * grp + e) * KT + 16 * ((kw * NB + n) ^ ((e >> 1) | ((grp & 1) << 1))) + q4;
  // V^T fragment of dims 16 dt: tokens 16 j + 4 grp + e of each 32-token step
  const int vrow = 4 * grp + e, vsw = D == 128 ? vrow & 7 : (vrow >> 1) & 3;
  uint32_t voff[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; dt++) voff[dt] = (kw * (KT / KW) + vrow) * D + 16 * (dt ^ vsw) + q4;

  // staging: one load fills 8 K rows (dims) or RPL V rows (tokens); lane l
  // writes physical chunk l % 8 (l % CPR), i.e. the source chunk it stands for
  constexpr int CPR = D / 8, RPL = kWave / CPR, UK = D / 8 / W, UV = KT / RPL / W;
  uint32_t fk[UK], fv[UV];  // byte offsets within a tile
#pragma unroll
  for (int u = 0; u < UK; u++) {
    const int row = 8 * (wv + u * W) + lane / 8, sw = ((row >> 1) & 1) | (((row >> 3) & 1) << 1);
    fk[u] = 2u * (uint32_t)(row * (int)a.k_ld + 8 * ((lane % 8) ^ (2 * sw)));
  }
#pragma unroll
  for (int u = 0; u < UV; u++) {
    const int row = RPL * (wv + u * W) + lane / CPR, sw = D == 128 ? row & 7 : (row >> 1) & 3;
    fv[u] = 2u * (uint32_t)(row * (int)a.v_ld + 8 * ((lane % CPR) ^ (2 * sw)));
  }
  auto fetch = [&](int t, uint16_t* st) __attribute__((always_inline)) {
    const int tok0 = c0 + t * KT;
    const char* kb = reinterpret_cast<const char*>(kg + tok0);
    const char* vb = reinterpret_cast<const char*>(vg + tok0 * a.v_ld);
    const bool whole = tok0 + KT <= a.L;
#pragma unroll
    for (int u = 0; u < UK; u++) {
      uint32_t off = fk[u];
      if (!whole) {  // tokens past L re-read the last 8 (masked)
        const int row = 8 * (wv + u * W) + lane / 8, sw = ((row >> 1) & 1) | (((row >> 3) & 1) << 1);
        off = 2u * (uint32_t)(row * (int)a.k_ld + min(8 * ((lane % 8) ^ (2 * sw)), a.L - 8 - tok0));
      }
      lds_load16(reinterpret_cast<const uint16_t*>(kb + off), st + 8 * (wv + u * W) * KT);
    }
#pragma unroll
    for (int u = 0; u < UV; u++) {
      uint32_t off = fv[u];
      if (!whole) {  // tokens past L re-read the last one
        const int row = RPL * (wv + u * W) + lane / CPR, sw = D == 128 ? row & 7 : (row >> 1) & 3;
        off = 2u * (uint32_t)(min(row, a.L - 1 - tok0) * (int)a.v_ld + 8 * ((lane % CPR) ^ (2 * sw)));
      }
      lds_load16(reinterpret_cast<const uint16_t*>(vb + off), st + KT * D + RPL * (wv + u * W) * D);
    }
  };
  fetch(0, st0);

  // Q^T as the B operand: column = query row, k = d 32 s + 8 grp .. +7
  uint4 qf[RB][NS];
  const int qr0 = qb * QR + 16 * RB * rw + col;
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int s = 0; s < NS; s++)
      qf[rb][s] = ldg16(a.q + g * a.q_bs + min(qr0 + 16 * rb, a.M - 1) * a.q_ld + 32 * s + 8 * grp);

  f32x4 acc[RB][NDT];  // O^T: row d 16 dt + 4 grp + i, column query row
  float m_i[RB], l_i[RB];  // l: this lane's tokens only until the loop ends
#pragma unroll
  for (int rb = 0; rb < RB; rb++) {
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) acc[rb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    l_i[rb] = 0.f;
    m_i[rb] = -INFINITY;
  }

  auto step = [&](int t, const uint16_t* st, auto edge_c) __attribute__((always_inline)) {
    constexpr bool EDGE = decltype(edge_c)::value;
    const uint16_t* vt = st + KT * D;
    f32x4 sc[RB][NB];
#pragma unroll
    for (int n = 0; n < NB; n++) {
      uint4 kf[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const uint2 lo = lds_tr4(&st[koff[n] + 32 * s * KT]), hi = lds_tr4(&st[koff[n] + (32 * s + 4) * KT]);
        kf[s] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; s++) c = mfma16<DT>(kf[s], qf[rb][s], c);
        if (EDGE) {
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (c0 + t * KT + kw * (KT / KW) + 16 * n + 4 * grp + i >= c1) c[i] = -INFINITY;
        }
        sc[rb][n] = c;
      }
    }
    uint4 pb[RB][NB / 2];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      float mx = -INFINITY;
#pragma unroll
      for (int n = 0; n < NB; n++)
#pragma unroll
        for (int i = 0; i < 4; i++) mx = fmaxf(mx, sc[rb][n][i]);
      mx = max_xor32(max_xor16(mx)) * a.scale_log2;
      // the running max moves only when it grows by more than kLazy
      const bool grow = mx > m_i[rb] + kLazy;
      if (__builtin_amdgcn_ballot_w64(grow)) {
        const float mnew = grow ? mx : m_i[rb];
        const float alpha = m_i[rb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_i[rb] - mnew);
        m_i[rb] = mnew;
        l_i[rb] *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) acc[rb][dt] *= alpha;
      }
      const float mref = m_i[rb] == -INFINITY ? 0.f : m_i[rb];
      // the row sum takes P before it is rounded for P V: an f16 P far below
      // the row's maximum rounds to 0, and many such tokens have a weight
      float p[NB][4], ls = 0.f;
#pragma unroll
      for (int n = 0; n < NB; n++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          p[n][i] = __builtin_amdgcn_exp2f(fmaf(sc[rb][n][i], a.scale_log2, -mref));
          ls += p[n][i];
        }
      l_i[rb] += ls;
      // k slot 8 grp + 4 j + i of step m <-> token 32 m + 16 j + 4 grp + i
#pragma unroll
      for (int m = 0; m < NB / 2; m++)
        pb[rb][m] = make_uint4(pack2<DT>(p[2 * m][0], p[2 * m][1]), pack2<DT>(p[2 * m][2], p[2 * m][3]),
                               pack2<DT>(p[2 * m + 1][0], p[2 * m + 1][1]),
                               pack2<DT>(p[2 * m + 1][2], p[2 * m + 1][3]));
    }
#pragma unroll
    for (int m = 0; m < NB / 2; m++)
#pragma unroll
      for (int dt = 0; dt < NDT; dt++) {
        const uint2 lo = lds_tr4(&vt[voff[dt] + 32 * m * D]), hi = lds_tr4(&vt[voff[dt] + (32 * m + 16) * D]);
        const uint4 vf = make_uint4(lo.x, lo.y, hi.x, hi.y);
#pragma unroll
        for (int rb = 0; rb < RB; rb++) acc[rb][dt] = mfma16<DT>(vf, pb[rb][m], acc[rb][dt]);
      }
  };
  auto tile = [&](int t, const uint16_t* st, uint16_t* next) __attribute__((always_inline)) {
    wait_vm();
    __syncthreads();  // tile t has landed, and every wave is done with tile t - 1
    if (t + 1 < ntile) fetch(t + 1, next);
    if (c0 + (t + 1) * KT <= c1) step(t, st, std::false_type{});
    else step(t, st, std::true_type{});
  };
  for (int t = 0; t < ntile; t += 2) {
    tile(t, st0, st1);
    if (t + 1 < ntile) tile(t + 1, st1, st0);
  }

#pragma unroll
  for (int rb = 0; rb < RB; rb++) l_i[rb] = add_xor32(add_xor16(l_i[rb]));
  auto weight = [](float m, float M) __attribute__((always_inline)) {
    return m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
  };
  if constexpr (KW > 1) {
    static_assert(KW == 2 && RW * RB * NDT * kWave * 16 <= (int)sizeof(st0), "the second token wave's O fits a stage");
    float4* so = reinterpret_cast<float4*>(st0);
    __syncthreads();
    if (kw == 1) {
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
          so[((rw * RB + rb) * NDT + dt) * kWave + lane] =
              make_float4(acc[rb][dt][0], acc[rb][dt][1], acc[rb][dt][2], acc[rb][dt][3]);
        s_ml[rw * RB + rb][lane] = make_float2(m_i[rb], l_i[rb]);
      }
    }
    __syncthreads();
    if (kw == 0) {
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        const float2 ml = s_ml[rw * RB + rb][lane];
        const float M = fmaxf(m_i[rb], ml.x), f0 = weight(m_i[rb], M), f1 = weight(ml.x, M);
        m_i[rb] = M;
        l_i[rb] = l_i[rb] * f0 + ml.y * f1;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) {
          const float4 o = so[((rw * RB + rb) * NDT + dt) * kWave + lane];
          acc[rb][dt] = acc[rb][dt] * f0 + f32x4{o.x, o.y, o.z, o.w} * f1;
        }
      }
    }
  }

  constexpr int REC = QR * (D + 2);
  const int pair = g * a.nqb + qb;
  float* rec0 = a.partial + (size_t)pair * a.splits * REC;
  auto put = [&](int row, int d0, f32x4 v) __attribute__((always_inline)) {
    *reinterpret_cast<uint2*>(a.o + g * a.o_bs + row * a.o_ld + d0) =
        make_uint2(pack2<DT>(v[0], v[1]), pack2<DT>(v[2], v[3]));
  };
  if (kw == 0) {
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      const int row = qr0 + 16 * rb;
      if (row >= a.M) continue;
      if (a.splits == 1) {
        const float inv = l_i[rb] > 0.f ? 1.f / l_i[rb] : 0.f;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) put(row, 16 * dt + 4 * grp, acc[rb][dt] * inv);
      } else {
        const int r = row - qb * QR;
        float* rec = rec0 + (size_t)split * REC;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
          st_agent4(rec + r * D + 16 * dt + 4 * grp,
                    make_float4(acc[rb][dt][0], acc[rb][dt][1], acc[rb][dt][2], acc[rb][dt][3]));
        if (grp == 0) {
          st_agent(rec + QR * D + 2 * r, m_i[rb]);
          st_agent(rec + QR * D + 2 * r + 1, l_i[rb]);
        }
      }
    }
  }
  if (a.splits == 1) return;
  if (!arrive_last(&a.tickets[pair], a.splits)) return;
  const int rows = min(QR, a.M - qb * QR);
  for (int i = tid; i < rows * (D / 4); i += 64 * W) {
    const int r = i / (D / 4), d0 = i % (D / 4) * 4;
    float M = -INFINITY, l = 0.f;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.splits; s0 += 8) {
      float mv[8], lv[8];
      float4 ov[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {  // past the last split: its record, with weight 0
        const float* rec = rec0 + (size_t)min(s0 + u, a.splits - 1) * REC;
        mv[u] = ld_agent(rec + QR * D + 2 * r);
        lv[u] = ld_agent(rec + QR * D + 2 * r + 1);
        ov[u] = ld_agent4(rec + r * D + d0);
      }
      float mb = M;
#pragma unroll
      for (int u = 0; u < 8; u++) mb = fmaxf(mb, mv[u]);
      const float f = weight(M, mb);
      l *= f;
      o *= f;
#pragma unroll
      for (int u = 0; u < 8; u++) {
        if (s0 + u < a.splits) {
          const float fu = weight(mv[u], mb);
          l += lv[u] * fu;
          o += f32x4{ov[u].x, ov[u].y, ov[u].z, ov[u].w} * fu;
        }
      }
      M = mb;
    }
    put(qb * QR + r, d0, o * (l > 0.f ? 1.f / l : 0.f));
  }
}

struct Plan {
  int cfg, nqb, splits, chunk;
  size_t bytes;  // split records
};

// Rows per workgroup and token splits.  32 rows with two token waves is the
// fastest tile while the tokens have to be split to fill the chip: the last
// workgroup merges all splits of its rows, so small tiles merge in parallel
// (16 groups of 256 rows over 4096 tokens, d = 64: 19.5 us, 22.4 with 64 rows,
// 28.5 with 128, 28.8 with 16, all before the reads' waits were loosened).  Without splits a fragment read should feed
// more rows: 64 (8 groups of 4096 rows, 2048 tokens, d = 128: 56 us, 72 with
// 32 rows), or 128 at d = 64 (16 groups: 53 us, 66 with 64 rows); at d = 128
// 128 rows spill registers.  Two workgroups per CU and at least 256 tokens per
// split: 256 workgroups took 27 us in the first case, 128-token splits 21 us
// instead of 15.5 for 2 groups.
static Plan plan(int G, int M, int L, int d) {
  constexpr long kTarget = 512;
  constexpr int kMinTiles = 4;
  constexpr int kRows[4] = {16, 32, 64, 128};
  auto pairs = [&](int c) { return (long)G * ((M + kRows[c] - 1) / kRows[c]); };
  Plan p;
  p.cfg = M <= 16 ? 0 : d == 64 && pairs(3) >= kTarget ? 3 : pairs(2) >= kTarget ? 2 : 1;
  const int qr = kRows[p.cfg];
  p.nqb = (M + qr - 1) / qr;
  const long np = pairs(p.cfg), tiles = (L + KT - 1) / KT, most = (tiles + kMinTiles - 1) / kMinTiles;
  // np < kTarget where it splits, so every pair has a ticket
  long sp = (kTarget + np - 1) / np;
  if (sp > most) sp = most;
  p.chunk = (int)((tiles + sp - 1) / sp) * KT;
  p.splits = (L + p.chunk - 1) / p.chunk;
  p.bytes = p.splits > 1 ? (size_t)np * p.splits * qr * (d + 2) * sizeof(float) : 0;
  return p;
}
static_assert(512 <= kMaxTickets, "a ticket per pair that splits");

template <int DT, int D>
static void launch(const Args& a, int cfg, hipStream_t st) {
  const dim3 grid(a.nwg);
  if (cfg == 0) hipLaunchKernelGGL((graph_attn_kernel<DT, D, 1, 2, 1>), grid, dim3(128), 0, st, a);
  else if (cfg == 1) hipLaunchKernelGGL((graph_attn_kernel<DT, D, 2, 2, 1>), grid, dim3(256), 0, st, a);
  else if (cfg == 2) hipLaunchKernelGGL((graph_attn_kernel<DT, D, 4, 1, 1>), grid, dim3(256), 0, st, a);
  else if constexpr (D == 64) hipLaunchKernelGGL((graph_attn_kernel<DT, D, 4, 1, 2>), grid, dim3(256), 0, st, a);
}

}  // namespace ga

bool graph_attn_direct(int G, int M, int L, int d, const long long* sq, const long long* sk, const long long* sv,
                       const long long* so) {
  if (d != 64 && d != 128) return false;
  if (L % 8 || sq[2] != 1 || sk[2] != 1 || sv[2] != 1 || so[2] != 1) return false;
  for (const long long* s : {sq, sk, sv, so})
    if (s[0] % 8 || s[1] % 8 || s[0] < 0 || s[1] < 0) return false;
  if (sk[1] >= (1 << 22) || sv[1] >= (1 << 22)) return false;  // 32-bit byte offsets within a tile
  const ga::Plan p = ga::plan(G, M, L, d);
  if ((long long)G * p.nqb * p.splits >= (1ll << 31)) return false;
  if (d == 64) return true;
  // d = 128: up to 16 rows (a power of two) stay on the decode kernel, whose
  // results equal paged decode's bit for bit.  From 1024 of its workgroups on
  // the prefill kernel fills the chip and, likewise, equals the prompt operator
  // bit for bit; below that the packing passes and its idle CUs cost more (8
  // groups of 4096 rows, 512 workgroups: 92 us against 56 us here).
  if (M <= 16 && (M & (M - 1)) == 0) return false;
  return (long long)G * ((M + 63) / 64) < 1024;
}

size_t graph_attn_direct_workspace(int G, int M, int L, int d) { return kTicketBytes + ga::plan(G, M, L, d).bytes; }

void graph_attn_plan(int G, int M, int L, int d, int* rows_chunk_splits) {
  const ga::Plan p = ga::plan(G, M, L, d);
  rows_chunk_splits[0] = 16 << p.cfg;
  rows_chunk_splits[1] = p.chunk;
  rows_chunk_splits[2] = p.splits;
}

int graph_attn_launch(const char* nm, const void* q, const void* k, const void* v, void* out, int G, int M, int L,
                      int d, const long long* sq, const long long* sk, const long long* sv, const long long* so,
                      float scale, int dtype, void* workspace, hipStream_t st) {
  if (!(scale > 0.f)) return fail(YR_E_INVALID, "%s: scale must be positive", nm);
  const ga::Plan p = ga::plan(G, M, L, d);
  ga::Args a;
  a.q = (const uint16_t*)q;
  a.k = (const uint16_t*)k;
  a.v = (const uint16_t*)v;
  a.o = (uint16_t*)out;
  a.q_bs = sq[0];
  a.k_bs = sk[0];
  a.v_bs = sv[0];
  a.o_bs = so[0];
  a.q_ld = sq[1];
  a.k_ld = sk[1];
  a.v_ld = sv[1];
  a.o_ld = so[1];
  a.tickets = (uint32_t*)workspace;
  a.partial = (float*)((char*)workspace + kTicketBytes);
  a.G = G;
  a.M = M;
  a.L = L;
  a.nqb = p.nqb;
  a.splits = p.splits;
  a.chunk = p.chunk;
  a.nwg = G * p.nqb * p.splits;
  a.scale_log2 = kLog2e * scale;
  const bool bf = dtype == YR_DTYPE_BF16;
  if (d == 64) bf ? ga::launch<DT_BF16, 64>(a, p.cfg, st) : ga::launch<DT_F16, 64>(a, p.cfg, st);
  else bf ? ga::launch<DT_BF16, 128>(a, p.cfg, st) : ga::launch<DT_F16, 128>(a, p.cfg, st);
  YR_CHECK_LAUNCH(nm);
  return YR_OK;
}

}  // namespace yr
