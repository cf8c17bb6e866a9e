// Flash-attention TRAINING backward (causal, GQA, bf16) for CDNA4 (gfx950).
//
// FA2-style recompute backward in two dispatches over LDS tiles of 64 rows
// (flash_tile.h), double-buffered as in the forward:
//   1. fa_bwd_dq: a wave owns 32 query rows and walks the keys up to them.
//        D    = rowsum(dO . O), also left in memory for 2.
//        S^T  = K Q^T, P^T = exp(scale S^T - LSE)           C[key][qrow]
//        dP^T = V dO^T, dS^T = P^T (dP^T - D)               C[key][qrow]
//        dQ^T += K^T dS^T                                   C[d][qrow]
//   2. fa_bwd_dkdv: a wave owns 32 keys and walks the queries from them on.
//        S  = Q K^T, P = exp(scale S - LSE)                 C[qrow][key]
//        dP = dO V^T, dS = P (dP - D)                       C[qrow][key]
//        dV^T += dO^T P, dK^T += Q^T dS                     C[d][key]
//   The factor `scale` of dQ and dK is applied to the sums.
//
// LSE and D enter as the first value of the accumulators (-LSE / scale, -D), so
// they cost no registers of their own. Scores stand in registers in the order
// in which the transposed reads take the rows, and are the next product's
// operand as they are. GQA: dK/dV are computed per q-head ([B,S,Hq,DH]); the
// group-sum to Hkv heads happens in the Python wrapper (ops/attention.py).
//
// What bounds it: the matrix cores, of whose time the exponentials, products
// and roundings between take half as much again; LDS reads (32 KB per 32 MFMA
// and wave) come next. dK/dV of 128 columns hold 128 registers of sums and 64 of
// operands: with one wave per SIMD (360 registers) they beat two (256, which
// spill 84): 7931 tokens, 32 query and 8 kv heads, 2068 against 3253 us.
// Measured, both kernels, before (tiles through registers, transposed copies
// made in LDS, one element at a time) and now:
//   3001 tokens, 32 query and 8 kv heads of 128    1864 -> 344 us, 751 TF/s
//   4 x 512 tokens, 32 heads of 128                 284 ->  79 us
//   4000 tokens, 32 heads of 64                     941 -> 260 us, 883 TF/s
// Since then, with loads to LDS that the compiler does not wait for, operands read
// ahead, and dK/dV's whole tiles in slots of a product and what stands beside it: 302 ->
// 283, 71 -> 69; 512 tokens, 32 heads of 128 42.5 -> 39.6. dQ in slots spills (256
// registers, two waves a SIMD): 333 us both kernels.
//
// mfma_f32_32x32x16_bf16 layouts:
//   A[i][k]: i = lane&31, k = (lane>>5)*8 + e
//   B[k][j]: j = lane&31, k = (lane>>5)*8 + e
//   C[i][j]: j = lane&31, i = (r&3) + 8*(r>>2) + 4*(lane>>5)

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <type_traits>

#include "flash_tile.h"

namespace {

using namespace flash;

constexpr float LOG2E = 1.4426950408889634f;

struct Args {
  const uint16_t *q, *k, *v, *dout, *out;
  const float *lse;                     // [B, Hq, S]
  float *dvec;                          // [B, Hq, S]
  uint16_t *dq, *dk, *dv;               // per q-head
  int B, S, Hq, Hkv;
  // elements between the tokens of q, of k and v, of dq, of dk and dv
  int64_t q_stride, kv_stride, dq_stride, dkv_stride;
  float scale;
};

// A row's operands along DH, from memory.
template <int DH>
RB_DEV void load_row(bf16x8v *f, const uint16_t *row, int hi) {
#pragma unroll
  for (int ks = 0; ks < DH / 16; ++ks)
    f[ks] = *reinterpret_cast<const bf16x8v *>(row + ks * 16 + hi * 8);
}

// C[d][col] times `scale` -> 16-bit rows.
template <int DH>
RB_DEV void store_row(uint16_t *row, const f32x16v *acc, float scale, int hi) {
#pragma unroll
  for (int dt = 0; dt < DH / 32; ++dt)
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      uint2 w;
      w.x = pack2(acc[dt][rq * 4] * scale, acc[dt][rq * 4 + 1] * scale);
      w.y = pack2(acc[dt][rq * 4 + 2] * scale, acc[dt][rq * 4 + 3] * scale);
      *reinterpret_cast<uint2 *>(row + dt * 32 + 8 * rq + 4 * hi) = w;
    }
}

// Scores count scale times; with a scale of zero they count once and Q is
// cleared, so that hidden ones stay at minus infinity.
RB_DEV float unit(float scale) { return scale == 0.0f ? 1.0f : scale; }

template <int DH>
RB_DEV void clear_if(bool yes, bf16x8v *f) {
  if (!yes) return;
#pragma unroll
  for (int ks = 0; ks < DH / 16; ++ks) f[ks] = (bf16x8v)(__bf16)0.0f;
}

// ORDERED: the counterpart of the ordered forward (attention_prefill.hip), with
// one order of its roundings too, as gradients make the next step's weights:
// rows in their own order, natural exponentials of scores less LSE, dP less D,
// each dS times the factor, D summed by quarters of a row. us, both kernels, 12
// heads of 64, 4 x 512 and 2047 tokens: 32 and 91, otherwise 28 and 77.
template <int DH, int NW, bool ORDERED>
__global__ __launch_bounds__(NW * 64, 2) void fa_bwd_dq_kernel(Args a) {
  constexpr int KSTEPS = DH / 16, DTILES = DH / 32;
  constexpr int QT = NW * 32, TILE = tile_bytes<DH>();
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, hi = lane >> 5, col = lane & 31;
  const int S = a.S;
  const Place at = place(blockIdx.x, (S + QT - 1) / QT, a.Hq, a.Hkv, a.B,
                         true);
  const int h_kv = at.head / (a.Hq / a.Hkv);
  const int wrow = at.tile * QT + wid * 32;
  const int qrow = wrow + col;
  const bool q_valid = qrow < S;

  const int64_t kv_stride = a.kv_stride;
  const int64_t kv0 = (int64_t)at.batch * S * kv_stride + h_kv * DH;
  const uint16_t *kb = a.k + kv0, *vb = a.v + kv0;
  const TileLoad<DH, NW> load(wid, lane, kv_stride);
  const int n_tiles = (min(S, at.tile * QT + QT) + ROWS - 1) / ROWS;
  load(kb, 0, S, smem, wid);
  load(vb, 0, S, smem + TILE, wid);

  const int64_t token = (int64_t)at.batch * S + (q_valid ? qrow : 0);
  const int64_t row0 = (token * a.Hq + at.head) * DH;    // of dout, out
  const int64_t stat = ((int64_t)at.batch * a.Hq + at.head) * S + qrow;
  bf16x8v qf[KSTEPS], dof[KSTEPS];
  load_row<DH>(qf, a.q + token * a.q_stride + at.head * DH, hi);
  clear_if<DH>(a.scale == 0.0f, qf);
  load_row<DH>(dof, a.dout + row0, hi);
  float dvec = 0.0f;
  if constexpr (ORDERED) {
    float part[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      part[c] = 0.0f;
#pragma unroll
      for (int v = 0; v < DH / 32; ++v) {
        float o[8], d[8];
        rb::VIO<uint16_t>::load(a.out + row0 + c * (DH / 4) + v * 8, o);
        rb::VIO<uint16_t>::load(a.dout + row0 + c * (DH / 4) + v * 8, d);
#pragma unroll
        for (int e = 0; e < 8; ++e) part[c] += o[e] * d[e];
      }
    }
    dvec = (part[0] + part[1]) + (part[2] + part[3]);
  } else {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const bf16x8v o = *reinterpret_cast<const bf16x8v *>(
          a.out + row0 + ks * 16 + hi * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) dvec += (float)o[e] * (float)dof[ks][e];
    }
    dvec += __shfl_xor(dvec, 32, 64);
  }
  if (q_valid && hi == 0) a.dvec[stat] = dvec;
  const float by = unit(a.scale), to2 = by * LOG2E;
  const float lse = q_valid ? a.lse[stat] : 0.0f;
  const float s0 = ORDERED ? 0.0f : -lse / by;
  const float d0 = ORDERED ? 0.0f : -dvec;

  f32x16v acc[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) acc[dt] = (f32x16v)(0.0f);

  auto keys = [&](const char *kt, const char *vt, int kbase, int r0,
                  auto masked) {
    f32x16v s = (f32x16v)(s0), dp = (f32x16v)(d0);
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          row_frag<DH>(kt, r0, ks, col, hi), qf[ks], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          row_frag<DH>(vt, r0, ks, col, hi), dof[ks], dp, 0, 0, 0);
    }
    // (ordered too: us of both kernels without and with, 12 heads of 64: 2000 tokens 93.5
    // and 87.2, 1000 47.5 and 45.1, 3 x 1000 58.0 and 55.0; 32 heads, 2000 106.2 and 101.0,
    // 4 x 512 42.3 and 41.6, 3 x 1000 82.9 and 85.1)
    reads_ahead<2 * KSTEPS, 4>();
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float p = ORDERED ? __expf(s[r] * by - lse)
                        : __builtin_amdgcn_exp2f(s[r] * to2);
      if constexpr (decltype(masked)::value)
        if (kbase + (r & 3) + 8 * (r >> 2) + 4 * hi > qrow) p = 0.0f;
      s[r] = ORDERED ? p * (dp[r] - dvec) * a.scale : p * dp[r];
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8v ds = score_frag<ORDERED>(s, ks);
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            column_frag<DH, ORDERED>(kt, r0 + ks * 16, dt, lane), ds, acc[dt],
            0, 0, 0);
    }
  };
  // waits for tile t and sends for the next one
  auto arrive = [&](int t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                    // nobody reads the other buffer any more
    if (t + 1 < n_tiles) {
      char *next = smem + (~t & 1) * 2 * TILE;
      load(kb, (t + 1) * ROWS, S, next, wid);
      load(vb, (t + 1) * ROWS, S, next + TILE, wid);
    }
  };
  const Walk mine = walk(wrow, S);
  int t = 0;
  for (; t < mine.full; ++t) {
    arrive(t);
    const char *kt = smem + (t & 1) * 2 * TILE;
#pragma unroll
    for (int r0 = 0; r0 < ROWS; r0 += 32)
      keys(kt, kt + TILE, t * ROWS + r0, r0, std::false_type{});
  }
  for (; t < n_tiles; ++t) {
    arrive(t);
    const char *kt = smem + (t & 1) * 2 * TILE;
#pragma unroll
    for (int r0 = 0; r0 < ROWS; r0 += 32)
      if (t * ROWS + r0 <= mine.last)
        keys(kt, kt + TILE, t * ROWS + r0, r0, std::true_type{});
  }
  if (q_valid)
    store_row<DH>(a.dq + token * a.dq_stride + at.head * DH, acc,
                  ORDERED ? 1.0f : a.scale, hi);
}

template <int DH, int NW, bool ORDERED>
__global__ __launch_bounds__(NW * 64, DH == 128 ? 1 : 2)
void fa_bwd_dkdv_kernel(Args a) {
  constexpr int KSTEPS = DH / 16, DTILES = DH / 32;
  constexpr int KT = NW * 32, TILE = tile_bytes<DH>();
  constexpr int STATS = ROWS * 4 * 2;   // bytes of a tile's LSE and D
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  const int S = a.S;
  const Place at = place(blockIdx.x, (S + KT - 1) / KT, a.Hq, a.Hkv, a.B,
                         false);
  const int h_kv = at.head / (a.Hq / a.Hkv);
  const int wkey = at.tile * KT + wid * 32;
  const int key = wkey + col;
  const bool k_valid = key < S;

  const int64_t o_stride = (int64_t)a.Hq * DH;
  const int64_t token0 = (int64_t)at.batch * S;
  const uint16_t *qb = a.q + token0 * a.q_stride + at.head * DH;
  const uint16_t *ob = a.dout + token0 * o_stride + at.head * DH;
  const int64_t stat = ((int64_t)at.batch * a.Hq + at.head) * S;
  const float by = unit(a.scale), to2 = by * LOG2E;
  const TileLoad<DH, NW> load_q(wid, lane, a.q_stride);
  const TileLoad<DH, NW> load_o(wid, lane, o_stride);
  const int tile0 = at.tile * KT / ROWS, n_tiles = (S + ROWS - 1) / ROWS;

  // tile t's rows and statistics; the latter through registers, stored when
  // the tile before it has been worked on
  auto send = [&](int t, char *tile) {
    load_q(qb, t * ROWS, S, tile, wid);
    load_o(ob, t * ROWS, S, tile + TILE, wid);
  };
  char *stats = smem + 4 * TILE;        // two buffers, like the tiles
  auto stat_of = [&](int t) {
    const int row = t * ROWS + (tid & 63);
    if (tid >= 2 * ROWS) return 0.0f;
    // rows past the end: weights of zero
    if constexpr (ORDERED) {
      if (tid >= ROWS) return row < S ? a.dvec[stat + row] : 0.0f;
      return row < S ? a.lse[stat + row] : INFINITY;
    }
    if (tid >= ROWS) return row < S ? -a.dvec[stat + row] : 0.0f;
    return row < S ? -a.lse[stat + row] / by : by < 0.0f ? INFINITY
                                                         : -INFINITY;
  };
  auto keep = [&](int t, float x) {
    if (tid < 2 * ROWS)
      reinterpret_cast<float *>(stats + (t & 1) * STATS)[tid] = x;
  };
  send(tile0, smem + (tile0 & 1) * 2 * TILE);
  keep(tile0, stat_of(tile0));

  bf16x8v kf[KSTEPS], vf[KSTEPS];
  {
    const int64_t row0 =
        (token0 + (k_valid ? key : 0)) * a.kv_stride + h_kv * DH;
    load_row<DH>(kf, a.k + row0, hi);
    clear_if<DH>(a.scale == 0.0f, kf);
    load_row<DH>(vf, a.v + row0, hi);
    // where the compiler sees it: otherwise it waits for these in the loop, and with
    // them for the tiles that are on their way
    __builtin_amdgcn_s_waitcnt(0x0f70);         // vmcnt(0)
  }
  f32x16v acc_dk[DTILES], acc_dv[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) {
    acc_dk[dt] = (f32x16v)(0.0f);
    acc_dv[dt] = (f32x16v)(0.0f);
  }

  // scores and dP of queries r0 .. r0 + 31 of a tile
  auto products = [&](f32x16v &s, f32x16v &dp, f32x16v &lse, f32x16v &dvec,
                      const char *qt, const float *st, int r0) {
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const float4 l = *reinterpret_cast<const float4 *>(
          st + r0 + 8 * rq + 4 * hi);
      const float4 d = *reinterpret_cast<const float4 *>(
          st + ROWS + r0 + 8 * rq + 4 * hi);
      lse[rq * 4] = l.x; lse[rq * 4 + 1] = l.y;
      lse[rq * 4 + 2] = l.z; lse[rq * 4 + 3] = l.w;
      dvec[rq * 4] = d.x; dvec[rq * 4 + 1] = d.y;
      dvec[rq * 4 + 2] = d.z; dvec[rq * 4 + 3] = d.w;
    }
    s = ORDERED ? (f32x16v)(0.0f) : lse;
    dp = ORDERED ? (f32x16v)(0.0f) : dvec;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          row_frag<DH>(qt, r0, ks, col, hi), kf[ks], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          row_frag<DH>(qt + TILE, r0, ks, col, hi), vf[ks], dp, 0, 0, 0);
    }
  };
  // P and dS, of queries qbase ..
  auto weigh = [&](f32x16v &s, f32x16v &dp, const f32x16v &lse,
                   const f32x16v &dvec, int qbase, auto masked) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float p = ORDERED ? __expf(s[r] * by - lse[r])
                        : __builtin_amdgcn_exp2f(s[r] * to2);
      if constexpr (decltype(masked)::value)
        if (qbase + (r & 3) + 8 * (r >> 2) + 4 * hi < key) p = 0.0f;
      s[r] = p;
      dp[r] = ORDERED ? p * (dp[r] - dvec[r]) * a.scale : dp[r] * p;
    }
  };
  auto add = [&](const f32x16v &s, const f32x16v &dp, const char *qt, int r0) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const bf16x8v pf = score_frag<ORDERED>(s, ks);
      const bf16x8v dsf = score_frag<ORDERED>(dp, ks);
#pragma unroll
      for (int dt = 0; dt < DTILES; ++dt) {
        acc_dv[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            column_frag<DH, ORDERED>(qt + TILE, r0 + ks * 16, dt, lane), pf,
            acc_dv[dt], 0, 0, 0);
        acc_dk[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            column_frag<DH, ORDERED>(qt, r0 + ks * 16, dt, lane), dsf,
            acc_dk[dt], 0, 0, 0);
      }
    }
  };
  auto queries = [&](const char *qt, const float *st, int qbase, int r0,
                     auto masked) {
    f32x16v s, dp, lse, dvec;
    products(s, dp, lse, dvec, qt, st, r0);
    weigh(s, dp, lse, dvec, qbase, masked);
    add(s, dp, qt, r0);
  };
  // A whole tile that is seen whole: its 8 KSTEPS products, each with what is issued
  // beside it. A SIMD has one wave of these, whose vector instructions (weights of a
  // half, 32 queries) take half as long as its products, and which does both at a
  // time only where they stand in turns; operands are read AHEAD products ahead.
  auto tile_of = [&](const char *qt, const float *st) {
    constexpr int N = 2 * KSTEPS, AHEAD = 8, SUMS = 2 * DTILES;
    static_assert(N == 2 * SUMS && 16 % N == 0, "as many products either way");
    f32x16v s[2], dp[2];
    bf16x8v ring[AHEAD], pf[2][2], df[2][2];
    auto statistics = [&](auto half) {
      constexpr int u = decltype(half)::value;
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const float4 l = *reinterpret_cast<const float4 *>(
            st + u * 32 + 8 * rq + 4 * hi);
        const float4 d = *reinterpret_cast<const float4 *>(
            st + ROWS + u * 32 + 8 * rq + 4 * hi);
        s[u][rq * 4] = l.x; s[u][rq * 4 + 1] = l.y;
        s[u][rq * 4 + 2] = l.z; s[u][rq * 4 + 3] = l.w;
        dp[u][rq * 4] = d.x; dp[u][rq * 4 + 1] = d.y;
        dp[u][rq * 4 + 2] = d.z; dp[u][rq * 4 + 3] = d.w;
      }
    };
    auto read = [&](auto at) {
      constexpr int q = decltype(at)::value, u = q / N % 2, i = q % N;
      const char *tile = qt + (q < 2 * N ? i % 2 : 1 - i % 2) * TILE;
      if constexpr (q < 2 * N)
        ring[q % AHEAD] = row_frag<DH>(tile, u * 32, i / 2, col, hi);
      else
        ring[q % AHEAD] = column_frag<DH>(tile, u * 32 + i / SUMS * 16,
                                          i % SUMS / 2, lane);
    };
    // elements of half u that stand beside product i
    auto weights = [&](auto half, auto at) {
      constexpr int u = decltype(half)::value, i = decltype(at)::value;
      constexpr int E = 16 / N, r0 = (i - 2) * E, r1 = i + 1 == N ? 16 : r0 + E;
#pragma unroll
      for (int r = r0; r < r1; ++r) {
        s[u][r] = __builtin_amdgcn_exp2f(s[u][r] * to2);
        dp[u][r] *= s[u][r];
        if (r % 8 == 7) {
          pf[u][r / 8] = score_frag(s[u], r / 8);
          df[u][r / 8] = score_frag(dp[u], r / 8);
        }
      }
    };
    auto slot = [&](auto at) __attribute__((always_inline)) {
      constexpr int q = decltype(at)::value, u = q / N % 2, i = q % N;
      __builtin_amdgcn_sched_barrier(0);
      const bf16x8v x = ring[q % AHEAD];
      if constexpr (q < 2 * N) {
        f32x16v &c = i % 2 == 0 ? s[u] : dp[u];
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            x, i % 2 == 0 ? kf[i / 2] : vf[i / 2], c, 0, 0, 0);
      } else {
        f32x16v &c = i % 2 == 0 ? acc_dv[i % SUMS / 2] : acc_dk[i % SUMS / 2];
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            x, i % 2 == 0 ? pf[u][i / SUMS] : df[u][i / SUMS], c, 0, 0, 0);
      }
      if constexpr (q + AHEAD < 4 * N)
        read(std::integral_constant<int, q + AHEAD>());
      if constexpr (q == 2) statistics(std::integral_constant<int, 1>());
      // of the first half beside the second one's scores, of the second beside the
      // first one's sums, two products behind the last that they need
      if constexpr ((q / N == 1 || q / N == 2) && i >= 2)
        weights(std::integral_constant<int, q / N - 1>(),
                std::integral_constant<int, i>());
      __builtin_amdgcn_sched_barrier(0);
    };
    statistics(std::integral_constant<int, 0>());
    each<AHEAD>(read);
    each<4 * N>(slot);
  };
  auto step = [&](int t, auto masked) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                    // nobody reads the other buffers any more
    float next = 0.0f;
    if (t + 1 < n_tiles) {
      send(t + 1, smem + (~t & 1) * 2 * TILE);
      next = stat_of(t + 1);
    }
    const char *qt = smem + (t & 1) * 2 * TILE;
    const float *st = reinterpret_cast<const float *>(stats +
                                                      (t & 1) * STATS);
    if constexpr (!ORDERED && !decltype(masked)::value) {
      tile_of(qt, st);
    } else {
#pragma unroll
      for (int r0 = 0; r0 < ROWS; r0 += 32)
        if (!decltype(masked)::value || t * ROWS + r0 + 31 >= wkey)
          queries(qt, st, t * ROWS + r0, r0, masked);
    }
    if (t + 1 < n_tiles) keep(t + 1, next);
  };
  // tiles that some of the workgroup's keys do not see whole, then the others
  const int diagonal = min(n_tiles, (at.tile * KT + KT + ROWS - 1) / ROWS);
  int t = tile0;
  for (; t < diagonal; ++t) step(t, std::true_type{});
  for (; t < n_tiles; ++t) step(t, std::false_type{});

  if (k_valid) {
    const int64_t row0 = (token0 + key) * a.dkv_stride + at.head * DH;
    store_row<DH>(a.dk + row0, acc_dk, ORDERED ? 1.0f : a.scale, hi);
    store_row<DH>(a.dv + row0, acc_dv, 1.0f, hi);
  }
}

template <int DH, int NW, bool ORDERED = false>
void launch_bwd(const Args &a, hipStream_t stream) {
  constexpr size_t sh_dq = 4 * tile_bytes<DH>();
  constexpr size_t sh_dkdv = sh_dq + 2 * ROWS * 4 * 2;
  static const bool once =
      hipFuncSetAttribute(
          reinterpret_cast<const void *>(&fa_bwd_dq_kernel<DH, NW, ORDERED>),
          hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh_dq) ==
          hipSuccess &&
      hipFuncSetAttribute(
          reinterpret_cast<const void *>(&fa_bwd_dkdv_kernel<DH, NW, ORDERED>),
          hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh_dkdv) ==
          hipSuccess;
  TORCH_CHECK(once, "fa_bwd: LDS size");
  const int64_t grid =
      (int64_t)((a.S + NW * 32 - 1) / (NW * 32)) * a.Hq * a.B;
  TORCH_CHECK(grid < (int64_t)1 << 31, "fa_bwd: grid");
  hipLaunchKernelGGL((fa_bwd_dq_kernel<DH, NW, ORDERED>), dim3((unsigned)grid),
                     dim3(NW * 64), sh_dq, stream, a);
  hipLaunchKernelGGL((fa_bwd_dkdv_kernel<DH, NW, ORDERED>), dim3((unsigned)grid),
                     dim3(NW * 64), sh_dkdv, stream, a);
}

void launch_bwd(int64_t DH, const Args &a, bool ordered = false) {
  auto stream = at::hip::getCurrentHIPStream();
  // Workgroups of two waves while there are too few tiles of 32 rows for four
  // waves on every CU (us for 2 and 4 waves: 200 tokens, 12 heads of 64, 84
  // tiles, 17 and 19; 512 tokens, 32 heads of 128, 512 tiles, 48 and 50; four
  // times those 81 and 79).
  const bool few = (int64_t)(a.S + 31) / 32 * a.Hq * a.B <= 512;
  if (ordered)
    few ? launch_bwd<64, 2, true>(a, stream)
        : launch_bwd<64, 4, true>(a, stream);
  else if (DH == 128)
    few ? launch_bwd<128, 2>(a, stream) : launch_bwd<128, 4>(a, stream);
  else
    few ? launch_bwd<64, 2>(a, stream) : launch_bwd<64, 4>(a, stream);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host wrappers
// ---------------------------------------------------------------------------

std::vector<at::Tensor> fa_bwd(at::Tensor dout, at::Tensor q, at::Tensor k,
                               at::Tensor v, at::Tensor out, at::Tensor lse,
                               double scale, bool ordered) {
  TORCH_CHECK(q.is_cuda() && q.is_contiguous() && k.is_contiguous() &&
              v.is_contiguous() && dout.is_contiguous() && out.is_contiguous(),
              "fa_bwd: contiguous GPU tensors");
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "fa_bwd: bf16 only");
  const int B = (int)q.size(0), S = (int)q.size(1), Hq = (int)q.size(2),
            DH = (int)q.size(3);
  const int Hkv = (int)k.size(2);
  TORCH_CHECK(DH == 64 || (DH == 128 && !ordered),
              "fa_bwd: DH must be 64 or 128, ordered 64");
  TORCH_CHECK(lse.scalar_type() == at::kFloat && lse.is_contiguous() &&
              lse.numel() == (int64_t)B * Hq * S, "fa_bwd: lse [B, Hq, S]");
  TORCH_CHECK(Hkv > 0 && Hq % Hkv == 0 &&
              k.sizes() == at::IntArrayRef({B, S, Hkv, DH}) &&
              v.sizes() == k.sizes() && dout.sizes() == q.sizes() &&
              out.sizes() == q.sizes() && k.scalar_type() == at::kBFloat16 &&
              v.scalar_type() == at::kBFloat16 &&
              dout.scalar_type() == at::kBFloat16 &&
              out.scalar_type() == at::kBFloat16, "fa_bwd: shapes, types");
  q = aligned16(q);
  k = aligned16(k);
  v = aligned16(v);
  dout = aligned16(dout);
  out = aligned16(out);

  auto dq = at::empty_like(q);
  // per-q-head dk/dv; group-summed by the caller when Hkv < Hq
  auto dk = at::empty({B, S, Hq, DH}, q.options());
  auto dv = at::empty({B, S, Hq, DH}, q.options());
  auto dvec = at::empty({B, Hq, S}, q.options().dtype(at::kFloat));

  if (dq.numel() == 0) return {dq, dk, dv};
  Args a{};
  a.q = (const uint16_t *)q.data_ptr();
  a.k = (const uint16_t *)k.data_ptr();
  a.v = (const uint16_t *)v.data_ptr();
  a.dout = (const uint16_t *)dout.data_ptr();
  a.out = (const uint16_t *)out.data_ptr();
  a.lse = lse.data_ptr<float>();
  a.dvec = dvec.data_ptr<float>();
  a.dq = (uint16_t *)dq.data_ptr();
  a.dk = (uint16_t *)dk.data_ptr();
  a.dv = (uint16_t *)dv.data_ptr();
  a.B = B; a.S = S; a.Hq = Hq; a.Hkv = Hkv;
  a.scale = (float)scale;
  a.q_stride = a.dq_stride = a.dkv_stride = (int64_t)Hq * DH;
  a.kv_stride = (int64_t)Hkv * DH;
  launch_bwd(DH, a, ordered);
  return {dq, dk, dv};
}

// The same for q, k and v side by side in the rows of y
// [B * S, (Hq + 2 Hkv) * DH]: {dy, dk, dv}. With fewer kv heads than query heads
// dk and dv are per query head ([B * S, Hq, DH]) and their columns of dy are
// not written; else dk and dv are empty.
std::vector<at::Tensor> fa_bwd_qkv(at::Tensor dout, at::Tensor y,
                                   at::Tensor out, at::Tensor lse, int64_t B,
                                   int64_t S, int64_t Hq, int64_t Hkv,
                                   int64_t DH, double scale) {
  const int64_t width = (Hq + 2 * Hkv) * DH;
  TORCH_CHECK(y.is_cuda() && y.is_contiguous() && y.dim() == 2 &&
              y.scalar_type() == at::kBFloat16 && y.size(0) == B * S &&
              y.size(1) == width && Hkv > 0 && Hq % Hkv == 0 &&
              (DH == 64 || DH == 128) &&
              reinterpret_cast<uintptr_t>(y.data_ptr()) % 16 == 0,
              "fa_bwd_qkv: y");
  TORCH_CHECK(dout.is_contiguous() && out.is_contiguous() &&
              dout.numel() == B * S * Hq * DH && out.numel() == dout.numel() &&
              dout.scalar_type() == at::kBFloat16 &&
              out.scalar_type() == at::kBFloat16 && lse.is_contiguous() &&
              lse.scalar_type() == at::kFloat && lse.numel() == B * Hq * S,
              "fa_bwd_qkv: dout, out, lse");
  dout = aligned16(dout);
  out = aligned16(out);
  auto dy = at::empty_like(y);
  const bool grouped = Hq != Hkv;
  auto dk = at::empty({grouped ? B * S : 0, Hq, DH}, y.options());
  auto dv = at::empty_like(dk);
  auto dvec = at::empty({B, Hq, S}, y.options().dtype(at::kFloat));
  if (dy.numel() == 0) return {dy, dk, dv};
  Args a{};
  a.q = (const uint16_t *)y.data_ptr();
  a.k = a.q + Hq * DH;
  a.v = a.k + Hkv * DH;
  a.dout = (const uint16_t *)dout.data_ptr();
  a.out = (const uint16_t *)out.data_ptr();
  a.lse = lse.data_ptr<float>();
  a.dvec = dvec.data_ptr<float>();
  a.dq = (uint16_t *)dy.data_ptr();
  a.dk = grouped ? (uint16_t *)dk.data_ptr() : a.dq + Hq * DH;
  a.dv = grouped ? (uint16_t *)dv.data_ptr() : a.dq + (Hq + Hkv) * DH;
  a.B = (int)B; a.S = (int)S; a.Hq = (int)Hq; a.Hkv = (int)Hkv;
  a.q_stride = a.kv_stride = a.dq_stride = width;
  a.dkv_stride = grouped ? Hq * DH : width;
  a.scale = (float)scale;
  launch_bwd(DH, a);
  return {dy, dk, dv};
}
