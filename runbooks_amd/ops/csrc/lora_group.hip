// Products of LoRA adapters of rank 16 that share their input, for CDNA4
// (gfx950): n <= 3 siblings side by side (q, k, v; gate, up; or one alone).
//
//   y [T, N]  = x [T, K] W^T            (a product of all siblings; where it runs
//                                       in tiles, gemm_tiles.hip, it ends with
//                                       the next but one)
//   t_i       = x A_i^T                                  lora_down
//   y_i      += s t_i B_i^T             (columns of i)   lora_add
//   dt_i      = s dy_i B_i                               lora_down (columns)
//   dB_i      = s dy_i^T t_i                             lora_grad
//   dA_i      = dt_i^T x                                 lora_grad
//   dx       += sum_i dt_i A_i                           lora_add (where the
//                                       product does not take it along)
//
// All are bound by the one large operand (x, y, dy, dx), which each reads
// once for all siblings, and writes once where it is changed; as library
// products with 16 rows or columns, with copies, factors and transposes in
// launches of their own, they took longer. us for 2048 rows, in the library, here
// with loads by registers and a launch for each gradient, and now, of q, k, v of
// 4096 columns and of gate, up of 11008 (x of 4096), and of down (x of 11008):
//   lora_down          19, 18, 7.7    19, 14, 6.5    -, 22, 11
//   lora_add (columns) 26, 18, 18     53, 42, 42
//   lora_down_columns  70, 13, 10     57, 25, 22     -, 7.2, 5.3
//   dB and dA          96, 29, 25     71, 40, 33     -, 30, 22
//   lora_add (sum)     18, 8, 8       18, 8, 8
// and no additions of dx, copies of t or transposes of A around them. (dB and dA take 2, 1
// and 1.5 us less since rows of t and dt go to LDS past the registers, lora_grad_tile.)
//
// mfma layouts: 16x16x32 A[i=l&15][k=(l>>4)*8+e], B[k][j=l&15],
// C[j=l&15][i=(l>>4)*4+r]; 32x32x16 as in flash_tile.h.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>

#include "flash_tile.h"

namespace {

using flash::bf16x8v;
using flash::f32x16v;
typedef __attribute__((ext_vector_type(4))) float f32x4v;

constexpr int R = 16, MOST = 3;

struct Adapters {
  const uint16_t *m[MOST];             // A_i [16, K] or B_i [N_i, 16]
  int start[MOST + 1];                 // first columns of the siblings in y
  int n;
};

RB_DEV bf16x8v load8(const uint16_t *p) {
  return *reinterpret_cast<const bf16x8v *>(p);
}

// 16 columns of 32 rows of a row-major [rows, 16] matrix, rows down: the
// second operand of a 16x16x32 product. `tile` holds the rows, 32 bytes each.
RB_DEV bf16x8v rows_frag(const char *tile, int lane) {
  const int i = lane & 15;
  const char *p = tile + ((lane >> 4) * 8 + (i >> 2)) * 32 + (i & 3) * 8;
  return rb::lds_column8(p, p + 4 * 32);
}

// ---------------------------------------------------------------------------
// t_i = x A_i^T (BY_COLUMNS: dt_i = scale x_i B_i, x_i the sibling's columns).
// 16 rows per workgroup, the contraction split over eight waves, 64 columns at a
// time. What a wave works on it fetches for itself, past the registers into LDS of
// its own, 8 to 18 kB ahead; there are no barriers until the waves' sums.
//
// Bound by what a CU takes out of L2, A with every 16 rows of x. Rows go by 128
// bytes (eight lanes): fetched as the operands lie, 64 bytes of each of 16 rows, at
// a distance that put them all in one channel of L2, three siblings of 4096 took as
// long for 300 rows as for 2048 (16 and 18 us; now 6 and 8). dt needs a second
// workgroup on a CU more than loads further ahead (two siblings of 11008 columns of
// 3001 rows 39 and 37 us, 44 by registers; 132 MB).
// ---------------------------------------------------------------------------
constexpr int DW = 8;

template <bool BY_COLUMNS, int NA> struct Down {
  static constexpr int NACC = BY_COLUMNS ? 1 : NA;
  static constexpr int STAGE = 2048 * (1 + NACC);   // bytes of 64 columns
  static constexpr int LOADS = STAGE / 1024;
  static constexpr int AHEAD = BY_COLUMNS ? 2 : NACC == 1 ? 4 : NACC == 2 ? 3 : 2;
  static constexpr int LDS = DW * AHEAD * STAGE;
};

template <bool BY_COLUMNS, int NA>
__global__ __launch_bounds__(DW * 64) void lora_down_kernel(
    const uint16_t *__restrict__ x, Adapters a, uint16_t *__restrict__ t,
    int64_t T, int K, float scale) {
  using D = Down<BY_COLUMNS, NA>;
  constexpr int NACC = D::NACC;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, i16 = lane & 15, grp = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * 16;
  const int which = BY_COLUMNS ? blockIdx.y : 0;
  const int c0 = BY_COLUMNS ? a.start[which] : 0;
  const int C = BY_COLUMNS ? a.start[which + 1] - c0 : K;

  // rows past the end are zeros
  const rb::u32x4v from_x = rb::buffer(
      x + row0 * K + c0,
      (uint32_t)(((int)min(T - row0, (int64_t)16) - 1) * K + C) * 2);
  rb::u32x4v from_m[NACC];
#pragma unroll
  for (int n = 0; n < NACC; ++n)
    from_m[n] = rb::buffer(a.m[BY_COLUMNS ? which : n],
                           (uint32_t)(BY_COLUMNS ? C * R : R * K) * 2);
  unsigned at_row[2];                  // of eight rows, pieces of 16 bytes mixed
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = i * 8 + (lane >> 3);
    at_row[i] = (unsigned)(row * K * 2 + ((lane & 7) ^ (row >> 1 & 7)) * 16);
  }
  const unsigned mine = wid * (D::AHEAD * D::STAGE);
  auto fetch = [&](int c, int stage) {
    const unsigned to = mine + stage * D::STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      rb::lds_load(from_x, at_row[i], c * 128, to + i * 1024);
#pragma unroll
    for (int n = 0; n < NACC; ++n)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        rb::lds_load(from_m[n],
                     BY_COLUMNS ? (unsigned)(i * 1024 + lane * 16) : at_row[i],
                     c * (BY_COLUMNS ? 2048 : 128),
                     to + (1 + n) * 2048 + i * 1024);
  };

  f32x4v acc[NACC];
#pragma unroll
  for (int n = 0; n < NACC; ++n) acc[n] = (f32x4v)(0.0f);
  // chunks of 64 columns go to the waves by twos, in which the last may lack its
  // second
  const int chunks = C / 64, pairs = (chunks + 1) / 2;
  const int turns = pairs > wid ? (pairs - wid + DW - 1) / DW : 0;
  auto chunk = [&](int j) { return (wid + (j >> 1) * DW) * 2 + (j & 1); };
  const int count = turns * 2 - (turns > 0 && chunk(turns * 2 - 1) >= chunks);
#pragma unroll
  for (int j = 0; j < D::AHEAD; ++j)
    if (j < count) fetch(chunk(j), j);
  int stage = 0;
  for (int j = 0; j < count; ++j) {
    if (j + D::AHEAD <= count)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D::AHEAD - 1) * D::LOADS)
                   : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char *b = smem + mine + stage * D::STAGE;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = i16 * 128 + ((s * 4 + grp) ^ (i16 >> 1)) * 16;
      const bf16x8v xf = *reinterpret_cast<const bf16x8v *>(b + at);
#pragma unroll
      for (int n = 0; n < NACC; ++n) {
        const char *m = b + (1 + n) * 2048;
        acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            xf,
            BY_COLUMNS ? rows_frag(m + s * 1024, lane)
                       : *reinterpret_cast<const bf16x8v *>(m + at),
            acc[n], 0, 0, 0);
      }
    }
    // read before it is written again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (j + D::AHEAD < count) fetch(chunk(j + D::AHEAD), stage);
    stage = stage + 1 == D::AHEAD ? 0 : stage + 1;
  }
  __syncthreads();
  // red[wave][adapter][16 rows][16, padded]
  float *red = reinterpret_cast<float *>(smem);
#pragma unroll
  for (int n = 0; n < NACC; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      red[((wid * NACC + n) * 16 + grp * 4 + r) * 17 + i16] = acc[n][r];
  __syncthreads();
  for (int e = threadIdx.x; e < NACC * 256; e += DW * 64) {
    const int n = e >> 8, row = e >> 4 & 15, r = e & 15;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < DW; ++w) sum += red[((w * NACC + n) * 16 + row) * 17 + r];
    if (row0 + row < T)
      t[((which + n) * T + row0 + row) * R + r] = rb::f32_to_bf16(sum * scale);
  }
}

// ---------------------------------------------------------------------------
// y_i += scale t_i B_i^T per sibling's columns, or (SUM) y += sum_i t_i A_i.
// 256 columns per workgroup, 32 rows at a time; products through LDS, so that
// a row is changed 512 bytes at a time. y is on its way during the product.
// ---------------------------------------------------------------------------
constexpr int AC = 256;

template <bool SUM, int NA>
__global__ __launch_bounds__(256) void lora_add_kernel(
    uint16_t *__restrict__ y, const uint16_t *__restrict__ t, Adapters a,
    int64_t T, int N, float scale, int tiles) {
  __shared__ __attribute__((aligned(16))) float prod[32][AC + 4];
  const int tid = threadIdx.x, wid = tid >> 6, lane = tid & 63;
  const int hi = lane >> 5, col = lane & 31;
  const int c0 = blockIdx.x * AC;
  const int width = min(AC, N - c0);
  // the operands of this wave's two tiles of 32 columns
  bf16x8v bf[2][NA];
  int of[2] = {0, 0};
  if constexpr (SUM) {
    // 16 rows of A_i, columns past the end: the last ones again, through LDS
    uint16_t *rows = reinterpret_cast<uint16_t *>(&prod[0][0]);
    constexpr int RW = AC + 8;
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = i * 8 + (tid >> 5), c = (tid & 31) * 8;
        *reinterpret_cast<uint4 *>(rows + (n * R + r) * RW + c) =
            *reinterpret_cast<const uint4 *>(a.m[n] + (int64_t)r * N +
                                             min(c0 + c, N - 8));
      }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        union { uint16_t u[8]; bf16x8v v; } w;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          w.u[e] = rows[(n * R + hi * 8 + e) * RW + wid * 64 + j * 32 + col];
        bf[j][n] = w.v;
      }
    __syncthreads();
  } else {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = min(c0 + wid * 64 + j * 32, N - 32);
      while (of[j] + 1 < a.n && c >= a.start[of[j] + 1]) ++of[j];
      bf[j][0] = load8(a.m[of[j]] +
                       (int64_t)(c - a.start[of[j]] + col) * R + hi * 8);
    }
  }
  const int rr = tid >> 5, cc = (tid & 31) * 8;
  const bool mine = cc < width;
  for (int b = 0; b < tiles; ++b) {
    const int64_t row0 = ((int64_t)blockIdx.y * tiles + b) * 32;
    if (row0 >= T) return;
    const int64_t row = min(row0 + col, T - 1);
    uint4 old[4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
      old[p] = *reinterpret_cast<const uint4 *>(
          y + min(row0 + p * 8 + rr, T - 1) * N + (mine ? c0 + cc : 0));
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x16v c = (f32x16v)(0.0f);
#pragma unroll
      for (int n = 0; n < NA; ++n)
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            load8(t + ((SUM ? n : of[j]) * T + row) * R + hi * 8), bf[j][n], c,
            0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        prod[(r & 3) + 8 * (r >> 2) + 4 * hi][wid * 64 + j * 32 + col] = c[r];
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (row0 + p * 8 + rr < T && mine) {
        union { uint4 v; uint16_t u[8]; } w;
        w.v = old[p];
        float f[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          f[e] = rb::bf16_to_f32(w.u[e]) + scale * prod[p * 8 + rr][cc + e];
        w.v.x = flash::pack2(f[0], f[1]); w.v.y = flash::pack2(f[2], f[3]);
        w.v.z = flash::pack2(f[4], f[5]); w.v.w = flash::pack2(f[6], f[7]);
        *reinterpret_cast<uint4 *>(y + (row0 + p * 8 + rr) * N + c0 + cc) = w.v;
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Sums over the rows: out[c][r] = sum_t x[t][c] m[t][r], for 64 columns of x and
// a share of its rows, 128 at a time (two LDS tiles of flash_tile.h, a wave per
// 32 rows). dB: m is the t of the columns' sibling, out [c, 16]. dA: m is all
// siblings' dt, out [16 n, c]. fp32 slices, one per share, summed afterwards.
// ---------------------------------------------------------------------------
struct Grad {
  const uint16_t *x, *m;
  float *parts;                        // [shares, elements of out]
  uint16_t *out;
  int C, tiles, shares;
  int64_t total;                       // elements of out
  float scale;
};

template <bool DA>
RB_DEV void lora_grad_tile(const Grad &g, const Adapters &a, int64_t T, int c0,
                           int share, char *smem) {
  const uint16_t *x = g.x, *m = g.m;
  const int C = g.C;
  constexpr int NB = DA ? 2 : 1;       // operands of 32 columns of m
  constexpr int TILE = flash::tile_bytes<64>();
  constexpr int MB = 128 * 32;         // bytes of 128 rows of one m
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  int of = 0;
  if (!DA)
    while (of + 1 < a.n && c0 >= a.start[of + 1]) ++of;
  const int mats = DA ? a.n : 1;
  const int BUF = 2 * TILE + mats * MB;
  const int64_t blocks = (T + 127) / 128;
  const int b0 = (int)(blocks * share / g.shares);
  const int b1 = (int)(blocks * (share + 1) / g.shares);

  // columns past the end: the last ones again, not stored
  const flash::TileLoad<64, 4> load(wid, lane, C);
  const uint16_t *xc = x + min(c0, C - 64);
  auto send = [&](int b, char *buf) {
    load(xc, b * 128, (int)T, buf, wid);
    load(xc, b * 128 + 64, (int)T, buf + TILE, wid);
    // m's rows past the registers too: by them, they were waited for as soon as they
    // were sent for, and what is ahead of them with them (dB and dA of 2048 rows, q, k, v
    // 27.2 and 25.3 us, gate and up 33.7 and 32.8, down 22.9 and 21.4)
    const int64_t row = (int64_t)b * 128;
    const uint32_t bytes = (uint32_t)max(min((int)(T - row), 128), 0) * (R * 2);
    const unsigned to = __builtin_amdgcn_readfirstlane(
        (unsigned)(size_t)(__attribute__((address_space(3))) char *)buf +
        2 * TILE + wid * 1024);
    for (int n = 0; n < mats; ++n)
      rb::lds_load(rb::buffer(m + ((of + n) * T + row) * R, bytes), tid * 16, 0,
                   to + n * MB);
  };
  f32x16v acc[2][NB];
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[d][j] = (f32x16v)(0.0f);
  if (b0 < b1) send(b0, smem);
  for (int b = b0; b < b1; ++b) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    char *buf = smem + ((b - b0) & 1) * BUF;
    if (b + 1 < b1) send(b + 1, smem + ((b - b0 + 1) & 1) * BUF);
    const char *tile = buf + (wid >> 1) * TILE;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int r0 = (wid & 1) * 32 + s * 16;
      bf16x8v mf[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        // columns 16 .. 31 of an operand: the next m, or none
        const int n = min(2 * j + (lane >> 4 & 1), mats - 1);
        const int i = lane & 15;
        const char *p = buf + 2 * TILE + n * MB +
                        ((wid >> 1) * 64 + r0 + 4 * hi + (i >> 2)) * 32 +
                        (i & 3) * 8;
        mf[j] = rb::lds_column8(p, p + 8 * 32);
      }
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const bf16x8v xf = flash::column_frag<64>(tile, r0, d, lane);
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[d][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              xf, mf[j], acc[d][j], 0, 0, 0);
      }
    }
  }
  // sum of the four waves, 32 columns of m at a time: red[wave][column of x][column
  // of m]
  constexpr int RS = 33;
  float *red = reinterpret_cast<float *>(smem);
  const int shift = c0 - min(c0, C - 64);
  const int cols = min(64, C - c0), wide = mats * R;
  float *o = g.parts + share * g.total;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (j * 32 >= wide) break;
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        red[(wid * 64 + d * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi) * RS + col] =
            acc[d][j][r];
    __syncthreads();
    const int here = min(32, wide - j * 32);
    for (int e = tid; e < 64 * here; e += 256) {
      const int c = DA ? e & 63 : e / R, r = DA ? e >> 6 : e % R;
      if (c >= cols) continue;
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) sum += red[(w * 64 + c + shift) * RS + r];
      if (DA) o[(int64_t)(j * 32 + r) * C + c0 + c] = sum;
      else o[(int64_t)(c0 + c) * R + r] = sum;
    }
  }
}

// Both kinds in one launch, and their sums of shares in another: each launch is 4 to
// 5 us, and what one kind leaves idle the other fills (4096 to 4096, 2048 rows: 22 us
// in four launches, 14 in two).
__global__ __launch_bounds__(256) void lora_grad_kernel(Grad db, Grad da,
                                                        Adapters a, int64_t T) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  int at = blockIdx.x;
  if (at < db.tiles * db.shares) {
    lora_grad_tile<false>(db, a, T, at % db.tiles * 64, at / db.tiles, smem);
  } else {
    at -= db.tiles * db.shares;
    lora_grad_tile<true>(da, a, T, at % da.tiles * 64, at / da.tiles, smem);
  }
}

// out = scale * sum of the parts, bf16
__global__ __launch_bounds__(256) void lora_sum_kernel(Grad db, Grad da) {
  int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const bool first = i < db.total;
  const Grad &g = first ? db : da;
  if (!first) i -= db.total;
  if (i >= g.total) return;
  float4 s = *reinterpret_cast<const float4 *>(g.parts + i);
  for (int p = 1; p < g.shares; ++p) {
    const float4 x =
        *reinterpret_cast<const float4 *>(g.parts + p * g.total + i);
    s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
  }
  uint2 w;
  w.x = flash::pack2(s.x * g.scale, s.y * g.scale);
  w.y = flash::pack2(s.z * g.scale, s.w * g.scale);
  *reinterpret_cast<uint2 *>(g.out + i) = w;
}

// Adapters of siblings; `by_rows`: B_i [N_i, 16], whose rows say the columns.
Adapters adapters(const std::vector<at::Tensor> &ms, const at::Tensor &like,
                  bool by_rows, int64_t columns) {
  Adapters a{};
  a.n = (int)ms.size();
  TORCH_CHECK(a.n >= 1 && a.n <= MOST, "lora: 1 to 3 siblings");
  int64_t at = 0;
  for (int i = 0; i < a.n; ++i) {
    const at::Tensor &m = ms[i];
    TORCH_CHECK(m.is_cuda() && m.is_contiguous() && m.dim() == 2 &&
                m.scalar_type() == at::kBFloat16 && m.device() == like.device()
                && m.size(by_rows ? 1 : 0) == R &&
                reinterpret_cast<uintptr_t>(m.data_ptr()) % 16 == 0,
                "lora: adapters of rank 16, bf16");
    if (by_rows) {
      TORCH_CHECK(m.size(0) % 64 == 0 && m.size(0) > 0, "lora: columns");
    } else {
      TORCH_CHECK(m.size(1) == columns, "lora: columns");
    }
    a.m[i] = (const uint16_t *)m.data_ptr();
    a.start[i] = (int)at;
    at += by_rows ? m.size(0) : 0;
  }
  for (int i = a.n; i <= MOST; ++i) a.start[i] = (int)at;
  TORCH_CHECK(!by_rows || at == columns, "lora: columns of the siblings");
  return a;
}

void check_rows(const at::Tensor &x) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.dim() == 2 &&
              x.scalar_type() == at::kBFloat16 && x.size(1) % 64 == 0 &&
              x.size(1) > 0 && x.size(0) > 0 &&
              x.size(0) <= (int64_t)1 << 24 && x.size(1) <= (int64_t)1 << 24 &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "lora: rows [T, 64 k] bf16");
}

void check_t(const at::Tensor &t, int n, int64_t T) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.dim() == 3 &&
              t.scalar_type() == at::kBFloat16 && t.size(0) == n &&
              t.size(1) == T && t.size(2) == R &&
              reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
              "lora: t [n, T, 16]");
}

}  // namespace

template <bool BY_COLUMNS, int NA>
static void run_down(const at::Tensor &x, const Adapters &a, at::Tensor &t,
                     double scale) {
  constexpr int lds = Down<BY_COLUMNS, NA>::LDS;
  auto kernel = lora_down_kernel<BY_COLUMNS, NA>;
  static const bool once =
      hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds) ==
      hipSuccess;
  TORCH_CHECK(once, "lora_down: LDS size");
  const int64_t T = x.size(0);
  hipLaunchKernelGGL(kernel,
                     dim3((unsigned)((T + 15) / 16), BY_COLUMNS ? a.n : 1),
                     dim3(DW * 64), lds, at::hip::getCurrentHIPStream(),
                     (const uint16_t *)x.data_ptr(), a,
                     (uint16_t *)t.data_ptr(), T, (int)x.size(1), (float)scale);
}

// t [n, T, 16] = x A_i^T
at::Tensor lora_down(at::Tensor x, std::vector<at::Tensor> as) {
  check_rows(x);
  const Adapters a = adapters(as, x, false, x.size(1));
  auto t = at::empty({a.n, x.size(0), R}, x.options());
  if (a.n == 1) run_down<false, 1>(x, a, t, 1.0);
  else if (a.n == 2) run_down<false, 2>(x, a, t, 1.0);
  else run_down<false, 3>(x, a, t, 1.0);
  return t;
}

// dt [n, T, 16] = scale dy_i B_i
at::Tensor lora_down_columns(at::Tensor dy, std::vector<at::Tensor> bs,
                             double scale) {
  check_rows(dy);
  const Adapters a = adapters(bs, dy, true, dy.size(1));
  auto t = at::empty({a.n, dy.size(0), R}, dy.options());
  run_down<true, 1>(dy, a, t, scale);
  return t;
}

// y_i += scale t_i B_i^T (sum=False, ms = B_i), y += scale sum_i t_i A_i
void lora_add_(at::Tensor y, at::Tensor t, std::vector<at::Tensor> ms,
               double scale, bool sum) {
  check_rows(y);
  const Adapters a = adapters(ms, y, !sum, y.size(1));
  const int64_t T = y.size(0), N = y.size(1);
  check_t(t, a.n, T);
  // tiles of 32 rows per workgroup: as many as leave 1024 workgroups, 4 at most
  const int64_t wide = (N + AC - 1) / AC, down = (T + 31) / 32;
  const int64_t tiles =
      std::max<int64_t>(std::min<int64_t>(4, wide * down / 1024),
                        (down + 65534) / 65535);
  const dim3 grid((unsigned)wide, (unsigned)((down + tiles - 1) / tiles));
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0,
                       at::hip::getCurrentHIPStream(),
                       (uint16_t *)y.data_ptr(),
                       (const uint16_t *)t.data_ptr(), a, T, (int)N,
                       (float)scale, (int)tiles);
  };
  if (!sum) go(lora_add_kernel<false, 1>);
  else if (a.n == 1) go(lora_add_kernel<true, 1>);
  else if (a.n == 2) go(lora_add_kernel<true, 2>);
  else go(lora_add_kernel<true, 3>);
}

// Sums of x's rows with those of t: `transposed` scale t_i^T x, [16 n, columns],
// otherwise scale x_i^T t_i, [columns, 16].
static Grad grad_of(const at::Tensor &x, const at::Tensor &t, double scale,
                    bool transposed, at::Tensor &out) {
  Grad g{};
  check_rows(x);
  const int64_t T = x.size(0), C = x.size(1);
  const int n = (int)t.size(0);
  TORCH_CHECK(n >= 1 && n <= MOST, "lora_grad: 1 to 3 siblings");
  check_t(t, n, T);
  const int64_t wide = transposed ? n * R : R;
  out = transposed ? at::empty({wide, C}, x.options())
                   : at::empty({C, wide}, x.options());
  g.x = (const uint16_t *)x.data_ptr();
  g.m = (const uint16_t *)t.data_ptr();
  g.out = (uint16_t *)out.data_ptr();
  g.C = (int)C;
  g.tiles = (int)(C / 64);
  g.total = C * wide;
  g.scale = (float)scale;
  // shares of the rows, of at least 128 each, until there are as many workgroups
  // as the CUs' LDS holds (dA of 2048 x 4096, three siblings: 20 us with twice
  // as many, 14 so)
  const int64_t want = transposed ? 512 : 1024;
  g.shares = (int)std::max<int64_t>(
      1, std::min<int64_t>((T + 127) / 128, (want + g.tiles - 1) / g.tiles));
  return g;
}

// Columns of the siblings in what `db` sums up.
static Adapters grad_widths(const std::vector<int64_t> &widths, int n,
                            int64_t C) {
  Adapters a{};
  a.n = n;
  int64_t at = 0;
  TORCH_CHECK((int)widths.size() == n, "lora_grad: widths");
  for (int i = 0; i < n; ++i) {
    TORCH_CHECK(widths[i] > 0 && widths[i] % 64 == 0, "lora_grad: widths");
    a.start[i] = (int)at;
    at += widths[i];
  }
  for (int i = n; i <= MOST; ++i) a.start[i] = (int)at;
  TORCH_CHECK(at == C, "lora_grad: widths");
  return a;
}

static void run_grads(Grad db, Grad da, const Adapters &a, const at::Tensor &x) {
  const int64_t first = db.shares * db.total, second = da.shares * da.total;
  auto parts = at::empty({first + second}, x.options().dtype(at::kFloat));
  db.parts = parts.data_ptr<float>();
  da.parts = db.parts + first;
  auto stream = at::hip::getCurrentHIPStream();
  // two buffers, or the waves' sums
  const size_t shmem = std::max<size_t>(
      2 * (2 * flash::tile_bytes<64>() + (da.tiles ? a.n : 1) * 128 * 32),
      4 * 64 * 33 * 4);
  static const bool once =
      hipFuncSetAttribute(reinterpret_cast<const void *>(&lora_grad_kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          80 * 1024) == hipSuccess;
  TORCH_CHECK(once && shmem <= 80 * 1024, "lora_grad: LDS size");
  hipLaunchKernelGGL(
      lora_grad_kernel,
      dim3((unsigned)(db.tiles * db.shares + da.tiles * da.shares)), dim3(256),
      shmem, stream, db, da, a, x.size(0));
  const int64_t total = db.total + da.total;
  hipLaunchKernelGGL(lora_sum_kernel, dim3((unsigned)((total + 1023) / 1024)),
                     dim3(256), 0, stream, db, da);
}

// One of the two by itself, what lora_grads is tested against (fine-tunes take both).
// transposed=False: scale x_i^T t_i, [columns, 16]; the columns of x belong to
// siblings of `widths`. transposed=True: scale t_i^T x, [16 n, columns].
at::Tensor lora_grad(at::Tensor x, at::Tensor t, std::vector<int64_t> widths,
                     double scale, bool transposed) {
  at::Tensor out;
  const Grad g = grad_of(x, t, scale, transposed, out);
  Adapters a{};
  a.n = (int)t.size(0);
  if (!transposed) a = grad_widths(widths, a.n, x.size(1));
  run_grads(transposed ? Grad{} : g, transposed ? g : Grad{}, a, x);
  return out;
}

// scale dy_i^T t_i, [columns, 16], and dt_i^T x, [16 n, columns].
std::vector<at::Tensor> lora_grads(at::Tensor dy, at::Tensor t, at::Tensor x,
                                   at::Tensor dt, std::vector<int64_t> widths,
                                   double scale) {
  TORCH_CHECK(dy.size(0) == x.size(0) && dy.device() == x.device() &&
              t.size(0) == dt.size(0), "lora_grads: rows");
  at::Tensor b, a;
  const Grad db = grad_of(dy, t, scale, false, b);
  const Grad da = grad_of(x, dt, 1.0, true, a);
  run_grads(db, da, grad_widths(widths, (int)t.size(0), dy.size(1)), x);
  return {b, a};
}
