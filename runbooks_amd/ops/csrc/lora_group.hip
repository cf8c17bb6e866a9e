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
//   dx       += sum_i dt_i A_i                           lora_add
//
// All are bound by the one large operand (x, y, dy, dx), which each reads
// once for all siblings, and writes once where it is changed; as library
// products with 16 rows or columns, with copies, factors and transposes in
// launches of their own, they took longer. us for 2048 rows, before and now,
// of q, k, v of 4096 columns and of gate, up of 11008 (x of 4096):
//   lora_down          19, 18      19, 14
//   lora_add (columns) 26, 18      53, 42
//   lora_down_columns  70, 13      57, 26
//   dB                 76, 15      51, 27
//   dA                 20, 14      20, 13
//   lora_add (sum)     18, 8       18, 8
// and no additions of dx, copies of t or transposes of A around them.
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
// 16 rows per workgroup, the contraction split over eight waves.
// ---------------------------------------------------------------------------
constexpr int DW = 8;

template <bool BY_COLUMNS, int NA>
__global__ __launch_bounds__(DW * 64) void lora_down_kernel(
    const uint16_t *__restrict__ x, Adapters a, uint16_t *__restrict__ t,
    int64_t T, int K, float scale) {
  constexpr int CHUNK = 128;           // columns of a wave's step
  constexpr int NACC = BY_COLUMNS ? 1 : NA;
  __shared__ __attribute__((aligned(16))) char rows[BY_COLUMNS
                                                        ? DW * CHUNK * 32 : 16];
  __shared__ float red[DW][NACC][16][17];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, i16 = lane & 15, grp = lane >> 4;
  const int64_t row0 = (int64_t)blockIdx.x * 16;
  const int which = BY_COLUMNS ? blockIdx.y : 0;
  const int c0 = BY_COLUMNS ? a.start[which] : 0;
  const int C = BY_COLUMNS ? a.start[which + 1] - c0 : K;
  const uint16_t *xr = x + min(row0 + i16, T - 1) * K + c0 + grp * 8;

  f32x4v acc[NACC];
#pragma unroll
  for (int n = 0; n < NACC; ++n) acc[n] = (f32x4v)(0.0f);
  for (int c = wid * CHUNK; c < C; c += DW * CHUNK) {
    bf16x8v xf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      xf[s] = load8(xr + min(c + s * 32, C - 32));
    if constexpr (BY_COLUMNS) {
      char *tile = rows + wid * CHUNK * 32;
      // rows past the end are not multiplied
      const uint16_t *src = a.m[which];
      uint4 b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = i * 64 + lane;            // 16 bytes: half a row
        b[i] = *reinterpret_cast<const uint4 *>(
            src + (int64_t)min(c + at / 2, C - 1) * R + at % 2 * 8);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint4 *>(tile + (i * 64 + lane) * 16) = b[i];
      // the tile is this wave's own
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (c + s * 32 < C)
          acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              xf[s], rows_frag(tile + s * 1024, lane), acc[0], 0, 0, 0);
      __builtin_amdgcn_wave_barrier();
    } else {
#pragma unroll
      for (int n = 0; n < NACC; ++n) {
        const uint16_t *ar = a.m[n] + (int64_t)i16 * K + grp * 8;
#pragma unroll
        for (int s = 0; s < 4; ++s)
          if (c + s * 32 < C)
            acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                xf[s], load8(ar + c + s * 32), acc[n], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int n = 0; n < NACC; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wid][n][grp * 4 + r][i16] = acc[n][r];
  __syncthreads();
  for (int e = threadIdx.x; e < NACC * 256; e += DW * 64) {
    const int n = e >> 8, row = e >> 4 & 15, r = e & 15;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < DW; ++w) sum += red[w][n][row][r];
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
template <bool DA>
__global__ __launch_bounds__(256) void lora_grad_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ m, Adapters a,
    float *__restrict__ out, int64_t T, int C) {
  constexpr int NB = DA ? 2 : 1;       // operands of 32 columns of m
  constexpr int TILE = flash::tile_bytes<64>();
  constexpr int MB = 128 * 32;         // bytes of 128 rows of one m
  constexpr int BUF = 2 * TILE + (DA ? 2 * NB : 1) * MB;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  const int c0 = blockIdx.x * 64;
  int of = 0;
  if (!DA)
    while (of + 1 < a.n && c0 >= a.start[of + 1]) ++of;
  const int mats = DA ? a.n : 1;
  const int64_t shares = gridDim.y, blocks = (T + 127) / 128;
  const int b0 = (int)(blocks * blockIdx.y / shares);
  const int b1 = (int)(blocks * (blockIdx.y + 1) / shares);

  // columns past the end: the last ones again, not stored
  const flash::TileLoad<64, 4> load(wid, lane);
  const uint16_t *xc = x + min(c0, C - 64);
  auto send = [&](int b, char *buf) {
    load(xc, C, b * 128, (int)T, buf, wid);
    load(xc, C, b * 128 + 64, (int)T, buf + TILE, wid);
    // m's rows: 16 bytes a lane, rows past the end as zeros
    for (int n = 0; n < mats; ++n) {
      const uint16_t *src = m + (of + n) * T * R;
      const int64_t row = (int64_t)b * 128 + tid / 2;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (row < T)
        v = *reinterpret_cast<const uint4 *>(src + row * R + tid % 2 * 8);
      *reinterpret_cast<uint4 *>(buf + 2 * TILE + n * MB + tid * 16) = v;
    }
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
    if ((b + 1) * 128 > T) {
      // rows past the end, which m's zeros would not hide if the last row,
      // which they repeat, is not finite
      for (int at = (int)(T - b * 128) * 128 + tid * 16; at < 2 * TILE;
           at += 256 * 16)
        *reinterpret_cast<uint4 *>(buf + at) = make_uint4(0, 0, 0, 0);
      __syncthreads();
    }
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
  // sum of the four waves: red[wave][column of x][column of m]
  __syncthreads();
  constexpr int RS = NB * 32 + 1;
  float *red = reinterpret_cast<float *>(smem);
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        red[(wid * 64 + d * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi) * RS +
            j * 32 + col] = acc[d][j][r];
  __syncthreads();
  const int shift = c0 - min(c0, C - 64);
  const int cols = min(64, C - c0), wide = mats * R;
  float *o = out + blockIdx.y * (int64_t)C * wide;
  for (int e = tid; e < 64 * wide; e += 256) {
    const int c = DA ? e & 63 : e / R, r = DA ? e >> 6 : e % R;
    if (c >= cols) continue;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) sum += red[(w * 64 + c + shift) * RS + r];
    if (DA) o[(int64_t)r * C + c0 + c] = sum;
    else o[(int64_t)(c0 + c) * R + r] = sum;
  }
}

// out = scale * sum of `n` slices, bf16
__global__ __launch_bounds__(256) void lora_sum_kernel(
    const float *__restrict__ parts, uint16_t *__restrict__ out, int n,
    int64_t total, float scale) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  float4 s = *reinterpret_cast<const float4 *>(parts + i);
  for (int p = 1; p < n; ++p) {
    const float4 x = *reinterpret_cast<const float4 *>(parts + p * total + i);
    s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
  }
  uint2 w;
  w.x = flash::pack2(s.x * scale, s.y * scale);
  w.y = flash::pack2(s.z * scale, s.w * scale);
  *reinterpret_cast<uint2 *>(out + i) = w;
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

// t [n, T, 16] = x A_i^T
at::Tensor lora_down(at::Tensor x, std::vector<at::Tensor> as) {
  check_rows(x);
  const Adapters a = adapters(as, x, false, x.size(1));
  const int64_t T = x.size(0);
  auto t = at::empty({a.n, T, R}, x.options());
  const dim3 grid((unsigned)((T + 15) / 16));
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(DW * 64), 0,
                       at::hip::getCurrentHIPStream(),
                       (const uint16_t *)x.data_ptr(), a,
                       (uint16_t *)t.data_ptr(), T, (int)x.size(1), 1.0f);
  };
  if (a.n == 1) go(lora_down_kernel<false, 1>);
  else if (a.n == 2) go(lora_down_kernel<false, 2>);
  else go(lora_down_kernel<false, 3>);
  return t;
}

// dt [n, T, 16] = scale dy_i B_i
at::Tensor lora_down_columns(at::Tensor dy, std::vector<at::Tensor> bs,
                             double scale) {
  check_rows(dy);
  const Adapters a = adapters(bs, dy, true, dy.size(1));
  const int64_t T = dy.size(0);
  auto t = at::empty({a.n, T, R}, dy.options());
  hipLaunchKernelGGL((lora_down_kernel<true, 1>),
                     dim3((unsigned)((T + 15) / 16), a.n), dim3(DW * 64), 0,
                     at::hip::getCurrentHIPStream(),
                     (const uint16_t *)dy.data_ptr(), a,
                     (uint16_t *)t.data_ptr(), T, (int)dy.size(1),
                     (float)scale);
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

// transposed=False: scale x_i^T t_i, [columns, 16]; the columns of x belong to
// siblings of `widths`. transposed=True: scale t_i^T x, [16 n, columns].
at::Tensor lora_grad(at::Tensor x, at::Tensor t, std::vector<int64_t> widths,
                     double scale, bool transposed) {
  check_rows(x);
  const int64_t T = x.size(0), C = x.size(1);
  Adapters a{};
  a.n = (int)t.size(0);
  TORCH_CHECK(a.n >= 1 && a.n <= MOST, "lora_grad: 1 to 3 siblings");
  check_t(t, a.n, T);
  if (!transposed) {
    int64_t at = 0;
    TORCH_CHECK((int)widths.size() == a.n, "lora_grad: widths");
    for (int i = 0; i < a.n; ++i) {
      TORCH_CHECK(widths[i] > 0 && widths[i] % 64 == 0, "lora_grad: widths");
      a.start[i] = (int)at;
      at += widths[i];
    }
    for (int i = a.n; i <= MOST; ++i) a.start[i] = (int)at;
    TORCH_CHECK(at == C, "lora_grad: widths");
  }
  const int64_t wide = transposed ? a.n * R : R;
  const int64_t tiles = C / 64;
  // shares of the rows, of at least 128 each, until there are as many workgroups
  // as the CUs' LDS holds (dA of 2048 x 4096, three siblings: 20 us with twice
  // as many, 14 so)
  const int64_t want = transposed ? 512 : 1024;
  const int64_t shares = std::max<int64_t>(
      1, std::min<int64_t>((T + 127) / 128, (want + tiles - 1) / tiles));
  auto parts = at::empty({shares, C * wide}, x.options().dtype(at::kFloat));
  auto out = transposed ? at::empty({wide, C}, x.options())
                        : at::empty({C, wide}, x.options());
  auto stream = at::hip::getCurrentHIPStream();
  constexpr size_t buf = 2 * flash::tile_bytes<64>();
  const size_t most_t = 2 * (buf + 4 * 128 * 32);
  const size_t red_t = 4 * 64 * 65 * 4, red_f = 4 * 64 * 33 * 4;
  const size_t shmem = transposed ? std::max(most_t, red_t)
                                  : std::max<size_t>(2 * (buf + 128 * 32),
                                                     red_f);
  static const bool once =
      hipFuncSetAttribute(
          reinterpret_cast<const void *>(&lora_grad_kernel<true>),
          hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) ==
          hipSuccess &&
      hipFuncSetAttribute(
          reinterpret_cast<const void *>(&lora_grad_kernel<false>),
          hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) ==
          hipSuccess;
  TORCH_CHECK(once && shmem <= 80 * 1024, "lora_grad: LDS size");
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)tiles, (unsigned)shares),
                       dim3(256), shmem, stream,
                       (const uint16_t *)x.data_ptr(),
                       (const uint16_t *)t.data_ptr(), a,
                       parts.data_ptr<float>(), T, (int)C);
  };
  if (transposed) go(lora_grad_kernel<true>);
  else go(lora_grad_kernel<false>);
  const int64_t total = C * wide;
  hipLaunchKernelGGL(lora_sum_kernel, dim3((unsigned)((total + 1023) / 1024)),
                     dim3(256), 0, stream, parts.data_ptr<float>(),
                     (uint16_t *)out.data_ptr(), (int)shares, total,
                     (float)scale);
  return out;
}
