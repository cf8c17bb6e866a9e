// Decode products that end in the residual (the output projection of attention,
// the second one of an MLP), with the sum and what the next norm needs of it:
//
//   r' = r + x W^T;   y = r' * w;   squares = parts of |r'|^2 of each row
//
// for up to 32 rows x. The norm's 1 / rms is a factor of a whole row, so the
// product that reads y applies it to its results (decode_ends.h): no
// workgroup has to wait for the sums of the others.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <type_traits>

#include "common.h"
#include "decode_ends.h"

namespace {

using ends::bf16x8v;
using ends::f32x4v;
using ends::u32x4v;

constexpr int WAVES = 8, BLOCK = WAVES * 64;

struct Sum {
  const uint16_t *xs;
  const uint8_t *ws;
  const float *scale;           // of W's rows (or null)
  const uint16_t *res, *norm;
  uint16_t *out, *y;
  bool rows;                    // y in rows, else as an operand
  float *squares;
  int M, N, K;
};

// A workgroup takes 16 rows of W and all of their sums, so that nothing is left
// to add up: of a width of 4096 that is a workgroup for every CU. Its eight
// waves take parts of the sums, U kilobytes of W at a time; B blocks of 16
// rows of x (16x16x32 products: A[i=l&15][k=(l>>4)*8+e], B[k][j=l&15],
// C[j=l&15][i=(l>>4)*4+r]). A lane's 16 bytes of e4m3 are of two products.
//
// Bound by the weight stream, by x with many long rows. us in a graph, weights
// out of cache, in parts that the norm's kernel adds up, and here, of 1, 16 and
// 32 rows:
//   4096 x 4096        11.8  7.7   12.7  8.5   13.8 10.3
//   4096 x 11008       21.2 19.3   22.3 21.0   25.2 25.1
//   3072 x 24576       34.5 31.9   37.2 37.6   42.1 49.5
//   4096 x 4096  e4m3   8.8  5.7    9.8  6.1   11.6  8.3
//   4096 x 11008 e4m3  14.0 12.5   15.0 13.0   18.4 18.0
template <bool FP8, int B, int U>
__global__ __launch_bounds__(BLOCK, 1) void decode_res_kernel(Sum a) {
  constexpr int X = FP8 ? 2 : 1;
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, i16 = lane & 15, grp = lane >> 4;
  const int steps = a.K / (32 * X);
  const int s0 = steps * wid / WAVES, s1 = steps * (wid + 1) / WAVES;
  const uint8_t *w = a.ws + (int64_t)(blockIdx.x >> 1) * a.K * (64 / X) +
                     ((blockIdx.x & 1) * 16 + i16) * 16 + grp * 512;
  const uint8_t *x = reinterpret_cast<const uint8_t *>(a.xs) +
                     (FP8 ? (grp >> 1) * 2048 + (grp & 1) * 512 : grp * 512);
  int xrow[B];                          // rows past M: the last one again
#pragma unroll
  for (int b = 0; b < B; ++b) xrow[b] = min(b * 16 + i16, a.M - 1) * 16;

  // this thread's place in the results
  const int em = tid >> 4, en = tid & 15, n = blockIdx.x * 16 + en;
  const int64_t at = (int64_t)min(em, a.M - 1) * a.N + n;
  const float r0 = rb::bf16_to_f32(a.res[at]);
  const float g = rb::bf16_to_f32(a.norm[n]);
  const float scale = a.scale == nullptr ? 1.0f : a.scale[n];

  struct Chunk { u32x4v w[U]; bf16x8v x[U][B][X]; };
  Chunk c0, c1;
  auto load = [&](Chunk &c, int s) {    // past the end: the last one again
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = min(s + u, s1 - 1);
      c.w[u] = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4v *>(w + t * 2048));
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < X; ++i)
          c.x[u][b][i] = ends::load8v(reinterpret_cast<const uint16_t *>(
              x + t * (2048 * X) + i * 1024 + xrow[b]));
    }
  };
  f32x4v acc[B];
#pragma unroll
  for (int b = 0; b < B; ++b) acc[b] = (f32x4v)(0.0f);
  auto multiply = [&](const Chunk &c, int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= s1) continue;
      bf16x8v wv[X];
      if constexpr (FP8) {
        wv[0] = ends::fp8_to_bf16(c.w[u][0], c.w[u][1]);
        wv[1] = ends::fp8_to_bf16(c.w[u][2], c.w[u][3]);
      } else {
        union { u32x4v u; bf16x8v v; } t;
        t.u = c.w[u];
        wv[0] = t.v;
      }
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < X; ++i)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wv[i], c.x[u][b][i], acc[b], 0, 0, 0);
    }
  };
  if (s0 < s1) {
    int s = s0;
    load(c0, s);
    for (; s + 2 * U < s1; s += 2 * U) {
      load(c1, s + U);
      multiply(c0, s);
      load(c0, s + 2 * U);
      multiply(c1, s + U);
    }
    if (s + U < s1) {
      load(c1, s + U);
      multiply(c0, s);
      multiply(c1, s + U);
    } else {
      multiply(c0, s);
    }
  }
  __shared__ float red[WAVES][B][16][17];
#pragma unroll
  for (int b = 0; b < B; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wid][b][grp * 4 + r][i16] = acc[b][r];
  __syncthreads();
  if (em >= min(a.M, 16 * B)) return;   // whole groups of 16 lanes
  float f = 0.0f;
#pragma unroll
  for (int v = 0; v < WAVES; ++v) f += red[v][em >> 4][en][em & 15];
  f = f * scale + r0;
  a.out[at] = rb::f32_to_bf16(f);
  a.y[a.rows ? at : (int64_t)blockIdx.x * 512 + (en >> 3) * 256 + em * 8 +
                        (en & 7)] = rb::f32_to_bf16(f * g);
  float ss = f * f;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if (en == 0) a.squares[(int64_t)em * gridDim.x + blockIdx.x] = ss;
}

// The same of 33 to 64 rows x as they lie, B blocks of 16. x is as long as W's share
// of a workgroup and longer, so all loads go past the registers: a wave has a ring
// of its own in LDS, of AHEAD pieces of 64 columns of x and W, and waits for no
// other. Rows of x go by 128 bytes, their pieces of 16 at their index ^ (row / 2) %
// 8, as in gemm_tiles.hip; W as the operands lie in its copy.
//
// Bound by what a CU takes out of L2, x and W together, and with long rows by W: as
// loads come back in order, W is no further ahead than x (16 to 24 kB a CU). us with
// the sums in parts that the norm adds up, and here: _add_rows in decode_chain.py.
constexpr int ROW_WAVES = 4;

template <int B> struct Ring {
  static constexpr int STAGE = (B + 1) * 2048, LOADS = 2 * B + 2;
  static constexpr int AHEAD = B == 4 ? 3 : 4;
  static constexpr int LDS = ROW_WAVES * AHEAD * STAGE;
};

template <int B>
__global__ __launch_bounds__(ROW_WAVES * 64, 1) void rows_res_kernel(Sum a) {
  using R = Ring<B>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, i16 = lane & 15, grp = lane >> 4;
  const int chunks = a.K / 64;
  const int c0 = chunks * wid / ROW_WAVES, c1 = chunks * (wid + 1) / ROW_WAVES;

  // this thread's places in the results: rows em, em + 16, ..
  const int em = tid >> 4, en = tid & 15, n = blockIdx.x * 16 + en;
  float r0[B];
#pragma unroll
  for (int b = 0; b < B; ++b)
    r0[b] = rb::bf16_to_f32(
        a.res[(int64_t)min(b * 16 + em, a.M - 1) * a.N + n]);
  const float g = rb::bf16_to_f32(a.norm[n]);

  const rb::u32x4v from_x = rb::buffer(a.xs, (uint32_t)(a.M * a.K) * 2);
  const rb::u32x4v from_w = rb::buffer(
      reinterpret_cast<const uint16_t *>(a.ws) +
          (int64_t)(blockIdx.x >> 1) * a.K * 32, (uint32_t)a.K * 64);
  unsigned at_x[2 * B];                 // rows past M: zeros
#pragma unroll
  for (int i = 0; i < 2 * B; ++i) {
    const int row = i * 8 + (lane >> 3);
    at_x[i] = (unsigned)(row * a.K * 2 + ((lane & 7) ^ (row >> 1 & 7)) * 16);
  }
  const unsigned at_w = ((blockIdx.x & 1) * 16 + i16) * 16 + grp * 512;
  const unsigned mine = wid * (R::AHEAD * R::STAGE);
  auto fetch = [&](int c, int stage) {
    const unsigned to = mine + stage * R::STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      rb::lds_load_once(from_w, at_w, c * 4096 + i * 2048, to + i * 1024);
#pragma unroll
    for (int i = 0; i < 2 * B; ++i)
      rb::lds_load(from_x, at_x[i], c * 128, to + 2048 + i * 1024);
  };
  f32x4v acc[B];
#pragma unroll
  for (int b = 0; b < B; ++b) acc[b] = (f32x4v)(0.0f);
#pragma unroll
  for (int j = 0; j < R::AHEAD; ++j)
    if (c0 + j < c1) fetch(c0 + j, j);
  int stage = 0;
  for (int c = c0; c < c1; ++c) {
    if (c + R::AHEAD <= c1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R::AHEAD - 1) * R::LOADS)
                   : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char *b = smem + mine + stage * R::STAGE;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bf16x8v wv =
          *reinterpret_cast<const bf16x8v *>(b + s * 1024 + lane * 16);
#pragma unroll
      for (int k = 0; k < B; ++k)
        acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            wv,
            *reinterpret_cast<const bf16x8v *>(
                b + 2048 + (k * 16 + i16) * 128 +
                ((s * 4 + grp) ^ (i16 >> 1)) * 16),
            acc[k], 0, 0, 0);
    }
    // read before it is written again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (c + R::AHEAD < c1) fetch(c + R::AHEAD, stage);
    stage = stage + 1 == R::AHEAD ? 0 : stage + 1;
  }
  __syncthreads();
  float *red = reinterpret_cast<float *>(smem);     // [wave][block][16][17]
#pragma unroll
  for (int b = 0; b < B; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      red[((wid * B + b) * 16 + grp * 4 + r) * 17 + i16] = acc[b][r];
  __syncthreads();
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int m = b * 16 + em;
    if (m >= a.M) return;               // whole groups of 16 lanes
    float f = 0.0f;
#pragma unroll
    for (int v = 0; v < ROW_WAVES; ++v)
      f += red[((v * B + b) * 16 + en) * 17 + em];
    f += r0[b];
    const int64_t at = (int64_t)m * a.N + n;
    a.out[at] = rb::f32_to_bf16(f);
    a.y[at] = rb::f32_to_bf16(f * g);
    float ss = f * f;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    if (en == 0) a.squares[(int64_t)m * gridDim.x + blockIdx.x] = ss;
  }
}

// The same of a product's parts [P, M, N], a thread four columns of a row: nothing
// waits for a row's squares, so that a row is as many workgroups' as it has 1024
// columns. 4.8 us of 45 x 4096 in four parts, where the norm's kernel, which has a
// workgroup for a row, takes 4.9: both are begin and end of a launch.
template <int P>
__global__ __launch_bounds__(256) void parts_res_kernel(
    const float *__restrict__ parts, const uint16_t *__restrict__ res,
    const uint16_t *__restrict__ norm, uint16_t *__restrict__ out,
    uint16_t *__restrict__ y, float *__restrict__ squares, int M, int N) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 4, m = blockIdx.y;
  if (c >= N) return;                   // whole groups of 16 lanes
  const int64_t at = (int64_t)m * N + c;
  float4 p[P];
#pragma unroll
  for (int i = 0; i < P; ++i)
    p[i] = *reinterpret_cast<const float4 *>(parts + (int64_t)i * M * N + at);
  float f[4], g[4];
  const uint2 r = *reinterpret_cast<const uint2 *>(res + at);
  const uint2 w = *reinterpret_cast<const uint2 *>(norm + c);
  f[0] = rb::bf16_to_f32((uint16_t)r.x);
  f[1] = rb::bf16_to_f32((uint16_t)(r.x >> 16));
  f[2] = rb::bf16_to_f32((uint16_t)r.y);
  f[3] = rb::bf16_to_f32((uint16_t)(r.y >> 16));
  g[0] = rb::bf16_to_f32((uint16_t)w.x);
  g[1] = rb::bf16_to_f32((uint16_t)(w.x >> 16));
  g[2] = rb::bf16_to_f32((uint16_t)w.y);
  g[3] = rb::bf16_to_f32((uint16_t)(w.y >> 16));
  float4 s = p[0];
#pragma unroll
  for (int i = 1; i < P; ++i) {
    s.x += p[i].x; s.y += p[i].y; s.z += p[i].z; s.w += p[i].w;
  }
  f[0] += s.x; f[1] += s.y; f[2] += s.z; f[3] += s.w;
  ends::put<4>(out + at, f);
  float ss = (f[0] * f[0] + f[1] * f[1]) + (f[2] * f[2] + f[3] * f[3]);
#pragma unroll
  for (int e = 0; e < 4; ++e) f[e] *= g[e];
  ends::put<4>(y + at, f);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if ((threadIdx.x & 15) == 0) squares[(int64_t)m * (N / 64) + c / 64] = ss;
}

}  // namespace

// Sizes that decode_res serves: its parts of the squares are one per 16 columns,
// 256 at most.
bool decode_res_supported(int64_t M, int64_t N, int64_t K, bool fp8) {
  return M >= 1 && M <= 32 && N > 0 && N % 64 == 0 && N <= 4096 && K > 0 &&
         K % (fp8 ? 64 : 32) == 0 && K < (1 << 24);
}

// {r', y, squares [M, N / 16]}, y as an operand or in rows; xs and ws (with its
// scale) as decode_gemm and decode_gemm_fp8 take them.
std::vector<at::Tensor> decode_res(at::Tensor xs, at::Tensor ws,
                                   c10::optional<at::Tensor> scale,
                                   at::Tensor res, at::Tensor norm,
                                   bool rows) {
  TORCH_CHECK(res.is_cuda() && res.dim() == 2 && res.is_contiguous() &&
              norm.is_contiguous() && norm.device() == res.device() &&
              res.scalar_type() == at::kBFloat16 &&
              norm.scalar_type() == at::kBFloat16 &&
              norm.numel() == res.size(1), "decode_res: residual, norm");
  const bool fp8 = ws.scalar_type() == at::kByte;
  const int64_t M = res.size(0), N = res.size(1);
  const int64_t K = N > 0 ? ws.numel() / N : 0;
  TORCH_CHECK(decode_res_supported(M, N, K, fp8), "decode_res: shape ", M, "x",
              N, "x", K);
  TORCH_CHECK(xs.device() == res.device() && ws.device() == res.device() &&
              xs.is_contiguous() && ws.is_contiguous() &&
              xs.scalar_type() == at::kBFloat16 &&
              (fp8 || ws.scalar_type() == at::kBFloat16) &&
              xs.numel() == (K / 16) * 512 && ws.numel() == N * K,
              "decode_res: operands");
  TORCH_CHECK(fp8 == scale.has_value() &&
              (!fp8 || (scale->device() == res.device() &&
                        scale->is_contiguous() && scale->numel() == N &&
                        scale->scalar_type() == at::kFloat)),
              "decode_res: scales");
  auto out = at::empty_like(res);
  auto y = rows ? at::empty_like(res)
                : at::empty({N / 16 * 512}, res.options());
  auto squares = at::empty({M, N / 16}, res.options().dtype(at::kFloat));
  Sum a{(const uint16_t *)xs.data_ptr(), (const uint8_t *)ws.data_ptr(),
        fp8 ? scale->data_ptr<float>() : nullptr,
        (const uint16_t *)res.data_ptr(), (const uint16_t *)norm.data_ptr(),
        (uint16_t *)out.data_ptr(), (uint16_t *)y.data_ptr(), rows,
        squares.data_ptr<float>(), (int)M, (int)N, (int)K};
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(N / 16)), dim3(BLOCK), 0,
                       at::cuda::getCurrentHIPStream(), a);
  };
  // Loads past the end of a wave's sums are made for nothing: of e4m3, whose waves have
  // few steps, by six or by eight, as fewer are loaded (us by six and by eight, of one
  // row and 2048, 4096, 5632, 11008 and 14336 columns, 4, 8, 11, 22 and 28 steps: 2048
  // rows 3.9 4.2, -, 6.0 6.8, 4096 rows -, 6.2 5.6, -, 12.3 12.4, 13.1 13.9).
  const int64_t steps = (K / 64 + WAVES - 1) / WAVES;
  if (M > 16)
    fp8 ? go(decode_res_kernel<true, 2, 4>) : go(decode_res_kernel<false, 2, 4>);
  else if (!fp8)
    go(decode_res_kernel<false, 1, 8>);
  else if ((steps + 7) / 8 * 8 <= (steps + 5) / 6 * 6)
    go(decode_res_kernel<true, 1, 8>);
  else
    go(decode_res_kernel<true, 1, 6>);
  return {out, y, squares};
}

// Whether rows_res takes rows [M, K] of W [N, K] in the decode layout: its parts of
// the squares are one per 16 columns, 256 at most.
bool rows_res_supported(int64_t M, int64_t N, int64_t K) {
  return M >= 33 && M <= 64 && N > 0 && N % 32 == 0 && N <= 4096 &&
         K % 64 == 0 && K >= 1024 && K < (1 << 22);
}

// {r', y, squares [M, N / 16]}, x and y in rows; ws as decode_gemm takes it.
std::vector<at::Tensor> rows_res(at::Tensor x, at::Tensor ws, at::Tensor res,
                                 at::Tensor norm) {
  TORCH_CHECK(res.is_cuda() && res.dim() == 2 && res.is_contiguous() &&
              norm.is_contiguous() && norm.device() == res.device() &&
              res.scalar_type() == at::kBFloat16 &&
              norm.scalar_type() == at::kBFloat16 &&
              norm.numel() == res.size(1), "rows_res: residual, norm");
  TORCH_CHECK(x.dim() == 2 && x.size(0) == res.size(0) && x.is_contiguous() &&
              ws.is_contiguous() && x.device() == res.device() &&
              ws.device() == res.device() &&
              x.scalar_type() == at::kBFloat16 &&
              ws.scalar_type() == at::kBFloat16 &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(ws.data_ptr()) % 16 == 0,
              "rows_res: operands");
  const int64_t M = res.size(0), N = res.size(1), K = x.size(1);
  TORCH_CHECK(rows_res_supported(M, N, K) && ws.numel() == N * K,
              "rows_res: shape ", M, "x", N, "x", K);
  auto out = at::empty_like(res);
  auto y = at::empty_like(res);
  auto squares = at::empty({M, N / 16}, res.options().dtype(at::kFloat));
  const Sum a{(const uint16_t *)x.data_ptr(), (const uint8_t *)ws.data_ptr(),
              nullptr, (const uint16_t *)res.data_ptr(),
              (const uint16_t *)norm.data_ptr(), (uint16_t *)out.data_ptr(),
              (uint16_t *)y.data_ptr(), true, squares.data_ptr<float>(), (int)M,
              (int)N, (int)K};
  auto go = [&](auto blocks) {
    constexpr int B = decltype(blocks)::value;
    auto kernel = rows_res_kernel<B>;
    static const bool once =
        hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            Ring<B>::LDS) == hipSuccess;
    TORCH_CHECK(once, "rows_res: LDS size");
    hipLaunchKernelGGL(kernel, dim3((unsigned)(N / 16)), dim3(ROW_WAVES * 64),
                       Ring<B>::LDS, at::cuda::getCurrentHIPStream(), a);
  };
  if (M <= 48) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 4>{});
  return {out, y, squares};
}

// Widths of parts_res: its parts of the squares are one per 64 columns, four at a
// time and 256 at most.
bool parts_res_supported(int64_t N) {
  return N > 0 && N % 256 == 0 && N <= 16384;
}

// {r', y, squares [M, N / 64]} of parts [P, M, N] of what is added, P 2, 4 or 8.
std::vector<at::Tensor> parts_res(at::Tensor parts, at::Tensor res,
                                  at::Tensor norm) {
  TORCH_CHECK(res.is_cuda() && res.dim() == 2 && res.is_contiguous() &&
              norm.is_contiguous() && norm.device() == res.device() &&
              res.scalar_type() == at::kBFloat16 &&
              norm.scalar_type() == at::kBFloat16 &&
              norm.numel() == res.size(1) &&
              reinterpret_cast<uintptr_t>(res.data_ptr()) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(norm.data_ptr()) % 8 == 0,
              "parts_res: residual, norm");
  const int64_t M = res.size(0), N = res.size(1);
  TORCH_CHECK(parts.device() == res.device() && parts.dim() == 3 &&
              parts.is_contiguous() && parts.scalar_type() == at::kFloat &&
              parts.size(1) == M && parts.size(2) == N &&
              reinterpret_cast<uintptr_t>(parts.data_ptr()) % 16 == 0 &&
              M >= 1 && M <= 65535 && parts_res_supported(N),
              "parts_res: parts [P, M, 256 n]");
  auto out = at::empty_like(res);
  auto y = at::empty_like(res);
  auto squares = at::empty({M, N / 64}, parts.options());
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((N + 1023) / 1024), (unsigned)M),
                       dim3(256), 0, at::cuda::getCurrentHIPStream(),
                       parts.data_ptr<float>(),
                       (const uint16_t *)res.data_ptr(),
                       (const uint16_t *)norm.data_ptr(),
                       (uint16_t *)out.data_ptr(), (uint16_t *)y.data_ptr(),
                       squares.data_ptr<float>(), (int)M, (int)N);
  };
  switch (parts.size(0)) {
    case 2: go(parts_res_kernel<2>); break;
    case 4: go(parts_res_kernel<4>); break;
    case 8: go(parts_res_kernel<8>); break;
    default: TORCH_CHECK(false, "parts_res: 2, 4 or 8 parts");
  }
  return {out, y, squares};
}
