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
// waves take parts of the sums, a kilobyte of W an instruction; B blocks of 16
// rows of x (16x16x32 products: A[i=l&15][k=(l>>4)*8+e], B[k][j=l&15],
// C[j=l&15][i=(l>>4)*4+r]). A lane's 16 bytes of e4m3 are of two products.
//
// Bound by the weight stream, by x with many long rows. us in a graph, weights
// out of cache, in parts that the norm's kernel adds up, and here, of 1, 16 and
// 32 rows:
//   4096 x 4096        12.0  8.1   13.2  8.4   13.8 10.1
//   4096 x 11008       21.0 19.1   22.0 20.5   23.8 24.0
//   3072 x 24576       34.9 31.5   34.2 33.7   39.7 45.7
//   4096 x 4096  e4m3  10.1  6.3   11.2  7.5   12.4  8.6
//   4096 x 11008 e4m3  16.0 12.3   16.4 13.0   18.4 17.8
template <bool FP8, int B>
__global__ __launch_bounds__(BLOCK, 1) void decode_res_kernel(Sum a) {
  constexpr int X = FP8 ? 2 : 1, U = B == 1 ? (FP8 ? 6 : 8) : 4;
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
  if (M <= 16) fp8 ? go(decode_res_kernel<true, 1>) : go(decode_res_kernel<false, 1>);
  else fp8 ? go(decode_res_kernel<true, 2>) : go(decode_res_kernel<false, 2>);
  return {out, y, squares};
}
