// Fused RMSNorm forward/backward for CDNA4 (gfx950).
//
// Replaces the eager 4-kernel torch sequence (pow/mean/rsqrt/mul) with one
// HBM-bound pass per direction. Reference semantics match the plain
// PyTorch fp32 RMSNorm used by the test-suite reference models
// (llama-family norm; the reference platform delegates this to external
// HuggingFace trainer images).
//
// Layout: x [N, D] row-major. One workgroup (256 threads) per row,
// grid-strided. All math in fp32; bf16 IO vectorized 8-wide (16 B/lane).

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

constexpr int BLOCK = 256;

// swz (optional, bf16 only): ALSO write the normed row into the decode
// GEMM's B-fragment lane order ([D/16][2][32][8], csrc/decode_gemm.hip)
// so the decode path needs no separate x-swizzle launch. Each thread's
// 8-element vector IS one swizzled 16 B slot: pos = (k/16)*512 +
// ((k/8)&1)*256 + row*8.
// res/sum_out (optional, together): normalize x + res instead of x and
// also write the sum — fuses the decode loop's residual add into the
// norm (one launch instead of two; the sum feeds the NEXT residual).
// res32/rsplit (optional, bf16 path): the residual arrives as the
// UNCOMBINED fp32 split-K slab [rsplit, n_rows, D] straight from
// decode_gemm_raw — folding the slices here saves the combine launch.
// One workgroup per row, any width (rows beyond the next kernel's).
template <typename T>
__global__ void rmsnorm_fwd_kernel(const T *__restrict__ x,
                                   const T *__restrict__ res,
                                   const float *__restrict__ res32,
                                   int rsplit,
                                   T *__restrict__ sum_out,
                                   const T *__restrict__ w,
                                   T *__restrict__ y,
                                   float *__restrict__ inv_rms,
                                   uint16_t *__restrict__ swz,
                                   int64_t n_rows, int D, float eps) {
  constexpr int W = rb::VIO<T>::W;
  __shared__ float red[BLOCK / RB_WAVE];
  const int nvec = D / W;

  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    const T *xr = x + row * D;
    T *yr = y + row * D;

    float ss = 0.0f;
    for (int i = threadIdx.x; i < nvec; i += BLOCK) {
      float f[W];
      rb::VIO<T>::load(xr + i * W, f);
      if (res != nullptr || res32 != nullptr) {
        if (res != nullptr) {
          float r[W];
          rb::VIO<T>::load(res + row * D + i * W, r);
#pragma unroll
          for (int k = 0; k < W; ++k) f[k] += r[k];
        } else {
          for (int sl = 0; sl < rsplit; ++sl) {
            const float *rp = res32 + ((int64_t)sl * n_rows + row) * D + i * W;
#pragma unroll
            for (int k = 0; k < W; k += 4) {
              float4 a = *reinterpret_cast<const float4 *>(rp + k);
              f[k] += a.x; f[k + 1] += a.y; f[k + 2] += a.z; f[k + 3] += a.w;
            }
          }
        }
        if (sum_out != nullptr)
          rb::VIO<T>::store(sum_out + row * D + i * W, f);
      }
#pragma unroll
      for (int k = 0; k < W; ++k) ss += f[k] * f[k];
    }
    ss = rb::block_reduce_sum(ss, red);
    const float ir = rsqrtf(ss / (float)D + eps);
    if (threadIdx.x == 0 && inv_rms != nullptr) inv_rms[row] = ir;

    for (int i = threadIdx.x; i < nvec; i += BLOCK) {
      float f[W], g[W];
      rb::VIO<T>::load(xr + i * W, f);     // L1-resident second read
      if (res != nullptr) {
        float r[W];
        rb::VIO<T>::load(res + row * D + i * W, r);
#pragma unroll
        for (int k = 0; k < W; ++k) f[k] += r[k];
      } else if (res32 != nullptr) {
        for (int sl = 0; sl < rsplit; ++sl) {
          const float *rp = res32 + ((int64_t)sl * n_rows + row) * D + i * W;
#pragma unroll
          for (int k = 0; k < W; k += 4) {
            float4 a = *reinterpret_cast<const float4 *>(rp + k);
            f[k] += a.x; f[k + 1] += a.y; f[k + 2] += a.z; f[k + 3] += a.w;
          }
        }
      }
      rb::VIO<T>::load(w + i * W, g);
#pragma unroll
      for (int k = 0; k < W; ++k) f[k] = f[k] * ir * g[k];
      rb::VIO<T>::store(yr + i * W, f);
      if constexpr (sizeof(T) == 2) {
        if (swz != nullptr) {
          const int k0 = i * 8;
          rb::VIO<T>::store(reinterpret_cast<T *>(swz) +
                            (k0 >> 4) * 512 + ((k0 >> 3) & 1) * 256 +
                            row * 8, f);
        }
      }
    }
    __syncthreads();
  }
}

// The same for rows of up to NV * BLOCK vectors: a thread's NV vectors stay in
// registers between the two passes, so x, the residual and its slices are read
// once. Vectors past the row's end read its last one again (a branch around a
// load would make the compiler wait for each) and count nothing.
template <typename T, int NV>
__global__ __launch_bounds__(BLOCK) void rmsnorm_fwd_reg_kernel(
    const T *__restrict__ x, const T *__restrict__ res,
    const float *__restrict__ res32, int rsplit, T *__restrict__ sum_out,
    const T *__restrict__ w, T *__restrict__ y, float *__restrict__ inv_rms,
    uint16_t *__restrict__ swz, int64_t n_rows, int D, float eps) {
  constexpr int W = rb::VIO<T>::W;
  __shared__ float red[BLOCK / RB_WAVE];
  const int nvec = D / W;
  int at[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v)
    at[v] = min(v * BLOCK + (int)threadIdx.x, nvec - 1) * W;

  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    float f[NV][W], g[NV][W];
#pragma unroll
    for (int v = 0; v < NV; ++v) rb::VIO<T>::load(x + row * D + at[v], f[v]);
    if (res != nullptr) {
#pragma unroll
      for (int v = 0; v < NV; ++v)
        rb::VIO<T>::load(res + row * D + at[v], g[v]);
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int k = 0; k < W; ++k) f[v][k] += g[v][k];
    } else if (res32 != nullptr) {
      for (int sl = 0; sl < rsplit; ++sl) {
        const float *rp = res32 + ((int64_t)sl * n_rows + row) * D;
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
          for (int k = 0; k < W; k += 4)
            rb::VIO<float>::load(rp + at[v] + k, g[v] + k);
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
          for (int k = 0; k < W; ++k) f[v][k] += g[v][k];
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) rb::VIO<T>::load(w + at[v], g[v]);
    float ss = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v * BLOCK + (int)threadIdx.x >= nvec) continue;
      if (sum_out != nullptr)
        rb::VIO<T>::store(sum_out + row * D + at[v], f[v]);
#pragma unroll
      for (int k = 0; k < W; ++k) ss += f[v][k] * f[v][k];
    }
    ss = rb::block_reduce_sum(ss, red);
    const float ir = rsqrtf(ss / (float)D + eps);
    if (threadIdx.x == 0 && inv_rms != nullptr) inv_rms[row] = ir;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v * BLOCK + (int)threadIdx.x >= nvec) continue;
#pragma unroll
      for (int k = 0; k < W; ++k) f[v][k] = f[v][k] * ir * g[v][k];
      rb::VIO<T>::store(y + row * D + at[v], f[v]);
      if constexpr (sizeof(T) == 2) {
        if (swz != nullptr)
          rb::VIO<T>::store(reinterpret_cast<T *>(swz) + (at[v] >> 4) * 512 +
                            ((at[v] >> 3) & 1) * 256 + row * 8, f[v]);
      }
    }
  }
}

template <typename T>
void launch_fwd(const T *x, const T *res, const float *res32, int rsplit,
                T *sum_out, const T *w, T *y, float *inv_rms, uint16_t *swz,
                int64_t n_rows, int D, float eps) {
  if (n_rows == 0) return;
  const int nv = (D / rb::VIO<T>::W + BLOCK - 1) / BLOCK;
  auto stream = at::hip::getCurrentHIPStream();
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(std::min<int64_t>(n_rows, 2048)),
                       dim3(BLOCK), 0, stream, x, res, res32, rsplit, sum_out,
                       w, y, inv_rms, swz, n_rows, D, eps);
  };
  if (nv <= 1) go(rmsnorm_fwd_reg_kernel<T, 1>);
  else if (nv == 2) go(rmsnorm_fwd_reg_kernel<T, 2>);
  else if (nv <= 4) go(rmsnorm_fwd_reg_kernel<T, 4>);
  else go(rmsnorm_fwd_kernel<T>);
}

// Backward: dx in one pass, rows of up to NV * BLOCK vectors in registers. With
// `add`, dx also takes the gradient that reaches the normed sum by other ways.
// DW: each thread's column set is FIXED across its rows, so its dw partials
// live in registers until the workgroup's row of `dw` [workgroups, D] is
// written, which rmsnorm_dw_kernel sums. Atomics of a row or a few per
// workgroup instead are what such a kernel then takes. us on [2048, 4096]: 66
// with them, 11 without dw, 14 with `add`, 25 with dw.
template <typename T, int NV, bool DW>
__global__ __launch_bounds__(BLOCK) void rmsnorm_bwd_reg_kernel(
    const T *__restrict__ x, const T *__restrict__ w,
    const T *__restrict__ dy, const float *__restrict__ inv_rms,
    const T *__restrict__ add, T *__restrict__ dx, float *__restrict__ dw,
    int64_t n_rows, int D) {
  constexpr int W = rb::VIO<T>::W;
  __shared__ float red[BLOCK / RB_WAVE];
  const int nvec = D / W;
  int at[NV];
  float wf[NV][W], acc[DW ? NV : 1][W];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    at[v] = min(v * BLOCK + (int)threadIdx.x, nvec - 1) * W;
    rb::VIO<T>::load(w + at[v], wf[v]);
    if constexpr (DW) {
#pragma unroll
      for (int k = 0; k < W; ++k) acc[v][k] = 0.0f;
    }
  }
  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    float xf[NV][W], df[NV][W], af[NV][W];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      rb::VIO<T>::load(x + row * D + at[v], xf[v]);
      rb::VIO<T>::load(dy + row * D + at[v], df[v]);
    }
    if (add != nullptr) {
#pragma unroll
      for (int v = 0; v < NV; ++v)
        rb::VIO<T>::load(add + row * D + at[v], af[v]);
    } else {
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int k = 0; k < W; ++k) af[v][k] = 0.0f;
    }
    const float ir = inv_rms[row];
    float s = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v * BLOCK + (int)threadIdx.x >= nvec) continue;
#pragma unroll
      for (int k = 0; k < W; ++k) s += df[v][k] * wf[v][k] * xf[v][k];
    }
    s = rb::block_reduce_sum(s, red);
    const float c = ir * ir * ir * s / (float)D;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v * BLOCK + (int)threadIdx.x >= nvec) continue;
      float o[W];
#pragma unroll
      for (int k = 0; k < W; ++k) {
        o[k] = af[v][k] + ir * wf[v][k] * df[v][k] - c * xf[v][k];
        if constexpr (DW) acc[v][k] += df[v][k] * xf[v][k] * ir;
      }
      rb::VIO<T>::store(dx + row * D + at[v], o);
    }
  }
  if constexpr (DW) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v * BLOCK + (int)threadIdx.x >= nvec) continue;
#pragma unroll
      for (int k = 0; k < W; k += 4)
        rb::VIO<float>::store(dw + (int64_t)blockIdx.x * D + at[v] + k,
                              acc[v] + k);
    }
  }
}

// Column sums of part [n, D]: 64 columns a workgroup, 16 rows at a time.
__global__ __launch_bounds__(BLOCK) void rmsnorm_dw_kernel(
    const float *__restrict__ part, float *__restrict__ dw, int n, int D) {
  __shared__ float4 red[BLOCK];
  const int c = blockIdx.x * 64 + (threadIdx.x & 15) * 4;
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  if (c < D)
    for (int r = threadIdx.x >> 4; r < n; r += 16) {
      const float4 x = *reinterpret_cast<const float4 *>(
          part + (int64_t)r * D + c);
      sum.x += x.x; sum.y += x.y; sum.z += x.z; sum.w += x.w;
    }
  red[threadIdx.x] = sum;
  __syncthreads();
  if (threadIdx.x >= 16 || c >= D) return;
  for (int r = 1; r < 16; ++r) {
    const float4 x = red[r * 16 + threadIdx.x];
    sum.x += x.x; sum.y += x.y; sum.z += x.z; sum.w += x.w;
  }
  *reinterpret_cast<float4 *>(dw + c) = sum;
}

// Wider rows: dw in LDS.
template <typename T>
__global__ void rmsnorm_bwd_kernel(const T *__restrict__ x,
                                           const T *__restrict__ w,
                                           const T *__restrict__ dy,
                                           const float *__restrict__ inv_rms,
                                           const T *__restrict__ add,
                                           T *__restrict__ dx,
                                           float *__restrict__ dw,
                                           int64_t n_rows, int D) {
  constexpr int W = rb::VIO<T>::W;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float *dw_loc = reinterpret_cast<float *>(smem);          // D floats
  float *red = dw_loc + D;                                  // BLOCK/64 floats
  const int nvec = D / W;

  for (int i = threadIdx.x; i < D; i += BLOCK) dw_loc[i] = 0.0f;
  __syncthreads();

  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    const T *xr = x + row * D;
    const T *dyr = dy + row * D;
    T *dxr = dx + row * D;
    const float ir = inv_rms[row];

    float s = 0.0f;
    for (int i = threadIdx.x; i < nvec; i += BLOCK) {
      float xf[W], wf[W], df[W];
      rb::VIO<T>::load(xr + i * W, xf);
      rb::VIO<T>::load(w + i * W, wf);
      rb::VIO<T>::load(dyr + i * W, df);
#pragma unroll
      for (int k = 0; k < W; ++k) s += df[k] * wf[k] * xf[k];
    }
    s = rb::block_reduce_sum(s, red);
    const float c = ir * ir * ir * s / (float)D;

    for (int i = threadIdx.x; i < nvec; i += BLOCK) {
      float xf[W], wf[W], df[W], o[W];
      rb::VIO<T>::load(xr + i * W, xf);
      rb::VIO<T>::load(w + i * W, wf);
      rb::VIO<T>::load(dyr + i * W, df);
#pragma unroll
      for (int k = 0; k < W; ++k) {
        o[k] = ir * wf[k] * df[k] - c * xf[k];
        dw_loc[i * W + k] += df[k] * xf[k] * ir;
      }
      if (add != nullptr) {
        rb::VIO<T>::load(add + row * D + i * W, xf);
#pragma unroll
        for (int k = 0; k < W; ++k) o[k] += xf[k];
      }
      rb::VIO<T>::store(dxr + i * W, o);
    }
    __syncthreads();
  }

  __syncthreads();
  for (int i = threadIdx.x; i < D; i += BLOCK)
    if (dw_loc[i] != 0.0f) atomicAdd(dw + i, dw_loc[i]);
}

}  // namespace

std::vector<at::Tensor> rmsnorm_fwd(at::Tensor x, at::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda(), "rmsnorm: tensors must be on GPU");
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous(), "rmsnorm: contiguous only");
  const int D = (int)x.size(-1);
  const int64_t n_rows = x.numel() / D;
  auto y = at::empty_like(x);
  auto inv_rms = at::empty({n_rows}, x.options().dtype(at::kFloat));

  if (x.scalar_type() == at::kBFloat16) {
    TORCH_CHECK(D % 8 == 0, "rmsnorm bf16: D must be a multiple of 8");
    launch_fwd<uint16_t>((const uint16_t *)x.data_ptr(),
                       (const uint16_t *)nullptr, (const float *)nullptr, 0,
                       (uint16_t *)nullptr,
                       (const uint16_t *)w.data_ptr(),
                       (uint16_t *)y.data_ptr(), inv_rms.data_ptr<float>(),
                       (uint16_t *)nullptr, n_rows, D, (float)eps);
  } else if (x.scalar_type() == at::kFloat) {
    TORCH_CHECK(D % 4 == 0, "rmsnorm f32: D must be a multiple of 4");
    launch_fwd<float>(x.data_ptr<float>(), (const float *)nullptr,
                       (const float *)nullptr, 0,
                       (float *)nullptr, w.data_ptr<float>(),
                       y.data_ptr<float>(),
                       inv_rms.data_ptr<float>(), (uint16_t *)nullptr,
                       n_rows, D, (float)eps);
  } else {
    TORCH_CHECK(false, "rmsnorm: unsupported dtype");
  }
  return {y, inv_rms};
}

// Decode-path variant: returns {y, y_swz} where y_swz is the decode
// GEMM's pre-swizzled B-operand ([D/16]x512 bf16, rows m >= n_rows left
// uninitialized: decode_gemm drops their outputs at the epilogue).
std::vector<at::Tensor> rmsnorm_fwd_dec(at::Tensor x, at::Tensor w,
                                        double eps) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && w.is_contiguous(),
              "rmsnorm_fwd_dec: contiguous GPU tensors");
  TORCH_CHECK(x.scalar_type() == at::kBFloat16, "rmsnorm_fwd_dec: bf16");
  const int64_t n_rows = x.numel() / x.size(-1);
  const int D = (int)x.size(-1);
  TORCH_CHECK(n_rows <= 32 && D % 16 == 0, "rmsnorm_fwd_dec: shape");
  auto y = at::empty_like(x);
  auto swz = at::empty({(int64_t)(D / 16) * 512}, x.options());
  launch_fwd<uint16_t>((const uint16_t *)x.data_ptr(),
                     (const uint16_t *)nullptr, (const float *)nullptr, 0,
                     (uint16_t *)nullptr,
                     (const uint16_t *)w.data_ptr(),
                     (uint16_t *)y.data_ptr(), (float *)nullptr,
                     (uint16_t *)swz.data_ptr(), n_rows, D, (float)eps);
  return {y, swz};
}

// Fused residual + norm + swizzle for the decode loop: returns
// {sum = x + res, y = rmsnorm(sum) * w, y_swz}. One launch replaces the
// eager residual add + the norm + the operand swizzle.
std::vector<at::Tensor> rmsnorm_res_fwd_dec(at::Tensor x, at::Tensor res,
                                            at::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && res.is_contiguous() &&
              w.is_contiguous(), "rmsnorm_res_fwd_dec: contiguous");
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 &&
              res.scalar_type() == at::kBFloat16, "rmsnorm_res_fwd_dec: bf16");
  TORCH_CHECK(x.sizes() == res.sizes(), "rmsnorm_res_fwd_dec: shape");
  const int64_t n_rows = x.numel() / x.size(-1);
  const int D = (int)x.size(-1);
  TORCH_CHECK(n_rows <= 32 && D % 16 == 0, "rmsnorm_res_fwd_dec: shape");
  auto sum = at::empty_like(x);
  auto y = at::empty_like(x);
  auto swz = at::empty({(int64_t)(D / 16) * 512}, x.options());
  launch_fwd<uint16_t>((const uint16_t *)x.data_ptr(),
                     (const uint16_t *)res.data_ptr(),
                     (const float *)nullptr, 0,
                     (uint16_t *)sum.data_ptr(),
                     (const uint16_t *)w.data_ptr(),
                     (uint16_t *)y.data_ptr(), (float *)nullptr,
                     (uint16_t *)swz.data_ptr(), n_rows, D, (float)eps);
  return {sum, y, swz};
}

// Residual + norm of any number of rows: {sum = x + res, y, inv_rms}.
std::vector<at::Tensor> rmsnorm_res_fwd(at::Tensor x, at::Tensor res,
                                        at::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && res.is_contiguous() &&
              w.is_contiguous() && x.sizes() == res.sizes() && x.dim() >= 1 &&
              w.numel() == x.size(-1), "rmsnorm_res_fwd: shapes");
  const int D = (int)x.size(-1);
  const int64_t n_rows = D ? x.numel() / D : 0;
  const bool bf16 = x.scalar_type() == at::kBFloat16;
  TORCH_CHECK((bf16 || x.scalar_type() == at::kFloat) &&
              res.scalar_type() == x.scalar_type() &&
              w.scalar_type() == x.scalar_type() && D % (bf16 ? 8 : 4) == 0,
              "rmsnorm_res_fwd: bf16 or f32, whole vectors");
  auto sum = at::empty_like(x), y = at::empty_like(x);
  auto inv_rms = at::empty({n_rows}, x.options().dtype(at::kFloat));
  if (bf16)
    launch_fwd<uint16_t>((const uint16_t *)x.data_ptr(),
                         (const uint16_t *)res.data_ptr(), nullptr, 0,
                         (uint16_t *)sum.data_ptr(),
                         (const uint16_t *)w.data_ptr(),
                         (uint16_t *)y.data_ptr(), inv_rms.data_ptr<float>(),
                         nullptr, n_rows, D, (float)eps);
  else
    launch_fwd<float>(x.data_ptr<float>(), res.data_ptr<float>(), nullptr, 0,
                      sum.data_ptr<float>(), w.data_ptr<float>(),
                      y.data_ptr<float>(), inv_rms.data_ptr<float>(), nullptr,
                      n_rows, D, (float)eps);
  return {sum, y, inv_rms};
}

// Same, with the residual as an UNCOMBINED fp32 split-K slab
// [split, n_rows, D] from decode_gemm_raw.
std::vector<at::Tensor> rmsnorm_res_slab_fwd_dec(at::Tensor x,
                                                 at::Tensor slabs,
                                                 at::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && slabs.is_contiguous() &&
              w.is_contiguous(), "rmsnorm_res_slab_fwd_dec: contiguous");
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 &&
              slabs.scalar_type() == at::kFloat &&
              slabs.dim() == 3, "rmsnorm_res_slab_fwd_dec: dtypes");
  const int64_t n_rows = x.numel() / x.size(-1);
  const int D = (int)x.size(-1);
  TORCH_CHECK(slabs.size(1) == n_rows && slabs.size(2) == D &&
              n_rows <= 32 && D % 16 == 0, "rmsnorm_res_slab_fwd_dec: shape");
  auto sum = at::empty_like(x);
  auto y = at::empty_like(x);
  auto swz = at::empty({(int64_t)(D / 16) * 512}, x.options());
  launch_fwd<uint16_t>((const uint16_t *)x.data_ptr(),
                     (const uint16_t *)nullptr,
                     (const float *)slabs.data_ptr(), (int)slabs.size(0),
                     (uint16_t *)sum.data_ptr(),
                     (const uint16_t *)w.data_ptr(),
                     (uint16_t *)y.data_ptr(), (float *)nullptr,
                     (uint16_t *)swz.data_ptr(), n_rows, D, (float)eps);
  return {sum, y, swz};
}

// The same of any number of rows, without the operand: {sum, y}.
std::vector<at::Tensor> rmsnorm_res_slab_fwd(at::Tensor x, at::Tensor slabs,
                                             at::Tensor w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() &&
              slabs.is_contiguous() && w.is_contiguous() &&
              x.scalar_type() == at::kBFloat16 &&
              w.scalar_type() == at::kBFloat16 &&
              slabs.scalar_type() == at::kFloat && slabs.dim() == 3 &&
              slabs.size(1) == x.size(0) && slabs.size(2) == x.size(1) &&
              w.numel() == x.size(1) && x.size(1) % 8 == 0,
              "rmsnorm_res_slab_fwd: x [T, 8 n] bf16, slabs [P, T, 8 n]");
  auto sum = at::empty_like(x), y = at::empty_like(x);
  launch_fwd<uint16_t>((const uint16_t *)x.data_ptr(), nullptr,
                       slabs.data_ptr<float>(), (int)slabs.size(0),
                       (uint16_t *)sum.data_ptr(),
                       (const uint16_t *)w.data_ptr(),
                       (uint16_t *)y.data_ptr(), nullptr, nullptr, x.size(0),
                       (int)x.size(1), (float)eps);
  return {sum, y};
}

// Norm of a 32-bit residual: x += delta in place, y = rmsnorm(x) * (offset + w)
// in w's dtype. `nd` delta terms of type DT (0: none; > 1: the uncombined split-K
// slab of decode_gemm_raw) lie n_rows * D apart. swz as above (bf16 only).
namespace {
template <typename T, typename DT, int V>
__global__ void rmsnorm_res32_kernel(float *__restrict__ x,
                                     const DT *__restrict__ delta, int nd,
                                     const T *__restrict__ w,
                                     T *__restrict__ y,
                                     uint16_t *__restrict__ swz,
                                     int64_t n_rows, int D, float eps,
                                     float offset) {
  __shared__ float red[BLOCK / RB_WAVE];
  const int nvec = D / V;
  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    float *xr = x + row * D;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < nvec; i += BLOCK) {
      float f[V];
      if constexpr (V == 8) {
        rb::VIO<float>::load(xr + i * 8, f);
        rb::VIO<float>::load(xr + i * 8 + 4, f + 4);
      } else {
        f[0] = xr[i];
      }
      for (int s = 0; s < nd; ++s) {
        const DT *dp = delta + ((int64_t)s * n_rows + row) * D + i * V;
        float d[V];
        if constexpr (V == 8) {
          rb::VIO<DT>::load(dp, d);
          if constexpr (rb::VIO<DT>::W == 4) rb::VIO<DT>::load(dp + 4, d + 4);
        } else {
          d[0] = rb::bf16_to_f32_or_id(*dp);
        }
#pragma unroll
        for (int k = 0; k < V; ++k) f[k] += d[k];
      }
      if (nd > 0) {
        if constexpr (V == 8) {
          rb::VIO<float>::store(xr + i * 8, f);
          rb::VIO<float>::store(xr + i * 8 + 4, f + 4);
        } else {
          xr[i] = f[0];
        }
      }
#pragma unroll
      for (int k = 0; k < V; ++k) ss += f[k] * f[k];
    }
    ss = rb::block_reduce_sum(ss, red);
    const float ir = 1.0f / sqrtf(ss / (float)D + eps);
    for (int i = threadIdx.x; i < nvec; i += BLOCK) {
      if constexpr (V == 8) {
        float f[8], g[8];               // this thread's own values of pass 1
        rb::VIO<float>::load(xr + i * 8, f);
        rb::VIO<float>::load(xr + i * 8 + 4, f + 4);
        rb::VIO<T>::load(w + i * 8, g);
        if constexpr (rb::VIO<T>::W == 4) rb::VIO<T>::load(w + i * 8 + 4, g + 4);
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = f[k] * ir * (offset + g[k]);
        rb::VIO<T>::store(y + row * D + i * 8, f);
        if constexpr (rb::VIO<T>::W == 4)
          rb::VIO<T>::store(y + row * D + i * 8 + 4, f + 4);
        if constexpr (sizeof(T) == 2) {
          if (swz != nullptr)
            rb::VIO<T>::store(swz + (i >> 1) * 512 + (i & 1) * 256 + row * 8,
                              f);
        }
      } else {
        rb::store_scalar(y + row * D + i,
                         xr[i] * ir * (offset + rb::bf16_to_f32_or_id(w[i])));
      }
    }
    __syncthreads();
  }
}
}  // namespace

std::vector<at::Tensor> rmsnorm_res32(at::Tensor x,
                                      c10::optional<at::Tensor> delta,
                                      at::Tensor w, double eps, bool want_swz,
                                      double offset) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && w.is_contiguous() &&
              x.dim() == 2 && x.scalar_type() == at::kFloat &&
              w.numel() == x.size(1), "rmsnorm_res32: x [T, D] f32, w [D]");
  const int64_t n_rows = x.size(0);
  const int D = (int)x.size(1);
  const bool bf16 = w.scalar_type() == at::kBFloat16;
  TORCH_CHECK(bf16 || w.scalar_type() == at::kFloat, "rmsnorm_res32: w dtype");
  TORCH_CHECK(!want_swz || (bf16 && n_rows <= 32 && D % 16 == 0),
              "rmsnorm_res32: operand shape");
  auto y = at::empty(x.sizes(), w.options());
  auto swz = at::empty({want_swz ? (int64_t)(D / 16) * 512 : 0}, w.options());
  int nd = 0;
  bool d16 = false;
  void *dp = nullptr;
  if (delta.has_value()) {
    const at::Tensor &d = *delta;
    TORCH_CHECK(d.is_cuda() && d.is_contiguous() && d.size(-1) == D &&
                d.size(-2) == n_rows && (d.dim() == 2 || d.dim() == 3),
                "rmsnorm_res32: delta shape");
    d16 = d.scalar_type() == at::kBFloat16;
    TORCH_CHECK(d16 || d.scalar_type() == at::kFloat,
                "rmsnorm_res32: delta dtype");
    nd = d.dim() == 3 ? (int)d.size(0) : 1;
    dp = d.data_ptr();
  }
  if (n_rows == 0) return {y, swz};
  auto stream = at::hip::getCurrentHIPStream();
  const dim3 grid(std::min<int64_t>(n_rows, 4096));
#define RB_RES32(T, DT, V)                                                   \
  hipLaunchKernelGGL((rmsnorm_res32_kernel<T, DT, V>), grid, dim3(BLOCK), 0, \
                     stream, x.data_ptr<float>(), (const DT *)dp, nd,        \
                     (const T *)w.data_ptr(), (T *)y.data_ptr(),             \
                     want_swz ? (uint16_t *)swz.data_ptr() : nullptr,        \
                     n_rows, D, (float)eps, (float)offset)
#define RB_RES32_V(V)                                  \
  if (bf16 && d16) RB_RES32(uint16_t, uint16_t, V);    \
  else if (bf16) RB_RES32(uint16_t, float, V);         \
  else if (d16) RB_RES32(float, uint16_t, V);          \
  else RB_RES32(float, float, V)
  if (D % 8 == 0) { RB_RES32_V(8); } else { RB_RES32_V(1); }
#undef RB_RES32_V
#undef RB_RES32
  return {y, swz};
}

namespace {
template <typename T>
void launch_bwd(const at::Tensor &x, const at::Tensor &w, const at::Tensor &dy,
                const at::Tensor &inv_rms, const at::Tensor *add,
                at::Tensor &dx, float *dw, int64_t n_rows, int D) {
  auto stream = at::hip::getCurrentHIPStream();
  const T *ap = add == nullptr ? nullptr : (const T *)add->data_ptr();
  const int nv = (D / rb::VIO<T>::W + BLOCK - 1) / BLOCK;
  auto go = [&](auto kernel, size_t shmem, int64_t most, float *out) {
    hipLaunchKernelGGL(kernel, dim3(std::min<int64_t>(n_rows, most)),
                       dim3(BLOCK), shmem, stream, (const T *)x.data_ptr(),
                       (const T *)w.data_ptr(), (const T *)dy.data_ptr(),
                       inv_rms.data_ptr<float>(), ap, (T *)dx.data_ptr(), out,
                       n_rows, D);
  };
  auto pick = [&](auto with_dw) {
    constexpr bool DW = decltype(with_dw)::value;
    const int64_t most = DW ? 512 : 2048;
    const int n = (int)std::min(n_rows, most);
    at::Tensor part;
    if (DW) part = at::empty({n, D}, x.options().dtype(at::kFloat));
    float *out = DW ? part.data_ptr<float>() : nullptr;
    if (nv <= 1) go(rmsnorm_bwd_reg_kernel<T, 1, DW>, 0, most, out);
    else if (nv == 2) go(rmsnorm_bwd_reg_kernel<T, 2, DW>, 0, most, out);
    else go(rmsnorm_bwd_reg_kernel<T, 4, DW>, 0, most, out);
    if (DW)
      hipLaunchKernelGGL(rmsnorm_dw_kernel, dim3((D + 63) / 64), dim3(BLOCK),
                         0, stream, out, dw, n, D);
  };
  if (nv > 4) {
    const size_t shmem = ((size_t)D + BLOCK / RB_WAVE) * sizeof(float);
    TORCH_CHECK(shmem <= 160 * 1024,
                "rmsnorm_bwd: D too large for LDS accumulation");
    go(rmsnorm_bwd_kernel<T>, shmem, 512, dw);
  } else if (dw != nullptr) {
    pick(std::true_type{});
  } else {
    pick(std::false_type{});
  }
}
}  // namespace

// {dx (+ add), dw fp32, undefined without need_dw}
std::vector<at::Tensor> rmsnorm_bwd(at::Tensor x, at::Tensor w, at::Tensor dy,
                                    at::Tensor inv_rms, bool need_dw,
                                    c10::optional<at::Tensor> add) {
  TORCH_CHECK(x.is_cuda() && dy.is_contiguous() && x.is_contiguous() &&
              dy.sizes() == x.sizes() && w.is_contiguous() &&
              dy.scalar_type() == x.scalar_type() &&
              w.scalar_type() == x.scalar_type(), "rmsnorm_bwd: bad args");
  TORCH_CHECK(!add.has_value() ||
              (add->is_contiguous() && add->sizes() == x.sizes() &&
               add->scalar_type() == x.scalar_type()), "rmsnorm_bwd: add");
  const int D = (int)x.size(-1);
  const int64_t n_rows = D ? x.numel() / D : 0;
  auto dx = at::empty_like(x);
  at::Tensor dw;
  // rows wider than the register kernels' always make dw
  const int wide = 4 * BLOCK * (x.scalar_type() == at::kBFloat16 ? 8 : 4);
  if (need_dw || D > wide)
    dw = at::zeros({D}, x.options().dtype(at::kFloat));
  float *dwp = dw.defined() ? dw.data_ptr<float>() : nullptr;
  const at::Tensor *ap = add.has_value() ? &*add : nullptr;
  if (n_rows == 0) return {dx, dw};
  if (x.scalar_type() == at::kBFloat16)
    launch_bwd<uint16_t>(x, w, dy, inv_rms, ap, dx, dwp, n_rows, D);
  else if (x.scalar_type() == at::kFloat)
    launch_bwd<float>(x, w, dy, inv_rms, ap, dx, dwp, n_rows, D);
  else
    TORCH_CHECK(false, "rmsnorm_bwd: unsupported dtype");
  return {dx, dw};
}
