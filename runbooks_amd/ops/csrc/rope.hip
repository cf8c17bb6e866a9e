// Rotary position embedding (RoPE, neox/llama rotate-half convention)
// forward + backward for CDNA4 (gfx950).
//
// cos/sin tables are precomputed on the HOST (guide: on-device trig turns
// a memory-bound op VALU-bound) as fp32 [max_pos, Dh/2].
//
//   y[p, h, i]        = x[i]  * cos[p, i] - x[i+Dh/2] * sin[p, i]
//   y[p, h, i+Dh/2]   = x[i+Dh/2] * cos[p, i] + x[i]  * sin[p, i]
//
// Backward is the inverse rotation (sin negated) — same kernel.
//
// x layout: [rows, Dh] contiguous, where row r belongs to token r / H
// (H heads per token) and positions[token] gives p. q and k are rotated in
// one call each from Python.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

namespace {

constexpr int BLOCK = 256;

// Each thread handles VP=4 (i, i+Dh/2) pairs: 8-byte bf16x4 loads per half.
template <typename T, bool BWD>
__global__ void rope_kernel(const T *__restrict__ x, T *__restrict__ y,
                            const float *__restrict__ cs,   // [max_pos, half] cos
                            const float *__restrict__ sn,   // [max_pos, half] sin
                            const int32_t *__restrict__ pos,  // [n_tokens]
                            int64_t n_rows, int heads, int half) {
  constexpr int VP = 4;
  const int nvec = half / VP;
  const int64_t total = n_rows * nvec;
  const int64_t stride = (int64_t)gridDim.x * BLOCK;

  for (int64_t idx = (int64_t)blockIdx.x * BLOCK + threadIdx.x; idx < total;
       idx += stride) {
    const int64_t row = idx / nvec;
    const int v = (int)(idx % nvec);
    const int64_t token = row / heads;
    const int p = pos[token];

    const T *x1 = x + row * 2 * half + v * VP;
    const T *x2 = x1 + half;
    T *y1 = y + row * 2 * half + v * VP;
    T *y2 = y1 + half;
    const float *c = cs + (int64_t)p * half + v * VP;
    const float *s = sn + (int64_t)p * half + v * VP;

#pragma unroll
    for (int k = 0; k < VP; ++k) {
      const float a = rb::bf16_to_f32_or_id(x1[k]);
      const float b = rb::bf16_to_f32_or_id(x2[k]);
      const float sk = BWD ? -s[k] : s[k];
      rb::store_scalar(y1 + k, a * c[k] - b * sk);
      rb::store_scalar(y2 + k, b * c[k] + a * sk);
    }
  }
}

}  // namespace

template <bool BWD>
static at::Tensor rope_apply_impl(at::Tensor x, at::Tensor cos, at::Tensor sin,
                                  at::Tensor positions, int64_t heads) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous(), "rope: x must be contiguous GPU");
  TORCH_CHECK(cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat,
              "rope: cos/sin must be fp32");
  TORCH_CHECK(positions.scalar_type() == at::kInt, "rope: positions must be int32");
  const int Dh = (int)x.size(-1);
  const int half = Dh / 2;
  TORCH_CHECK(half % 4 == 0, "rope: Dh/2 must be a multiple of 4");
  TORCH_CHECK(cos.size(-1) == half, "rope: cos table must be [max_pos, Dh/2]");
  const int64_t n_rows = x.numel() / Dh;
  auto y = at::empty_like(x);
  auto stream = at::hip::getCurrentHIPStream();
  const int grid = rb::rb_grid_1d(n_rows * (half / 4), BLOCK);

  if (x.scalar_type() == at::kBFloat16) {
    hipLaunchKernelGGL((rope_kernel<uint16_t, BWD>), dim3(grid), dim3(BLOCK), 0, stream,
                       (const uint16_t *)x.data_ptr(), (uint16_t *)y.data_ptr(),
                       cos.data_ptr<float>(), sin.data_ptr<float>(),
                       positions.data_ptr<int32_t>(), n_rows, (int)heads, half);
  } else if (x.scalar_type() == at::kFloat) {
    hipLaunchKernelGGL((rope_kernel<float, BWD>), dim3(grid), dim3(BLOCK), 0, stream,
                       x.data_ptr<float>(), y.data_ptr<float>(),
                       cos.data_ptr<float>(), sin.data_ptr<float>(),
                       positions.data_ptr<int32_t>(), n_rows, (int)heads, half);
  } else {
    TORCH_CHECK(false, "rope: unsupported dtype");
  }
  return y;
}

at::Tensor rope_fwd(at::Tensor x, at::Tensor cos, at::Tensor sin,
                    at::Tensor positions, int64_t heads) {
  return rope_apply_impl<false>(x, cos, sin, positions, heads);
}

at::Tensor rope_bwd(at::Tensor dy, at::Tensor cos, at::Tensor sin,
                    at::Tensor positions, int64_t heads) {
  return rope_apply_impl<true>(dy, cos, sin, positions, heads);
}

// ---------------------------------------------------------------------------
// q, k and v side by side in the rows of y [T, (hq + 2 hkv) * dh]: rotates q and
// k in place. INVERSE, of gradients: the other way round; with dk and dv per
// query head ([T, hq, dh]) the heads of a group are summed first, into y's
// columns. A lane takes 8 values and the 8 they rotate with.
// ---------------------------------------------------------------------------
namespace {

template <bool INVERSE>
__global__ __launch_bounds__(BLOCK) void rope_qkv_kernel(
    uint16_t *__restrict__ y, const uint16_t *__restrict__ dk,
    const uint16_t *__restrict__ dv, const float *__restrict__ cs,
    const float *__restrict__ sn, const int32_t *__restrict__ pos, int64_t T,
    int hq, int hkv, int dh) {
  const int half = dh / 2, lanes = half / 8, heads = hq + 2 * hkv;
  const int used = INVERSE && dk != nullptr ? heads : hq + hkv;
  const int group = hq / hkv;
  const int64_t total = T * used * lanes;
  const int64_t stride = (int64_t)gridDim.x * BLOCK;
  for (int64_t idx = (int64_t)blockIdx.x * BLOCK + threadIdx.x; idx < total;
       idx += stride) {
    const int64_t row = idx / lanes;
    const int d = (int)(idx % lanes) * 8;
    const int64_t t = row / used;
    const int h = (int)(row % used);
    uint16_t *at = y + (t * heads + h) * dh + d;
    float a[8], b[8];
    if (INVERSE && dk != nullptr && h >= hq) {
      const bool is_v = h >= hq + hkv;
      const int kh = h - hq - (is_v ? hkv : 0);
      const uint16_t *src =
          (is_v ? dv : dk) + (t * hq + (int64_t)kh * group) * dh + d;
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] = b[e] = 0.0f;
      for (int g = 0; g < group; ++g) {
        float u[8], w[8];
        rb::VIO<uint16_t>::load(src + (int64_t)g * dh, u);
        rb::VIO<uint16_t>::load(src + (int64_t)g * dh + half, w);
#pragma unroll
        for (int e = 0; e < 8; ++e) { a[e] += u[e]; b[e] += w[e]; }
      }
    } else {
      rb::VIO<uint16_t>::load(at, a);
      rb::VIO<uint16_t>::load(at + half, b);
    }
    if (h < hq + hkv) {
      const int64_t p = (int64_t)pos[t] * half + d;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float c = cs[p + e], s = INVERSE ? -sn[p + e] : sn[p + e];
        const float u = a[e];
        a[e] = u * c - b[e] * s;
        b[e] = b[e] * c + u * s;
      }
    }
    rb::VIO<uint16_t>::store(at, a);
    rb::VIO<uint16_t>::store(at + half, b);
  }
}

}  // namespace

void rope_qkv_(at::Tensor y, at::Tensor cos, at::Tensor sin,
               at::Tensor positions, int64_t hq, int64_t hkv, int64_t dh,
               bool inverse, c10::optional<at::Tensor> dk,
               c10::optional<at::Tensor> dv) {
  TORCH_CHECK(y.is_cuda() && y.is_contiguous() && y.dim() == 2 &&
              y.scalar_type() == at::kBFloat16 && hkv > 0 && hq % hkv == 0 &&
              y.size(1) == (hq + 2 * hkv) * dh && dh % 16 == 0 &&
              positions.scalar_type() == at::kInt &&
              positions.is_contiguous() && positions.numel() >= y.size(0) &&
              cos.size(-1) == dh / 2 && sin.sizes() == cos.sizes() &&
              cos.scalar_type() == at::kFloat && cos.is_contiguous() &&
              sin.is_contiguous() && sin.scalar_type() == at::kFloat,
              "rope_qkv_: y, tables");
  const int64_t T = y.size(0);
  const bool grouped = dk.has_value() && dk->numel() > 0;
  TORCH_CHECK(!grouped || (inverse && dv.has_value() && dk->is_contiguous() &&
                           dv->is_contiguous() &&
                           dk->numel() == T * hq * dh &&
                           dv->numel() == dk->numel() &&
                           dk->scalar_type() == at::kBFloat16 &&
                           dv->scalar_type() == at::kBFloat16),
              "rope_qkv_: dk, dv per query head");
  if (T == 0) return;
  const int64_t rows = T * (hq + (grouped ? 2 : 1) * hkv);
  const int grid = rb::rb_grid_1d(rows * (dh / 16), BLOCK);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(BLOCK), 0,
                       at::hip::getCurrentHIPStream(),
                       (uint16_t *)y.data_ptr(),
                       grouped ? (const uint16_t *)dk->data_ptr() : nullptr,
                       grouped ? (const uint16_t *)dv->data_ptr() : nullptr,
                       cos.data_ptr<float>(), sin.data_ptr<float>(),
                       positions.data_ptr<int32_t>(), T, (int)hq, (int)hkv,
                       (int)dh);
  };
  if (inverse) go(rope_qkv_kernel<true>);
  else go(rope_qkv_kernel<false>);
}
