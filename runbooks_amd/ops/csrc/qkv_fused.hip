// What follows the fused QKV product of the serving path for CDNA4 (gfx950).
//
// y [T, (Hq + 2 Hkv) * Dh] -> RoPE'd q, RoPE'd k and plain v appended straight
// into the paged KV cache (kvcache.hip's layouts: rows or transposed values,
// bf16 or e4m3). In decoding q goes to a tensor of its own; in prompts q and k
// are rotated in place and the flash kernel reads q, k and v out of y, so that
// one launch stands for three slice copies, two rotations and the append.
//
// Memory-bound: a lane takes 8 values of a head's first half and the 8 of its
// second half they rotate with (16-byte accesses). Transposed values of prompts
// go 16 tokens at a time, a cache block's 16 columns: 64 contiguous bytes a
// lane instead of 2 at a stride. us for a prompt of 7931 tokens, 32 query and 8
// kv heads of 128: 127 -> 37 (512 tokens, 32 heads: 27 -> 6).
//
// RoPE is rotate-half with fp32 host tables (rope.hip).

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

namespace {

constexpr int BLOCK = 256;
constexpr int GROUP = 16;        // tokens of a cache block

struct Args {
  uint16_t *y;                   // rotated in place when q == nullptr
  uint16_t *q;
  void *k_cache, *v_cache;
  const float *cs, *sn;
  const int32_t *pos, *slots;
  int64_t T;
  int hq, hkv, dh, bs;
  int row_blocks;                // workgroups of rows; the others transpose
};

template <int V> struct Chunk {
  uint16_t v[V];
  RB_DEV void load(const uint16_t *p) {
    *this = *reinterpret_cast<const Chunk *>(p);
  }
  RB_DEV void store(uint16_t *p) const { *reinterpret_cast<Chunk *>(p) = *this; }
};
template <> RB_DEV void Chunk<8>::load(const uint16_t *p) {
  *reinterpret_cast<uint4 *>(v) = *reinterpret_cast<const uint4 *>(p);
}
template <> RB_DEV void Chunk<8>::store(uint16_t *p) const {
  *reinterpret_cast<uint4 *>(p) = *reinterpret_cast<const uint4 *>(v);
}

// A row's two chunks as e4m3 with the row's scale; its `lanes` lanes are
// neighbours.
template <int V>
RB_DEV float quantize(const Chunk<V> &a, const Chunk<V> &b, int lanes,
                      uint8_t *qa, uint8_t *qb) {
  float amax = 1e-8f;
#pragma unroll
  for (int e = 0; e < V; ++e)
    amax = fmaxf(amax, fmaxf(fabsf(rb::bf16_to_f32(a.v[e])),
                             fabsf(rb::bf16_to_f32(b.v[e]))));
  for (int off = lanes / 2; off > 0; off >>= 1)
    amax = fmaxf(amax, __shfl_xor(amax, off, 64));
  const float scale = amax / 448.0f, inv = 1.0f / scale;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    qa[e] = rb::f32_to_fp8(rb::bf16_to_f32(a.v[e]) * inv);
    qb[e] = rb::f32_to_fp8(rb::bf16_to_f32(b.v[e]) * inv);
  }
  return scale;
}

template <int V, bool FP8, bool VT>
__global__ __launch_bounds__(BLOCK) void qkv_rope_append_kernel(Args a) {
  const int half = a.dh / 2, lanes = half / V;
  const int heads = a.hq + 2 * a.hkv;
  const int64_t width = (int64_t)heads * a.dh;

  if ((int)blockIdx.x >= a.row_blocks) {
    // bf16 values of 16 tokens at a time, a wave for each head
    if constexpr (!FP8 && VT) {
      const int lane = threadIdx.x & 63;
      const int64_t unit = (int64_t)(blockIdx.x - a.row_blocks) * (BLOCK / 64) +
                           (threadIdx.x >> 6);
      const int64_t t0 = unit / a.hkv * GROUP;
      const int h = (int)(unit % a.hkv);
      if (t0 >= a.T) return;
      const int n = (int)min((int64_t)GROUP, a.T - t0);
      const int first = a.slots[t0];
      const bool whole = __all(
          lane >= GROUP || (lane < n && first % GROUP == 0 && first >= 0 &&
                            a.slots[t0 + min(lane, n - 1)] == first + lane));
      const uint16_t *src = a.y + t0 * width + (int64_t)(a.hq + a.hkv + h) * a.dh;
      uint16_t *vc = (uint16_t *)a.v_cache;
      for (int d = lane * 2; d < a.dh; d += 128) {
        uint32_t x[GROUP];
#pragma unroll
        for (int i = 0; i < GROUP; ++i)
          x[i] = *reinterpret_cast<const uint32_t *>(
              src + min(i, n - 1) * width + d);
        if (whole) {
          uint16_t *dst =
              vc + (((int64_t)(first / GROUP) * a.hkv + h) * a.dh + d) * GROUP;
#pragma unroll
          for (int r = 0; r < 4; ++r) {          // two rows of 16 columns
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const uint32_t lo = x[r % 2 * 8 + 2 * i];
              const uint32_t up = x[r % 2 * 8 + 2 * i + 1];
              w[i] = r < 2 ? (lo & 0xffff) | up << 16
                           : lo >> 16 | (up & 0xffff0000u);
            }
            reinterpret_cast<uint4 *>(dst)[r] =
                make_uint4(w[0], w[1], w[2], w[3]);
          }
        } else {
#pragma unroll
          for (int i = 0; i < GROUP; ++i) {
            const int slot = a.slots[t0 + min(i, n - 1)];
            if (i >= n || slot < 0) continue;
            uint16_t *dst = vc + (((int64_t)(slot / GROUP) * a.hkv + h) *
                                  a.dh + d) * GROUP + slot % GROUP;
            dst[0] = (uint16_t)x[i];
            dst[GROUP] = (uint16_t)(x[i] >> 16);
          }
        }
      }
    }
    return;
  }

  // without transposing workgroups this one's rows include the values
  const bool values = gridDim.x == (unsigned)a.row_blocks;
  const int used = values ? heads : a.hq + a.hkv;
  const int64_t total = a.T * used * lanes;
  const int64_t stride = (int64_t)a.row_blocks * BLOCK;
  for (int64_t idx = (int64_t)blockIdx.x * BLOCK + threadIdx.x; idx < total;
       idx += stride) {
    const int64_t row = idx / lanes;
    const int d = (int)(idx % lanes) * V;
    const int64_t t = row / used;
    const int h = (int)(row % used);
    uint16_t *src = a.y + t * width + (int64_t)h * a.dh + d;
    Chunk<V> x, z;
    x.load(src);
    z.load(src + half);
    // before the rotation waits for the position
    const int slot = a.slots[t];
    if (h < a.hq + a.hkv) {
      const int64_t p = (int64_t)a.pos[t] * half + d;
      float cs[V], sn[V];
      __builtin_memcpy(cs, a.cs + p, sizeof(cs));   // tables begin anywhere
      __builtin_memcpy(sn, a.sn + p, sizeof(sn));
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float u = rb::bf16_to_f32(x.v[e]), w = rb::bf16_to_f32(z.v[e]);
        const float c = cs[e], s = sn[e];
        x.v[e] = rb::f32_to_bf16(u * c - w * s);
        z.v[e] = rb::f32_to_bf16(w * c + u * s);
      }
      if (a.q == nullptr) {
        x.store(src);
        z.store(src + half);
      } else if (h < a.hq) {
        uint16_t *dst = a.q + (t * a.hq + h) * a.dh + d;
        x.store(dst);
        z.store(dst + half);
      }
      if (h < a.hq) continue;
    }
    const bool is_v = h >= a.hq + a.hkv;
    const int kh = h - a.hq - (is_v ? a.hkv : 0);
    uint8_t qx[V], qz[V];
    float scale = 0.0f;
    // all lanes of a row take part, whatever its slot
    if constexpr (FP8) scale = quantize(x, z, lanes, qx, qz);
    if (slot < 0) continue;
    const int64_t head = (int64_t)(slot / a.bs) * a.hkv + kh;
    const int off = slot % a.bs;
    if constexpr (FP8) {
      if (VT && is_v) {
        uint8_t *vb = (uint8_t *)a.v_cache + head * (a.dh + 4) * a.bs;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          vb[(int64_t)(d + e) * a.bs + off] = qx[e];
          vb[(int64_t)(half + d + e) * a.bs + off] = qz[e];
        }
        if (d == 0)
          *reinterpret_cast<float *>(vb + (int64_t)a.dh * a.bs + off * 4) =
              scale;
      } else {
        uint8_t *dst = (uint8_t *)(is_v ? a.v_cache : a.k_cache) +
                       (head * a.bs + off) * (a.dh + 16) + d;
        __builtin_memcpy(dst, qx, V);
        __builtin_memcpy(dst + half, qz, V);
        if (d == 0) *reinterpret_cast<float *>(dst + a.dh) = scale;
      }
    } else if (VT && is_v) {
      uint16_t *vb = (uint16_t *)a.v_cache + head * a.dh * a.bs + off;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        vb[(int64_t)(d + e) * a.bs] = x.v[e];
        vb[(int64_t)(half + d + e) * a.bs] = z.v[e];
      }
    } else {
      uint16_t *dst = (uint16_t *)(is_v ? a.v_cache : a.k_cache) +
                      (head * a.bs + off) * a.dh + d;
      x.store(dst);
      z.store(dst + half);
    }
  }
}

void run(const at::Tensor &y, uint16_t *q, const at::Tensor &cos,
         const at::Tensor &sin, const at::Tensor &positions,
         const at::Tensor &k_cache, const at::Tensor &v_cache,
         const at::Tensor &slots, int64_t hq) {
  TORCH_CHECK(y.is_cuda() && y.is_contiguous() && y.dim() == 2 &&
              y.scalar_type() == at::kBFloat16 &&
              reinterpret_cast<uintptr_t>(y.data_ptr()) % 16 == 0,
              "qkv_rope_append: y");
  TORCH_CHECK(positions.scalar_type() == at::kInt &&
              slots.scalar_type() == at::kInt && positions.is_contiguous() &&
              slots.is_contiguous(), "qkv_rope_append: idx");
  const bool fp8 = k_cache.scalar_type() == at::kByte;
  TORCH_CHECK((fp8 || k_cache.scalar_type() == at::kBFloat16) &&
              v_cache.scalar_type() == k_cache.scalar_type() &&
              k_cache.is_contiguous() && v_cache.is_contiguous(),
              "qkv_rope_append: caches");
  Args a{};
  a.y = (uint16_t *)y.data_ptr();
  a.q = q;
  a.k_cache = k_cache.data_ptr();
  a.v_cache = v_cache.data_ptr();
  a.cs = cos.data_ptr<float>();
  a.sn = sin.data_ptr<float>();
  a.pos = positions.data_ptr<int32_t>();
  a.slots = slots.data_ptr<int32_t>();
  a.T = y.size(0);
  a.hq = (int)hq;
  a.hkv = (int)k_cache.size(1);
  a.bs = (int)k_cache.size(2);
  a.dh = (int)k_cache.size(3) - (fp8 ? 16 : 0);
  TORCH_CHECK((int64_t)(a.hq + 2 * a.hkv) * a.dh == y.size(1),
              "qkv_rope_append: packed width mismatch");
  TORCH_CHECK(positions.numel() >= a.T && slots.numel() >= a.T &&
              cos.size(-1) == a.dh / 2 && sin.sizes() == cos.sizes(),
              "qkv_rope_append: sizes");
  TORCH_CHECK((a.dh / 2) % 4 == 0, "qkv_rope_append: Dh/2 % 4");
  TORCH_CHECK(!fp8 || a.dh == 64 || a.dh == 128 || a.dh == 256,
              "qkv_rope_append: fp8 Dh");
  const bool vt = v_cache.size(3) == a.bs &&
                  v_cache.size(2) == a.dh + (fp8 ? 4 : 0) && a.dh != a.bs;
  if (a.T == 0) return;
  const int V = (a.dh / 2) % 8 == 0 ? 8 : 4;
  // fewer tokens than this are no whole blocks worth a wave each
  const bool transpose = vt && !fp8 && a.bs == GROUP && a.dh % 2 == 0 &&
                         a.T >= 64;
  a.row_blocks = rb::rb_grid_1d(
      a.T * (a.hq + (transpose ? 1 : 2) * a.hkv) * (a.dh / 2 / V), BLOCK);
  int64_t grid = a.row_blocks;
  if (transpose)
    grid += ((a.T + GROUP - 1) / GROUP * a.hkv + BLOCK / 64 - 1) / (BLOCK / 64);
  TORCH_CHECK(grid < (int64_t)1 << 31, "qkv_rope_append: grid");
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(BLOCK), 0,
                       at::hip::getCurrentHIPStream(), a);
  };
  if (fp8)
    vt ? go(qkv_rope_append_kernel<8, true, true>)
       : go(qkv_rope_append_kernel<8, true, false>);
  else if (V == 8)
    vt ? go(qkv_rope_append_kernel<8, false, true>)
       : go(qkv_rope_append_kernel<8, false, false>);
  else
    vt ? go(qkv_rope_append_kernel<4, false, true>)
       : go(qkv_rope_append_kernel<4, false, false>);
}

}  // namespace

// Rotated q [T, hq, Dh]; y stays as it is.
at::Tensor qkv_rope_append(at::Tensor y, at::Tensor cos, at::Tensor sin,
                           at::Tensor positions, at::Tensor k_cache,
                           at::Tensor v_cache, at::Tensor slot_mapping,
                           int64_t hq) {
  const int64_t dh =
      k_cache.size(3) - (k_cache.scalar_type() == at::kByte ? 16 : 0);
  auto q = at::empty({y.size(0), hq, dh}, y.options());
  if (reinterpret_cast<uintptr_t>(y.data_ptr()) % 16) y = y.clone();
  run(y, (uint16_t *)q.data_ptr(), cos, sin, positions, k_cache, v_cache,
      slot_mapping, hq);
  return q;
}

// q and k rotated within y.
void qkv_rope_append_(at::Tensor y, at::Tensor cos, at::Tensor sin,
                      at::Tensor positions, at::Tensor k_cache,
                      at::Tensor v_cache, at::Tensor slot_mapping,
                      int64_t hq) {
  run(y, nullptr, cos, sin, positions, k_cache, v_cache, slot_mapping, hq);
}
