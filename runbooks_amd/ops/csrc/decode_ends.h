// What becomes of a decode product's sums (decode_gemm.hip) before they leave
// the kernel: the gate of a gated unit, the rotation of queries and keys and
// their way into the paged cache, the factor of a norm that was left out of the
// product's input.
//
// A launch of its own for each of these takes 2 to 4 us of a captured step,
// whatever it computes. Gate and unit of a column, and the two halves of a
// head's rotation, have to meet in one thread for it: copies of such weights
// hold their rows in pairs (decode_swizzle_w, `half`), block n of 32 rows being
// 16 rows and the 16 that lie `half` rows further on.
//
// us in a graph, weights out of cache, apart and here, of 1, 16 and 32 rows:
//   q, k, v and rotation  12288 x 4096       22.1 20.5  23.7 21.7  25.2 23.2
//                         12288 x 4096 e4m3  16.3 13.7  16.4 14.5  19.8 17.9
//                         6144 x 4096        16.9 12.2  18.2 12.8  19.4 13.7
//   gated unit            22016 x 4096       35.1 33.3  35.2 32.5  35.8 32.9
//                         22016 x 4096 e4m3  22.0 20.4  23.0 20.8  27.4 24.2
//                         49152 x 3072       51.0 49.2  50.1 47.0  57.6 52.8
// (6144 columns were split before, for their number of workgroups; the products are
// faster since, decode_gemm.hip, with their ends and without). The sums of
// squares add 0.3 us. A step of llama2-7b, with the residual sums of
// decode_res.hip and attention by whole sequences: one sequence 3335 -> 2972, 32
// 7026 -> 6534.
#pragma once

#include "common.h"

namespace ends {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8v;
typedef __attribute__((ext_vector_type(16))) float f32x16v;
typedef __attribute__((ext_vector_type(4))) float f32x4v;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4v;

RB_DEV bf16x8v load8v(const uint16_t *p) {
  union { u32x4v u; bf16x8v v; } c;
  c.u = *reinterpret_cast<const u32x4v *>(p);
  return c.v;
}

// Two words of e4m3 -> 8 bf16 (exact).
RB_DEV bf16x8v fp8_to_bf16(unsigned lo, unsigned up) {
  union { unsigned u[4]; bf16x8v v; } c;
  c.u[0] = rb::fp8_pair_bf16<false>(lo);
  c.u[1] = rb::fp8_pair_bf16<true>(lo);
  c.u[2] = rb::fp8_pair_bf16<false>(up);
  c.u[3] = rb::fp8_pair_bf16<true>(up);
  return c.v;
}

enum Kind {
  SLAB,     // fp32 parts of the sums
  PLAIN,    // y [M, N] bf16
  GLU,      // act(first half) * second half, [M, N / 2]
  QKV,      // rotated q; rotated k and v to the cache
};

struct Ends {
  uint16_t *y;            // PLAIN, GLU: rows; QKV: rows of all heads (or null)
  float *slabs;
  const float *scale;     // of W's rows, in their own order (or null)
  int half;               // distance of paired rows; 0: rows in order
  uint16_t *operand;      // GLU: [N / 32][2][32][8] (or null)
  // input without its norm's 1 / rms: sums of squares of its rows [M, parts],
  // parts a multiple of 4 (or null)
  const float *squares;
  int parts;
  float inv_d, eps;
  bool gelu;              // GLU: tanh-GELU, else SiLU
  uint16_t *q;            // QKV: [M, hq, dh] (or null)
  uint16_t *k_cache, *v_cache;
  const float *cs, *sn;
  const int32_t *pos, *slots;
  int hq, hkv, dh, bs;
  bool vt;
};

// Column of y of row r of W's block n.
RB_DEV int column(int half, int n, int r) {
  if (half == 0) return n * 32 + r;
  const int p = n * 16;
  return p / half * 2 * half + p % half + (r < 16 ? r : half + r - 16);
}

RB_DEV float gate(float g, float u, bool gelu) {
  if (gelu) {           // 0.5 (1 + tanh(z)) = 1 / (1 + exp(-2 z))
    const float z2 = 1.5957691216057308f * (g + 0.044715f * g * g * g);
    return g * __builtin_amdgcn_rcpf(1.0f + __expf(-z2)) * u;
  }
  return g / (1.0f + __expf(-g)) * u;
}

template <int V> RB_DEV void put(uint16_t *p, const float *f) {
  static_assert(V == 2 || V == 4, "pieces");
  if constexpr (V == 2)
    *reinterpret_cast<uint32_t *>(p) = rb::pack_bf16x2(f[0], f[1]);
  else
    *reinterpret_cast<uint2 *>(p) = make_uint2(rb::pack_bf16x2(f[0], f[1]),
                                               rb::pack_bf16x2(f[2], f[3]));
}

// Angles and slot of row m, pairs p .. p + V.
template <int V> struct Turn {
  float c[V], s[V];
  int slot;
  RB_DEV void load(const Ends &e, int m, int p, int position) {
    const int half = e.dh / 2;
    const int64_t at = (int64_t)position * half + p % half;
#pragma unroll
    for (int i = 0; i < V; i += 2) {
      const float2 x = *reinterpret_cast<const float2 *>(e.cs + at + i);
      const float2 z = *reinterpret_cast<const float2 *>(e.sn + at + i);
      c[i] = x.x; c[i + 1] = x.y;
      s[i] = z.x; s[i + 1] = z.y;
    }
    slot = e.slots[m];
  }
};

// The pairs (a[i], b[i]) of row m with the numbers p + i, V of them within 16.
template <int V>
RB_DEV void put_gated(const Ends &e, int m, int p, int N, const float *a,
                      const float *b) {
  float h[V];
#pragma unroll
  for (int i = 0; i < V; ++i) h[i] = gate(a[i], b[i], e.gelu);
  if (e.operand != nullptr)
    put<V>(e.operand + (p >> 4) * 512 + (p >> 3 & 1) * 256 + m * 8 + (p & 7),
           h);
  if (e.y != nullptr) put<V>(e.y + (int64_t)m * (N / 2) + p, h);
}

template <int V>
RB_DEV void put_heads(const Ends &e, const Turn<V> &t, int m, int p, int N,
                      float *a, float *b) {
  const int half = e.dh / 2, h = p / half, d = p % half;
  if (h < e.hq + e.hkv) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const float x = a[i], z = b[i];
      a[i] = x * t.c[i] - z * t.s[i];
      b[i] = z * t.c[i] + x * t.s[i];
    }
  }
  if (e.y != nullptr) {
    uint16_t *dst = e.y + (int64_t)m * N + h * e.dh + d;
    put<V>(dst, a);
    put<V>(dst + half, b);
  }
  if (h < e.hq) {
    if (e.q == nullptr) return;
    uint16_t *dst = e.q + ((int64_t)m * e.hq + h) * e.dh + d;
    put<V>(dst, a);
    put<V>(dst + half, b);
    return;
  }
  if (t.slot < 0) return;
  const bool value = h >= e.hq + e.hkv;
  const int kh = h - e.hq - (value ? e.hkv : 0);
  const int64_t head = (int64_t)(t.slot / e.bs) * e.hkv + kh;
  const int off = t.slot % e.bs;
  if (value && e.vt) {
    uint16_t *dst = e.v_cache + (head * e.dh + d) * e.bs + off;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      dst[i * e.bs] = rb::f32_to_bf16(a[i]);
      dst[(int64_t)(half + i) * e.bs] = rb::f32_to_bf16(b[i]);
    }
  } else {
    uint16_t *dst = (value ? e.v_cache : e.k_cache) +
                    (head * e.bs + off) * e.dh + d;
    put<V>(dst, a);
    put<V>(dst + half, b);
  }
}

}  // namespace ends
