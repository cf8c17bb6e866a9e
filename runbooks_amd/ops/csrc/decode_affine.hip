// Decode of layer-norm models with biases (opt, gpt2) of up to 32 rows:
// act(x W^T + bias), with the norm before it and the residual sum or the cache
// write behind it.
//
// The residual is fp32 [M, D] of up to 1024 columns: every workgroup of a product
// (every wave, of up to 4 rows) norms it for itself, while its part of W is on its
// way, which is cheaper than a launch for the norm. A step of opt-125m with this,
// the embeddings in one launch and attention by whole sequences, with the block
// tables of a server: one sequence of 37 tokens 454 -> 289 us, 4 of 300 493 -> 366,
// 16 of 300 562 -> 457, 32 of 700 706 -> 597.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/macros/Macros.h>

#include "common.h"
#include "decode_ends.h"

namespace {

using ends::bf16x8v;
using ends::f32x4v;
using ends::load8v;

constexpr int BLOCK = 256;      // 4 waves
constexpr int MMAX = 32;
constexpr int WIDEST = 1024;    // columns of a residual that is normed here
constexpr int FEW = 4;          // rows of affine_few_kernel

// What the loads of W need comes first: the arguments of a launch are read from
// memory, 64 bytes at a time (with rows and columns of x behind it all, the
// products of gpt2-xl's step of one sequence took 0.4 us longer, of 8).
struct Affine {
  const uint16_t *w[3];                 // [rows, K] each
  int end[3];                           // columns before the next matrix
  int act;                              // 0 none, 1 relu, 2 gelu, 3 gelu_tanh
  const uint16_t *bias[3];              // may be null
  uint16_t *out[3];
  bool operand;                         // out[0] as [N/16][2][32][8]
  // x is the norm of a residual [M, K]
  const float *res;
  const uint16_t *gain, *shift;
  float eps;
  float *into;                          // [M, N] += the result
  // matrices 1 and 2 go to the cache as keys and values
  uint16_t *k_cache, *v_cache;
  const int32_t *slots;
  int hkv, dh, bs;
  bool vt;
};

__device__ __forceinline__ float activate(float x, int act) {
  if (act == 1) return x < 0.0f ? 0.0f : x;
  if (act == 2) return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
  if (act == 3)
    return 0.5f * x * (1.0f + tanhf(0.79788456080286536f *
                                    (x + 0.044715f * x * x * x)));
  return x;
}

// The matrix of column n, and its first column.
RB_DEV int matrix_of(const Affine &a, int n, int &first) {
  const int of = n < a.end[0] ? 0 : n < a.end[1] ? 1 : 2;
  first = of == 0 ? 0 : a.end[of - 1];
  return of;
}

// Columns c .. c + V of a key or value of sequence m to its slot.
template <int V>
RB_DEV void cache(const Affine &a, bool value, int m, int c,
                  const uint16_t *o) {
  const int slot = a.slots[m];
  if (slot < 0) return;
  const int64_t head = (int64_t)(slot / a.bs) * a.hkv + c / a.dh;
  const int d = c % a.dh, off = slot % a.bs;
  if (value && a.vt) {
#pragma unroll
    for (int j = 0; j < V; ++j)
      a.v_cache[(head * a.dh + d + j) * a.bs + off] = o[j];
  } else {
    uint16_t *dst = (value ? a.v_cache : a.k_cache) +
                    (head * a.bs + off) * a.dh + d;
    if constexpr (V == 1) {
      *dst = *o;
    } else {
#pragma unroll
      for (int j = 0; j < V; j += 2)
        *reinterpret_cast<uint32_t *>(dst + j) =
            *reinterpret_cast<const uint32_t *>(o + j);
    }
  }
}

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2v;
typedef __attribute__((ext_vector_type(2))) float f32x2v;

RB_DEV uint32_t pack2(float lo, float up) {
  union { bf16x2v v; uint32_t u; } c;
  c.v = __builtin_convertvector((f32x2v){lo, up}, bf16x2v);
  return c.u;
}
// c + the dot product of two pairs
RB_DEV float dot2(uint32_t a, uint32_t b, float c) {
  union { uint32_t u; bf16x2v v; } x, y;
  x.u = a;
  y.u = b;
  return __builtin_amdgcn_fdot2_f32_bf16(x.v, y.v, c, false);
}
RB_DEV float lower(uint32_t u) { return __uint_as_float(u << 16); }
RB_DEV float upper(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// The operand [K/8][M][8] of the residual's norm, in LDS: a row for a wave at a
// time, the next one on its way.
RB_DEV void normed_operand(const Affine &a, int M, int K, uint16_t *x) {
  constexpr int J = WIDEST / 256;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int c[J];
  uint2 gain[J], shift[J];
  float4 ahead[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {         // past the end: the last ones again
    c[j] = min(j * 256 + lane * 4, K - 4);
    ahead[j] = *reinterpret_cast<const float4 *>(
        a.res + (int64_t)min(wid, M - 1) * K + c[j]);
    gain[j] = *reinterpret_cast<const uint2 *>(a.gain + c[j]);
    shift[j] = *reinterpret_cast<const uint2 *>(a.shift + c[j]);
  }
  const float inv_k = 1.0f / (float)K;
  for (int m = wid; m < M; m += BLOCK / 64) {
    float f[J][4], sum[1] = {0.0f}, dev[1] = {0.0f};
#pragma unroll
    for (int j = 0; j < J; ++j) {
      f[j][0] = ahead[j].x; f[j][1] = ahead[j].y;
      f[j][2] = ahead[j].z; f[j][3] = ahead[j].w;
      ahead[j] = *reinterpret_cast<const float4 *>(
          a.res + (int64_t)min(m + BLOCK / 64, M - 1) * K + c[j]);
      if (j * 256 + lane * 4 < K)
        sum[0] += (f[j][0] + f[j][1]) + (f[j][2] + f[j][3]);
    }
    rb::lane_sums<64>(sum);
    const float mean = sum[0] * inv_k;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[j][i] -= mean;
        if (j * 256 + lane * 4 < K) dev[0] += f[j][i] * f[j][i];
      }
    rb::lane_sums<64>(dev);
    const float inv = rsqrtf(dev[0] * inv_k + a.eps);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (j * 256 + lane * 4 >= K) continue;
      const uint2 o = make_uint2(
          pack2(f[j][0] * inv * lower(gain[j].x) + lower(shift[j].x),
                f[j][1] * inv * upper(gain[j].x) + upper(shift[j].x)),
          pack2(f[j][2] * inv * lower(gain[j].y) + lower(shift[j].y),
                f[j][3] * inv * upper(gain[j].y) + upper(shift[j].y)));
      *reinterpret_cast<uint2 *>(x + ((c[j] >> 3) * M + m) * 8 + (c[j] & 7)) = o;
    }
  }
  // loads of W stay on their way
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The columns go to up to three matrices (q, k, v), or to the operand of the next
// product. W and bias are the parameters themselves, so that captured steps
// follow them too: a workgroup takes 16 rows of W as they lie, its waves parts of
// the sums, 64 bytes of each row an instruction (16x16x32 products:
// A[i=l&15][k=(l>>4)*8+e], B[k][j=l&15], C[j=l&15][i=(l>>4)*4+r]).
//
// us in a graph, weights out of cache, on the library without the activation, in
// the layout of decode_gemm (32 rows a workgroup) and here, of 1 and 32 rows:
//   q, k, v 768 x 768   21  4.3  3.6   20  5.1  4.0
//   768 x 768            6.8 4.1 3.5    6.6 4.8 3.9
//   3072 x 768           8  4.3  3.9    9  4.9  4.7
//   768 x 3072          13  7.2  6.4    9  9.2  8.5
//   q, k, v 1600 x 1600 38  6.8  8.5   35  7.4  9.1
//   16384 x 4096        35 24   29     31 27   35 (5.5 and 4.7 TB/s of 1 row)
// so wide weights would gain by the layout's copies, which follow nothing.
//
// R blocks of 16 rows of W by B of x: R = 1, which is the most workgroups, while
// they are no more than the CUs or x is no longer than their part of W.
template <int R, int B, bool NORM>
__global__ __launch_bounds__(BLOCK, 2) void decode_affine_kernel(
    const uint16_t *__restrict__ xs, int M, int K, Affine a) {
  constexpr int U = R == 1 ? 8 : 4;
  extern __shared__ __attribute__((aligned(16))) uint16_t normed[];
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, i16 = lane & 15, grp = lane >> 4;
  // ends are multiples of 32: a workgroup's rows are of one matrix
  const int n0 = blockIdx.x * 16 * R;
  int first;
  const int of = matrix_of(a, n0, first);
  const uint16_t *w = a.w[of] + (int64_t)(n0 - first + i16) * K + grp * 8;
  const uint16_t *x = NORM ? normed + grp * M * 8
                           : xs + (grp >> 1) * 512 + (grp & 1) * 256;
  const int xstep = NORM ? M * 32 : 1024;
  int xrow[B];                          // rows past M: the last one again
#pragma unroll
  for (int b = 0; b < B; ++b) xrow[b] = min(b * 16 + i16, M - 1) * 8;
  const int steps = K / 32, s0 = steps * wid / 4, s1 = steps * (wid + 1) / 4;

  f32x4v acc[R][B];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int b = 0; b < B; ++b) acc[i][b] = (f32x4v)(0.0f);
  struct Chunk { bf16x8v w[U][R], x[U][B]; };
  Chunk c0, c1;
  auto load_w = [&](Chunk &c, int s) {  // past the end: the last one again
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < R; ++i)
        c.w[u][i] = load8v(w + (int64_t)i * 16 * K + min(s + u, s1 - 1) * 32);
  };
  auto load_x = [&](Chunk &c, int s) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int b = 0; b < B; ++b)
        c.x[u][b] = load8v(x + (int64_t)min(s + u, s1 - 1) * xstep + xrow[b]);
  };
  auto load = [&](Chunk &c, int s) {
    load_w(c, s);
    load_x(c, s);
  };
  auto multiply = [&](const Chunk &c, int s) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s1) {
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int b = 0; b < B; ++b)
            acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                c.w[u][i], c.x[u][b], acc[i][b], 0, 0, 0);
      }
  };
  if (s0 < s1) load_w(c0, s0);
  if constexpr (NORM) normed_operand(a, M, K, normed);
  if (s0 < s1) {
    int s = s0;
    load_x(c0, s);
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
  __shared__ float red[4][16 * R][16 * B + 1];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[wid][i * 16 + grp * 4 + r][b * 16 + i16] = acc[i][b][r];
  __syncthreads();
  constexpr int V = 2 * R;              // columns of a thread
  const int m = tid >> 3, en = (tid & 7) * V;
  if (m >= min(M, 16 * B)) return;
  const int n = n0 + en;
  float f[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    f[j] = red[0][en + j][m] + red[1][en + j][m] + red[2][en + j][m] +
           red[3][en + j][m];
    if (a.bias[of] != nullptr)
      f[j] += rb::bf16_to_f32(a.bias[of][n - first + j]);
    f[j] = activate(f[j], a.act);
  }
  if (a.into != nullptr) {
    float *dst = a.into + (int64_t)m * a.end[0] + n;
#pragma unroll
    for (int j = 0; j < V; ++j) dst[j] += f[j];
    return;
  }
  __attribute__((aligned(8))) uint16_t o[V];
#pragma unroll
  for (int j = 0; j < V; ++j) o[j] = rb::f32_to_bf16(f[j]);
  if (a.k_cache != nullptr && of > 0) {
    cache<V>(a, of == 2, m, n - first, o);
    return;
  }
  uint16_t *dst =
      a.operand ? a.out[0] + (n >> 4) * 512 + (n >> 3 & 1) * 256 + m * 8 +
                      (n & 7)
                : a.out[of] + (int64_t)m * (a.end[of] - first) + n - first;
  if constexpr (R == 1)
    *reinterpret_cast<uint32_t *>(dst) = *reinterpret_cast<uint32_t *>(o);
  else
    *reinterpret_cast<uint64_t *>(dst) = *reinterpret_cast<uint64_t *>(o);
}

// The same of up to 4 rows x [M, K] (or the norm of a residual): a wave takes R
// rows of W, its lanes 8 columns each of every 512, in dot products of pairs.
//
// Such a product is over when its first loads have come back. With matrix
// instructions a workgroup reads 15 rows of x that are not there, and its 16
// rows of W and as much of x keep one CU's loads busy for most of that time: 768 x
// 3072 takes 48 workgroups there, 192 here. us in a graph, there and here, of 1
// and 4 rows: 768 x 3072 6.4 3.3  6.6 4.1, 768 x 768 3.6 2.2  3.7 2.8; with the norm,
// 2304 x 768 5.6 4.1  5.4 5.3, 3072 x 768 5.3 3.8  5.3 5.3. From 5 rows it is even.
// Four rows of W a wave rather than two: 2304 x 768 of 4 rows 6.3 -> 5.3.
template <int M, int CH, int R, bool NORM>
__global__ __launch_bounds__(BLOCK, 2) void affine_few_kernel(
    const uint16_t *__restrict__ x, int K, Affine a) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = (blockIdx.x * (BLOCK / 64) + wid) * R;
  int first;
  const int of = matrix_of(a, n0, first);
  const uint16_t *w = a.w[of] + (int64_t)(n0 - first) * K;
  int c[CH];                            // past the end: the last ones again
#pragma unroll
  for (int j = 0; j < CH; ++j) c[j] = min(j * 512 + lane * 8, K - 8);
  uint4 wv[R][CH];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int j = 0; j < CH; ++j)
      wv[r][j] = *reinterpret_cast<const uint4 *>(w + (int64_t)r * K + c[j]);
  uint4 xv[M][CH];
  if constexpr (NORM) {
    const float inv_k = 1.0f / (float)K;
    float f[M][CH][8], sum[M], dev[M];
    uint4 gain[CH], shift[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        rb::VIO<float>::load(a.res + (int64_t)m * K + c[j], f[m][j]);
        rb::VIO<float>::load(a.res + (int64_t)m * K + c[j] + 4, f[m][j] + 4);
      }
      gain[j] = *reinterpret_cast<const uint4 *>(a.gain + c[j]);
      shift[j] = *reinterpret_cast<const uint4 *>(a.shift + c[j]);
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      sum[m] = 0.0f;
#pragma unroll
      for (int j = 0; j < CH; ++j)
        if (j * 512 + lane * 8 < K) {
#pragma unroll
          for (int i = 0; i < 8; ++i) sum[m] += f[m][j][i];
        }
    }
    rb::lane_sums<64>(sum);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float mean = sum[m] * inv_k;
      dev[m] = 0.0f;
#pragma unroll
      for (int j = 0; j < CH; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          f[m][j][i] -= mean;
          if (j * 512 + lane * 8 < K) dev[m] += f[m][j][i] * f[m][j][i];
        }
    }
    rb::lane_sums<64>(dev);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float inv = rsqrtf(dev[m] * inv_k + a.eps);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const uint32_t g[4] = {gain[j].x, gain[j].y, gain[j].z, gain[j].w};
        const uint32_t b[4] = {shift[j].x, shift[j].y, shift[j].z, shift[j].w};
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = pack2(
              f[m][j][2 * i] * inv * lower(g[i]) + lower(b[i]),
              f[m][j][2 * i + 1] * inv * upper(g[i]) + upper(b[i]));
        xv[m][j] = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int j = 0; j < CH; ++j)
        xv[m][j] =
            *reinterpret_cast<const uint4 *>(x + (int64_t)m * K + c[j]);
  }
  // what the lane that writes row m, column n0 + r adds, on its way meanwhile
  const int mine = min(lane, M * R - 1), m = mine / R, r = mine % R;
  const int n = n0 + r;
  const float add = a.bias[of] == nullptr
                        ? 0.0f : rb::bf16_to_f32(a.bias[of][n - first]);
  const float old =
      a.into == nullptr ? 0.0f : a.into[(int64_t)m * a.end[0] + n];
  float dot[M * R];
#pragma unroll
  for (int i = 0; i < M * R; ++i) {
    dot[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      if (j * 512 + lane * 8 >= K) continue;
      const uint4 u = wv[i % R][j], v = xv[i / R][j];
      dot[i] = dot2(u.x, v.x, dot[i]);
      dot[i] = dot2(u.y, v.y, dot[i]);
      dot[i] = dot2(u.z, v.z, dot[i]);
      dot[i] = dot2(u.w, v.w, dot[i]);
    }
  }
  rb::lane_sums<64>(dot);
  if (lane >= M * R) return;
  float f = dot[0];
#pragma unroll
  for (int i = 1; i < M * R; ++i) f = lane == i ? dot[i] : f;
  f = activate(f + add, a.act);
  if (a.into != nullptr) {
    a.into[(int64_t)m * a.end[0] + n] = old + f;
    return;
  }
  const uint16_t o = rb::f32_to_bf16(f);
  if (a.k_cache != nullptr && of > 0)
    cache<1>(a, of == 2, m, n - first, &o);
  else
    a.out[of][(int64_t)m * (a.end[of] - first) + n - first] = o;
}

// A row's embeddings of token and position, added up in fp32.
__global__ __launch_bounds__(BLOCK) void embed_res32_kernel(
    const int64_t *__restrict__ tokens, const int32_t *__restrict__ positions,
    const uint16_t *__restrict__ table, const uint16_t *__restrict__ places,
    float *__restrict__ res, int64_t words, int64_t longest, int D) {
  const int m = blockIdx.x;
  const int64_t t = tokens[m], p = positions[m];
  CUDA_KERNEL_ASSERT(t >= 0 && t < words && p >= 0 && p < longest);
  for (int c = threadIdx.x * 8; c < D; c += BLOCK * 8) {
    float f[8], g[8];
    rb::VIO<uint16_t>::load(table + t * D + c, f);
    rb::VIO<uint16_t>::load(places + p * D + c, g);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] += g[i];
    rb::VIO<float>::store(res + (int64_t)m * D + c, f);
    rb::VIO<float>::store(res + (int64_t)m * D + c + 4, f + 4);
  }
}

// Checks up to three parameters W [N_i, K] and their biases; returns all
// columns.
int64_t set_matrices(Affine &a, const std::vector<at::Tensor> &ws,
                     const std::vector<c10::optional<at::Tensor>> &biases,
                     at::Device device) {
  TORCH_CHECK(!ws.empty() && ws.size() <= 3 && biases.size() == ws.size(),
              "decode_affine: matrices");
  const int64_t K = ws[0].dim() == 2 ? ws[0].size(1) : 0;
  TORCH_CHECK(K > 0 && K % 32 == 0 && K < (1 << 24), "decode_affine: columns");
  int64_t N = 0;
  for (size_t i = 0; i < ws.size(); ++i) {
    const at::Tensor &w = ws[i];
    TORCH_CHECK(w.device() == device && w.dim() == 2 && w.size(1) == K &&
                w.size(0) > 0 && w.size(0) % 32 == 0 && w.is_contiguous() &&
                w.scalar_type() == at::kBFloat16 &&
                reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
                "decode_affine: weights [32 n, 32 k] bf16");
    const auto &b = biases[i];
    TORCH_CHECK(!b.has_value() ||
                (b->device() == device && b->is_contiguous() &&
                 b->numel() == w.size(0) &&
                 b->scalar_type() == at::kBFloat16), "decode_affine: bias");
    a.w[i] = (const uint16_t *)w.data_ptr();
    a.bias[i] = b.has_value() ? (const uint16_t *)b->data_ptr() : nullptr;
    N += w.size(0);
    TORCH_CHECK(N < (int64_t)1 << 31, "decode_affine: columns");
    a.end[i] = (int)N;
  }
  return N;
}

const uint16_t *operand_of(const at::Tensor &xs, int64_t K, at::Device device) {
  TORCH_CHECK(xs.is_cuda() && xs.device() == device && xs.is_contiguous() &&
              xs.scalar_type() == at::kBFloat16 &&
              xs.numel() == (K / 16) * 512, "decode_affine: operand");
  return (const uint16_t *)xs.data_ptr();
}

std::vector<at::Tensor> set_outputs(Affine &a, int64_t M, size_t n,
                                    bool operand, at::TensorOptions options) {
  std::vector<at::Tensor> out;
  a.operand = operand;
  for (size_t i = 0; i < n; ++i) {
    const int64_t N = a.end[i] - (i == 0 ? 0 : a.end[i - 1]);
    out.push_back(operand ? at::empty({N / 16 * 512}, options)
                          : at::empty({M, N}, options));
    a.out[i] = (uint16_t *)out[i].data_ptr();
  }
  return out;
}

void check_residual(const at::Tensor &res) {
  TORCH_CHECK(res.is_cuda() && res.dim() == 2 && res.is_contiguous() &&
              res.scalar_type() == at::kFloat && res.size(0) >= 1 &&
              res.size(0) <= MMAX && res.size(1) > 0 && res.size(1) % 32 == 0 &&
              reinterpret_cast<uintptr_t>(res.data_ptr()) % 16 == 0,
              "decode_affine: residual");
}

void launch(const Affine &a, const uint16_t *xs, int64_t M, int64_t N,
            int64_t K) {
  const bool norm = a.res != nullptr;
  auto go = [&](auto kernel, int rows) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(N / rows)), dim3(BLOCK),
                       norm ? M * K * 2 : 0, at::cuda::getCurrentHIPStream(),
                       xs, (int)M, (int)K, a);
  };
  if (norm)
    M <= 16 ? go(decode_affine_kernel<1, 1, true>, 16)
            : go(decode_affine_kernel<1, 2, true>, 16);
  else if (M <= 16) go(decode_affine_kernel<1, 1, false>, 16);
  else if (N <= 16 * 256) go(decode_affine_kernel<1, 2, false>, 16);
  else go(decode_affine_kernel<2, 2, false>, 32);
}

// affine_few_kernel: K up to 4096, 1024 with the norm. Four rows of W a wave
// where one would be more waves than the chip has at once.
bool few_supported(int64_t M, int64_t K) {
  return M >= 1 && M <= FEW && K % 8 == 0 && K <= 4096;
}
void launch_few(const Affine &a, const uint16_t *x, int64_t M, int64_t N,
                int64_t K) {
  auto go = [&](auto kernel, int rows) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(N / (rows * (BLOCK / 64)))),
                       dim3(BLOCK), 0, at::cuda::getCurrentHIPStream(), x,
                       (int)K, a);
  };
  auto rows = [&](auto m, auto ch, auto norm) {
    constexpr int MM = decltype(m)::value, CH = decltype(ch)::value;
    constexpr bool NORM = decltype(norm)::value;
    if (N >= 2048 && CH * MM <= 8)
      go(affine_few_kernel<MM, CH, CH * MM <= 8 ? 4 : 1, NORM>, 4);
    else
      go(affine_few_kernel<MM, CH, 1, NORM>, 1);
  };
  auto chunks = [&](auto m) {
    if (a.res != nullptr)
      rows(m, std::integral_constant<int, 2>{}, std::true_type{});
    else if (K <= 1024)
      rows(m, std::integral_constant<int, 2>{}, std::false_type{});
    else if (K <= 3072)
      rows(m, std::integral_constant<int, 6>{}, std::false_type{});
    else
      rows(m, std::integral_constant<int, 8>{}, std::false_type{});
  };
  // rows past M would be read: a kernel for each number of them
  switch (M) {
    case 1: return chunks(std::integral_constant<int, 1>{});
    case 2: return chunks(std::integral_constant<int, 2>{});
    case 3: return chunks(std::integral_constant<int, 3>{});
    default: chunks(std::integral_constant<int, 4>{});
  }
}

}  // namespace

// act(x W^T + bias) with up to three parameters W [N_i, K] and their biases, to a
// matrix each, or as the operand of the next product; xs as in decode_gemm.
std::vector<at::Tensor> decode_affine(
    at::Tensor xs, std::vector<at::Tensor> ws,
    std::vector<c10::optional<at::Tensor>> biases, int64_t M, int64_t act,
    bool operand) {
  TORCH_CHECK(M >= 1 && M <= MMAX && act >= 0 && act <= 3,
              "decode_affine: rows, act");
  Affine a{};
  const int64_t N = set_matrices(a, ws, biases, xs.device());
  const int64_t K = ws[0].size(1);
  const uint16_t *x = operand_of(xs, K, xs.device());
  TORCH_CHECK(!operand || ws.size() == 1, "decode_affine: matrices");
  auto out = set_outputs(a, M, ws.size(), operand, xs.options());
  a.act = (int)act;
  launch(a, x, M, N, K);
  return out;
}

// Rows and columns of a residual that a product's workgroups norm for themselves
// (an operand of up to 48 KB in LDS).
bool normed_affine_supported(int64_t M, int64_t K) {
  return M >= 1 && M <= MMAX && K > 0 && K % 32 == 0 && K <= WIDEST &&
         M * K <= 24576;
}

// Whether products of M rows read and write rows rather than operands.
bool affine_in_rows(int64_t M) { return M <= FEW; }

// decode_affine of the layer norm of a residual, a single result in rows or as an
// operand (affine_in_rows). With caches, of three matrices q, k and v the last two
// go there and q is the only result.
std::vector<at::Tensor> normed_affine(
    at::Tensor res, at::Tensor gain, at::Tensor shift, double eps,
    std::vector<at::Tensor> ws,
    std::vector<c10::optional<at::Tensor>> biases, int64_t act, bool operand,
    c10::optional<at::Tensor> k_cache, c10::optional<at::Tensor> v_cache,
    c10::optional<at::Tensor> slots) {
  check_residual(res);
  const int64_t M = res.size(0), K = res.size(1);
  TORCH_CHECK(act >= 0 && act <= 3 && normed_affine_supported(M, K),
              "normed_affine: rows, act");
  for (const at::Tensor &t : {gain, shift})
    TORCH_CHECK(t.device() == res.device() && t.is_contiguous() &&
                t.numel() == K && t.scalar_type() == at::kBFloat16 &&
                reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
                "normed_affine: norm");
  Affine a{};
  const int64_t N = set_matrices(a, ws, biases, res.device());
  TORCH_CHECK(ws[0].size(1) == K && (!operand || ws.size() == 1) &&
              !(operand && affine_in_rows(M)), "normed_affine: matrices");
  a.res = res.data_ptr<float>();
  a.gain = (const uint16_t *)gain.data_ptr();
  a.shift = (const uint16_t *)shift.data_ptr();
  a.eps = (float)eps;
  a.act = (int)act;
  size_t results = ws.size();
  if (k_cache.has_value()) {
    TORCH_CHECK(ws.size() == 3 && v_cache.has_value() && slots.has_value() &&
                k_cache->device() == res.device() &&
                v_cache->device() == res.device() &&
                slots->device() == res.device() && k_cache->dim() == 4 &&
                v_cache->dim() == 4 && k_cache->is_contiguous() &&
                v_cache->is_contiguous() &&
                k_cache->scalar_type() == at::kBFloat16 &&
                v_cache->scalar_type() == at::kBFloat16 &&
                v_cache->numel() == k_cache->numel() &&
                v_cache->size(1) == k_cache->size(1) &&
                slots->scalar_type() == at::kInt && slots->is_contiguous() &&
                slots->numel() >= M, "normed_affine: caches");
    a.hkv = (int)k_cache->size(1);
    a.bs = (int)k_cache->size(2);
    a.dh = (int)k_cache->size(3);
    TORCH_CHECK(a.dh > 0 && a.dh % 4 == 0 && a.bs > 0 &&
                ws[1].size(0) == (int64_t)a.hkv * a.dh &&
                ws[2].size(0) == ws[1].size(0) &&
                reinterpret_cast<uintptr_t>(k_cache->data_ptr()) % 8 == 0 &&
                reinterpret_cast<uintptr_t>(v_cache->data_ptr()) % 8 == 0,
                "normed_affine: cache sizes");
    a.vt = v_cache->size(3) == a.bs && v_cache->size(2) == a.dh &&
           a.dh != a.bs;
    a.k_cache = (uint16_t *)k_cache->data_ptr();
    a.v_cache = (uint16_t *)v_cache->data_ptr();
    a.slots = slots->data_ptr<int32_t>();
    results = 1;
  }
  auto out = set_outputs(a, M, results, operand,
                         res.options().dtype(at::kBFloat16));
  if (affine_in_rows(M)) launch_few(a, nullptr, M, N, K);
  else launch(a, nullptr, M, N, K);
  return out;
}

// res += x W^T + bias; x in rows [M, K] of up to 4096 columns or as an operand
// (affine_in_rows).
void affine_add_(at::Tensor x, at::Tensor w, c10::optional<at::Tensor> bias,
                 at::Tensor res) {
  check_residual(res);
  Affine a{};
  const int64_t N = set_matrices(a, {w}, {bias}, res.device());
  const int64_t M = res.size(0), K = w.size(1);
  TORCH_CHECK(res.size(1) == N, "affine_add_: columns");
  a.into = res.data_ptr<float>();
  if (x.dim() == 1) {
    launch(a, operand_of(x, K, res.device()), M, N, K);
    return;
  }
  TORCH_CHECK(x.device() == res.device() && x.dim() == 2 && x.size(0) == M &&
              x.size(1) == K && x.is_contiguous() &&
              x.scalar_type() == at::kBFloat16 && few_supported(M, K) &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "affine_add_: rows");
  launch_few(a, (const uint16_t *)x.data_ptr(), M, N, K);
}

// Residual [M, D] fp32 of tokens at positions.
at::Tensor embed_res32(at::Tensor tokens, at::Tensor positions,
                       at::Tensor table, at::Tensor places) {
  TORCH_CHECK(tokens.is_cuda() && tokens.dim() == 1 && tokens.is_contiguous() &&
              tokens.scalar_type() == at::kLong && positions.is_contiguous() &&
              positions.device() == tokens.device() &&
              positions.scalar_type() == at::kInt &&
              positions.numel() == tokens.numel(), "embed_res32: tokens");
  for (const at::Tensor &t : {table, places})
    TORCH_CHECK(t.device() == tokens.device() && t.dim() == 2 &&
                t.is_contiguous() && t.scalar_type() == at::kBFloat16 &&
                t.size(1) == table.size(1) &&
                reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
                "embed_res32: tables");
  const int64_t M = tokens.numel(), D = table.size(1);
  TORCH_CHECK(M >= 1 && D > 0 && D % 8 == 0 && D < (1 << 24),
              "embed_res32: sizes");
  auto res = at::empty({M, D}, table.options().dtype(at::kFloat));
  hipLaunchKernelGGL(embed_res32_kernel, dim3((unsigned)M), dim3(BLOCK), 0,
                     at::cuda::getCurrentHIPStream(),
                     tokens.data_ptr<int64_t>(), positions.data_ptr<int32_t>(),
                     (const uint16_t *)table.data_ptr(),
                     (const uint16_t *)places.data_ptr(),
                     res.data_ptr<float>(), table.size(0), places.size(0),
                     (int)D);
  return res;
}
