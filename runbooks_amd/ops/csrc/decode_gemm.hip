// Decode GEMM v2 for CDNA4 (gfx950): y[M,N] = x[M,K] @ W[N,K]^T,
// M <= 32 (decode batch; to 128 rows: decode_gemm_rows_kernel), bf16 in / bf16
// out, fp32 accumulate.
//
// The M<=32 decode GEMM is >99% W traffic, so the ONLY thing that
// matters is shaping the weight read as perfectly coalesced nontemporal
// bursts with enough in flight (MI355X ~6.3 TB/s achievable; hipBLASLt
// measured ~2.4 TB/s in the eager decode loop, and a fragment-shaped
// direct-load variant measured ~1.5 TB/s because every wave instruction
// became 32 scattered 32 B requests). This version therefore streams
// BOTH operands from layouts pre-swizzled into MFMA fragment-lane order:
//
//  * W is stored fragment-major at model-load time (decode_swizzle_w:
//    [N/32][K/16][lane][8] bf16) so each wave instruction is one 1 KiB
//    contiguous nontemporal read. 288 GB HBM3E per GPU makes the second
//    weight copy the right trade (same pattern as the fp8 registry);
//    prefill/training keep using the original [N,K] tensor via hipBLASLt.
//  * x (tiny: M*K <= 0.7 MB) is swizzled per call by decode_swizzle_x —
//    one extra ~microsecond kernel — into [K/16][lane][8] with zero
//    padding for m >= M; after that every wave reads the same contiguous
//    L2-resident stream.
//  * One wave owns 32 W rows x a DEEP contiguous k-range (K/(4*SPLIT)),
//    no LDS and no barrier in the main loop: a ring of two chunks in
//    registers.
//  * 4 waves per WG take adjacent k-quarters; one 16 KB LDS reduction
//    combines them. SPLIT (1 for N>=16k, 2-4 for N=4096 shapes) adds
//    fp32 slabs [SPLIT,M,N] reduced by a combine kernel (~1 MB next to
//    the 32-90 MB W stream).
//
// Fragment maps (v_mfma_f32_32x32x16_bf16, A=W so C cols = m):
//   A lane l -> A[row=l&31][k=(l>>5)*8+i];  B lane l -> B[k][col=l&31];
//   C lane l -> C[row=(r&3)+8*(r>>2)+4*(l>>5)][col=l&31], r = 0..15.
// The swizzles bake exactly these maps into the storage order.
//
// Reference parity: replaces hipBLASLt for the decode hot loop the way
// the reference's external server image leans on cuBLAS
// (substratusai/runbooks docs/container-contract.md serving contract).

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <type_traits>

#include "common.h"

namespace {

constexpr int BLOCK = 256;   // 4 waves
constexpr int MMAX = 32;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8v;
typedef __attribute__((ext_vector_type(16))) float f32x16v;
typedef __attribute__((ext_vector_type(4))) float f32x4v;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4v;

__device__ __forceinline__ bf16x8v load8v(const uint16_t *p) {
  union { u32x4v u; bf16x8v v; } c;
  c.u = *reinterpret_cast<const u32x4v *>(p);
  return c.v;
}

// Sums the four waves' accumulators of 32 rows of W and stores them, times the
// rows' scales where there are any: y, or a slice of the slabs.
template <bool STORE_BF16>
__device__ __forceinline__ void finish(const f32x16v &acc, const float *scale,
                                       uint16_t *yp, float *slabs, int M,
                                       int N) {
  const int tid = threadIdx.x, wid = tid >> 6;
  const int hi = (tid & 63) >> 5, col = tid & 31;
  const int nblk = blockIdx.x, kslice = blockIdx.y;
  __shared__ __attribute__((aligned(16))) float red[4][32][MMAX];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int n_local = (r & 3) + 8 * (r >> 2) + 4 * hi;
    red[wid][n_local][col] = acc[r];
  }
  __syncthreads();

  // 1024 outputs, 4 per thread, n fastest so bf16 stores coalesce 8 B.
  const int em = tid >> 3;               // 0..31
  const int en = (tid & 7) * 4;          // 0,4,..,28
  if (em < M) {
    float sum[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sum[j] = red[0][en + j][em] + red[1][en + j][em] +
               red[2][en + j][em] + red[3][en + j][em];
      if (scale != nullptr) sum[j] *= scale[nblk * 32 + en + j];
    }
    if (STORE_BF16) {
      union { uint16_t u[4]; uint64_t q; } o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o.u[j] = rb::f32_to_bf16(sum[j]);
      *reinterpret_cast<uint64_t *>(
          yp + (int64_t)em * N + nblk * 32 + en) = o.q;
    } else {
      float *slab = slabs + ((int64_t)kslice * M + em) * N + nblk * 32 + en;
      *reinterpret_cast<float4 *>(slab) =
          make_float4(sum[0], sum[1], sum[2], sum[3]);
    }
  }
}

// Two words of e4m3 -> 8 bf16 (exact).
__device__ __forceinline__ bf16x8v fp8_to_bf16(unsigned lo, unsigned up) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2v;
  union { bf16x2v h[4]; bf16x8v v; } c;
  c.h[0] = __builtin_convertvector(
      __builtin_amdgcn_cvt_pk_f32_fp8(lo, false), bf16x2v);
  c.h[1] = __builtin_convertvector(
      __builtin_amdgcn_cvt_pk_f32_fp8(lo, true), bf16x2v);
  c.h[2] = __builtin_convertvector(
      __builtin_amdgcn_cvt_pk_f32_fp8(up, false), bf16x2v);
  c.h[3] = __builtin_convertvector(
      __builtin_amdgcn_cvt_pk_f32_fp8(up, true), bf16x2v);
  return c.v;
}

// What a lane holds of a kilobyte of W: operands of 32 rows x 16 columns, or of
// 32 rows x 32 columns in e4m3 (decode_swizzle_w, decode_swizzle_w8).
template <bool FP8> struct Step {
  static constexpr int X = FP8 ? 2 : 1;  // operands of x that go with it
  u32x4v w;
  bf16x8v x[X];
};

// STORE_BF16: write y bf16 directly (SPLIT == 1). Otherwise store an
// fp32 slab slice at slabs + kslice*M*N for decode_gemm_combine.
//
// W nontemporal (streamed once, must not evict L2); x plain (re-read by every
// n-block: L2 is exactly where it wants to live). Columns past M read the last
// row again: their results are not stored, and x stays as short as it is.
// Loads run a chunk of U kilobytes ahead, without a branch among them (one
// makes the compiler wait for all of them); past a wave's range they read its
// last kilobyte again.
//
// Bound by the weight stream, and with 32 rows by x (as long as W, or twice as
// long as e4m3). us before -> now, weights out of cache, for N x K of
// 12288 x 4096, 22016 x 4096, 4096 x 4096 and 4096 x 11008:
//   bf16  1 row    23.1 -> 20.0  36.9 -> 32.3  8.9 -> 8.2  21.3 -> 17.3
//         16 rows  24.3 -> 22.5  37.5 -> 33.1  9.1 -> 8.6  21.6 -> 17.7
//         32 rows  23.5 -> 23.6  37.5 -> 38.3  9.3 -> 9.3  21.9 -> 20.2
//   e4m3 (before: tiles through LDS, a slab slice per 256 columns)
//         1 row    31.9 -> 13.8  47.3 -> 20.1  17.7 -> 6.3  39.5 -> 12.4
//         16 rows  32.5 -> 14.1  49.3 -> 20.8  17.7 -> 6.5  37.7 -> 12.8
//         32 rows  34.7 -> 17.7  56.5 -> 26.4  18.1 -> 7.7  38.1 -> 16.0
template <bool FP8>
__device__ __forceinline__ f32x16v weight_stream(
    const uint16_t *__restrict__ xs, const uint8_t *__restrict__ ws, int M,
    int K) {
  constexpr int X = Step<FP8>::X, U = FP8 ? 4 : 8;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int hi = lane >> 5, col = lane & 31;
  const int steps = K / (16 * X), groups = gridDim.y * 4;
  const int g = blockIdx.y * 4 + wid;
  const int s0 = (int)((int64_t)steps * g / groups);
  const int s1 = (int)((int64_t)steps * (g + 1) / groups);
  const uint8_t *wseg = ws + (int64_t)blockIdx.x * steps * 1024;
  const unsigned wlane = lane * 16;
  const unsigned xlane = (hi * 32 + min(col, M - 1)) * 8;

  f32x16v acc = (f32x16v)(0.0f);
  Step<FP8> a[U], b[U];
  auto load = [&](Step<FP8> (&c)[U], int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t at = min(s + u, s1 - 1);
      c[u].w = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4v *>(wseg + at * 1024 + wlane));
#pragma unroll
      for (int i = 0; i < X; ++i)
        c[u].x[i] = load8v(xs + (at * X + i) * 512 + xlane);
    }
  };
  auto multiply = [&](const Step<FP8> &c) {
    if constexpr (FP8) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          fp8_to_bf16(c.w[0], c.w[1]), c.x[0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          fp8_to_bf16(c.w[2], c.w[3]), c.x[1], acc, 0, 0, 0);
    } else {
      union { u32x4v u; bf16x8v v; } w;
      w.u = c.w;
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w.v, c.x[0], acc, 0, 0, 0);
    }
  };
  if (s0 < s1) {
    int s = s0;
    load(a, s);
    for (; s + 2 * U < s1; s += 2 * U) {
      load(b, s + U);
#pragma unroll
      for (int u = 0; u < U; ++u) multiply(a[u]);
      load(a, s + 2 * U);
#pragma unroll
      for (int u = 0; u < U; ++u) multiply(b[u]);
    }
    load(b, s + U);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s1) multiply(a[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + U + u < s1) multiply(b[u]);
  }
  return acc;
}

template <bool FP8, bool STORE_BF16>
__global__ __launch_bounds__(BLOCK, 1) void decode_gemm_kernel(
    const uint16_t *__restrict__ xs, const uint8_t *__restrict__ ws,
    const float *__restrict__ scale, uint16_t *__restrict__ yp,
    float *__restrict__ slabs, int M, int N, int K) {
  const f32x16v acc = weight_stream<FP8>(xs, ws, M, K);
  finish<STORE_BF16>(acc, scale, yp, slabs, M, N);
}

// act(x W^T + bias) of models whose decode is bound by its launches: the columns
// go to up to three matrices (q, k, v), or to the operand of the next product.
// W and bias are the parameters themselves, so that captured steps follow them
// too: a workgroup takes 16 rows of W as they lie, its waves parts of the sums,
// 64 bytes of each row an instruction (16x16x32 products: A[i=l&15][k=(l>>4)*8+e],
// B[k][j=l&15], C[j=l&15][i=(l>>4)*4+r]).
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
struct Affine {
  const uint16_t *w[3], *bias[3];       // [rows, K] each; bias may be null
  uint16_t *out[3];
  int end[3];                           // columns before the next matrix
  int act;                              // 0 none, 1 relu, 2 gelu, 3 gelu_tanh
  bool operand;                         // out[0] as [N/16][2][32][8]
};

__device__ __forceinline__ float activate(float x, int act) {
  if (act == 1) return x < 0.0f ? 0.0f : x;
  if (act == 2) return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
  if (act == 3)
    return 0.5f * x * (1.0f + tanhf(0.79788456080286536f *
                                    (x + 0.044715f * x * x * x)));
  return x;
}

// R blocks of 16 rows of W by B of x: R = 1, which is the most workgroups, while
// they are no more than the CUs or x is no longer than their part of W.
template <int R, int B>
__global__ __launch_bounds__(BLOCK, 2) void decode_affine_kernel(
    const uint16_t *__restrict__ xs, Affine a, int M, int K) {
  constexpr int U = R == 1 ? 8 : 4;
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, i16 = lane & 15, grp = lane >> 4;
  // ends are multiples of 32: a workgroup's rows are of one matrix
  const int n0 = blockIdx.x * 16 * R;
  const int of = n0 < a.end[0] ? 0 : n0 < a.end[1] ? 1 : 2;
  const int first = of == 0 ? 0 : a.end[of - 1];
  const uint16_t *w = a.w[of] + (int64_t)(n0 - first + i16) * K + grp * 8;
  const uint16_t *x = xs + (grp >> 1) * 512 + (grp & 1) * 256;
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
  auto load = [&](Chunk &c, int s) {    // past the end: the last one again
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = min(s + u, s1 - 1);
#pragma unroll
      for (int i = 0; i < R; ++i)
        c.w[u][i] = load8v(w + (int64_t)i * 16 * K + at * 32);
#pragma unroll
      for (int b = 0; b < B; ++b)
        c.x[u][b] = load8v(x + (int64_t)at * 1024 + xrow[b]);
    }
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
  __attribute__((aligned(8))) uint16_t o[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    float f = red[0][en + j][m] + red[1][en + j][m] + red[2][en + j][m] +
              red[3][en + j][m];
    if (a.bias[of] != nullptr)
      f += rb::bf16_to_f32(a.bias[of][n - first + j]);
    o[j] = rb::f32_to_bf16(activate(f, a.act));
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

// 17 to 128 rows (RB blocks of 32): x is longer than W's share of a workgroup, so
// NWN waves with blocks of 32 rows of W of their own share its tiles, in LDS, as
// they are in memory; 4 / NWN such groups take parts of the sums. A chunk is CH
// steps of 16 columns: W's next chunk and x's are on their way, in registers,
// during the products of this one. Pieces of 16 bytes of a tile's row r lie
// at their index ^ r, so that a column of 32 rows spreads over the banks.
// Rows past M, steps past the range: the last ones again; the former are not
// stored, the latter not multiplied.
//
// Bound by the weight stream (22016 x 4096 at 5 TB/s with 64 rows), with 128
// rows by the tiles of x (3.8 TB/s). W two chunks ahead and a chunk's operands
// of x read at once: 22016 x 4096 of 45 rows 40.6 -> 34.0 us, 4096 x 4096 15.0 ->
// 13.5 (library 43 and 23).
template <int RB, int NWN, int CH, bool STORE_BF16>
__global__ __launch_bounds__(BLOCK, 2) void decode_gemm_rows_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ ws,
    uint16_t *__restrict__ yp, float *__restrict__ slabs, int M, int N, int K) {
  constexpr int KG = 4 / NWN, P = 2 * CH;          // pieces of a row
  constexpr int XL = RB * CH / NWN;                // of x, a lane and chunk
  constexpr int TILE = RB * 32 * P * 16;
  static_assert(XL * NWN == RB * CH && (KG == 1 || 2 * KG * TILE >= NWN * RB * 4096),
                "tiles");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, hi = lane >> 5, col = lane & 31;
  const int wn = wid % NWN, kg = wid / NWN;
  const int blocks = N / 32, nblk = blockIdx.x * NWN + wn;
  const int steps = K / 16, groups = gridDim.y * KG;
  const int g = blockIdx.y * KG + kg;
  const int s0 = (int)((int64_t)steps * g / groups);
  const int s1 = (int)((int64_t)steps * (g + 1) / groups);
  const int full = steps / groups / CH;            // chunks of every group
  const int chunks = ((steps + groups - 1) / groups + CH - 1) / CH;
  const uint8_t *wseg =
      ws + (int64_t)min(nblk, blocks - 1) * steps * 1024 + lane * 16;
  char *mine = smem + kg * TILE;                   // buffers KG * TILE apart

  struct X { u32x4v v[XL]; };
  struct W { u32x4v v[CH]; };
  int64_t xrow[XL];                                // where a lane's pieces begin
  int xstep[XL], xput[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int p = (i * NWN + wn) * 64 + lane, row = p / P, c = p % P;
    xrow[i] = (int64_t)min(row, M - 1) * K + (c & 1) * 8;
    xstep[i] = c / 2;
    xput[i] = (row * P + (c ^ (row & (P - 1)))) * 16;
  }
  auto load_x = [&](X &d, int s) {
#pragma unroll
    for (int i = 0; i < XL; ++i)
      d.v[i] = *reinterpret_cast<const u32x4v *>(
          x + xrow[i] + min(s + xstep[i], s1 - 1) * 16);
  };
  auto load_w = [&](W &d, int s) {
#pragma unroll
    for (int u = 0; u < CH; ++u)
      d.v[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4v *>(
          wseg + (int64_t)min(s + u, s1 - 1) * 1024));
  };
  auto put_x = [&](const X &d, char *tile) {
#pragma unroll
    for (int i = 0; i < XL; ++i)
      *reinterpret_cast<u32x4v *>(tile + xput[i]) = d.v[i];
  };
  auto meet = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  f32x16v acc[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) acc[b] = (f32x16v)(0.0f);
  auto read = [&](bf16x8v (&xv)[RB], const char *tile, int u) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int row = b * 32 + col, c = u * 2 + hi;
      xv[b] = *reinterpret_cast<const bf16x8v *>(
          tile + (row * P + (c ^ (row & (P - 1)))) * 16);
    }
  };
  X xr;
  W w0, w1;
  load_x(xr, s0);
  load_w(w0, s0);
  put_x(xr, mine);
  load_x(xr, s0 + CH);
  load_w(w1, s0 + CH);
  meet();
  // chunk c, of which `w` holds W and then W of chunk c + 2
  auto step = [&](W &w, int c, auto whole) {
    const int s = s0 + c * CH;
    put_x(xr, mine + (~c & 1) * KG * TILE);
    load_x(xr, s + 2 * CH);
    const char *tile = mine + (c & 1) * KG * TILE;
    bf16x8v xv[CH][RB];
#pragma unroll
    for (int u = 0; u < CH; ++u) read(xv[u], tile, u);
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      union { u32x4v u; bf16x8v v; } a;
      a.u = w.v[u];
      if (whole || s + u < s1) {
#pragma unroll
        for (int b = 0; b < RB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, xv[u][b],
                                                           acc[b], 0, 0, 0);
      }
      w.v[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4v *>(
          wseg + (int64_t)min(s + 2 * CH + u, s1 - 1) * 1024));
    }
    meet();
  };
  int c = 0;
  for (; c + 2 <= full; c += 2) {
    step(w0, c, std::true_type{});
    step(w1, c + 1, std::true_type{});
  }
  for (; c < chunks; c += 2) {
    step(w0, c, std::false_type{});
    step(w1, c + 1, std::false_type{});
  }
  // sum of the groups
  if constexpr (KG == 2) {
    float *red = reinterpret_cast<float *>(smem) + wn * RB * 1024 + lane;
    if (kg == 1) {
#pragma unroll
      for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[(b * 16 + r) * 64] = acc[b][r];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][r] += red[(b * 16 + r) * 64];
  }
  if (nblk >= blocks) return;
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const int m = b * 32 + col;
    if (m >= M) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = nblk * 32 + 8 * q + 4 * hi;
      if (STORE_BF16) {
        union { uint16_t u[4]; uint64_t q; } o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o.u[j] = rb::f32_to_bf16(acc[b][4 * q + j]);
        *reinterpret_cast<uint64_t *>(yp + (int64_t)m * N + n) = o.q;
      } else {
        *reinterpret_cast<float4 *>(
            slabs + ((int64_t)blockIdx.y * M + m) * N + n) =
            make_float4(acc[b][4 * q], acc[b][4 * q + 1], acc[b][4 * q + 2],
                        acc[b][4 * q + 3]);
      }
    }
  }
}

// slabs [SPLIT, M, N] f32 -> y [M, N] bf16
__global__ void decode_gemm_combine_kernel(
    const float *__restrict__ slabs, uint16_t *__restrict__ yp,
    int split, int64_t mn) {
  const int64_t i0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x * 4;
  for (int64_t i = i0; i < mn; i += stride) {
    float4 s = *reinterpret_cast<const float4 *>(slabs + i);
    for (int k = 1; k < split; ++k) {
      float4 t = *reinterpret_cast<const float4 *>(slabs + (int64_t)k * mn + i);
      s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
    }
    union { uint16_t u[4]; uint64_t q; } o;
    o.u[0] = rb::f32_to_bf16(s.x); o.u[1] = rb::f32_to_bf16(s.y);
    o.u[2] = rb::f32_to_bf16(s.z); o.u[3] = rb::f32_to_bf16(s.w);
    *reinterpret_cast<uint64_t *>(yp + i) = o.q;
  }
}

// x [M, K] row-major -> xs [K/16][64 lanes][8] bf16 (B-fragment lane
// order: lane = hi*32 + m, elems = x[m][s*16 + hi*8 + i]; zeros for
// m >= M). One scattered read pass of <= 0.7 MB, coalesced writes.
__global__ void decode_swizzle_x_kernel(
    const uint16_t *__restrict__ xp, uint16_t *__restrict__ xs,
    int M, int K) {
  const int steps = K / 16;
  const int64_t total = (int64_t)steps * 64;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
       idx < total; idx += stride) {
    const int s = (int)(idx >> 6);
    const int l = (int)(idx & 63);
    const int m = l & 31;
    const int hi = l >> 5;
    rb::bf16x8 v;
    if (m < M) {
      v = *reinterpret_cast<const rb::bf16x8 *>(
          xp + (int64_t)m * K + s * 16 + hi * 8);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v.v[e] = 0;
    }
    *reinterpret_cast<rb::bf16x8 *>(xs + idx * 8) = v;
  }
}

}  // namespace

// Pick the cross-WG k-split by LOAD BALANCE: the kernel is a pure
// weight stream, so wall time = (WG waves over the 256 CUs) = ceil(
// nWG/256) rounds, and utilization = nWG / (256 * rounds).
// A microbench tracks this exactly: 384 WGs -> 75% -> 4.2 TB/s,
// 688 -> 90% -> 4.7, 1000 -> 98% -> 5.2. Score each legal split and
// keep the best; ties go to fewer splits (a split adds a slab round
// trip + combine kernel ~5-6 us inside the captured graph).
int64_t decode_gemm_split(int64_t N, int64_t K) {
  // Split only when the grid cannot cover the 256 CUs (o_proj/down_proj
  // N=4096 -> 128 WGs). Measured: splitting an already-covering
  // grid loses (gateup 688 WGs split 4: -10%; qkv 384 split 2 gained
  // ~2% on the kernel but pays a combine launch inside the graph).
  const int64_t nblocks = N / 32;
  int64_t split = 1;
  while (split < 8 && nblocks * split < 256 &&
         (K / 16) % (split * 4) == 0 && K / (split * 2) >= 1024) {
    split *= 2;
  }
  return split;
}

bool decode_gemm_supported(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= MMAX && N % 32 == 0 && K % 16 == 0 && K >= 1024;
}

// One-time weight swizzle (host-side tensor ops): [N,K] ->
// [N/32][K/16][2][32][8] = fragment-lane-major chunks of 1 KiB.
at::Tensor decode_swizzle_w(at::Tensor w) {
  TORCH_CHECK(w.dim() == 2 && w.scalar_type() == at::kBFloat16 &&
              w.is_contiguous(), "decode_swizzle_w: contiguous bf16 [N,K]");
  const int64_t N = w.size(0), K = w.size(1);
  TORCH_CHECK(N % 32 == 0 && K % 16 == 0, "decode_swizzle_w: shape");
  return w.view({N / 32, 32, K / 16, 2, 8})
      .permute({0, 2, 3, 1, 4}).contiguous();
}

at::Tensor decode_swizzle_x(at::Tensor x) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() &&
              x.scalar_type() == at::kBFloat16, "decode_swizzle_x: x");
  const int M = x.size(0), K = x.size(1);
  TORCH_CHECK(M <= MMAX && K % 16 == 0, "decode_swizzle_x: shape");
  auto xs = at::empty({(int64_t)(K / 16) * 512}, x.options());
  auto stream = at::cuda::getCurrentHIPStream();
  const int grid = rb::rb_grid_1d((int64_t)(K / 16) * 64, 256);
  hipLaunchKernelGGL(decode_swizzle_x_kernel, dim3(grid), dim3(256), 0,
                     stream, (const uint16_t *)x.data_ptr(),
                     (uint16_t *)xs.data_ptr(), M, K);
  return xs;
}

// e4m3 bytes [N,K] -> [N/32][K/32][2][32][2][8]: a lane's 16 bytes are its
// operands of two steps of 16 columns.
at::Tensor decode_swizzle_w8(at::Tensor w8) {
  TORCH_CHECK(w8.dim() == 2 && w8.scalar_type() == at::kByte &&
              w8.is_contiguous(), "decode_swizzle_w8: contiguous bytes [N,K]");
  const int64_t N = w8.size(0), K = w8.size(1);
  TORCH_CHECK(N % 32 == 0 && K % 32 == 0, "decode_swizzle_w8: shape");
  return w8.view({N / 32, 32, K / 32, 2, 2, 8})
      .permute({0, 2, 4, 1, 3, 5}).contiguous();
}

// Raw variant for fused consumers: split == 1 returns y bf16 [M, N] (with
// f32 a slab of one slice); split > 1 returns the fp32 slab [split, M, N]
// UNCOMBINED — the consumer kernel (rmsnorm_res_slab_fwd_dec) folds the
// slices while it reads, saving the combine launch inside the decode graph.
template <bool FP8>
static void launch(const at::Tensor &xs, const at::Tensor &ws,
                   const float *scale, at::Tensor *y, at::Tensor *slabs,
                   int split, int64_t M, int64_t N, int64_t K) {
  const dim3 grid((unsigned)(N / 32), (unsigned)split);
  auto stream = at::cuda::getCurrentHIPStream();
  if (slabs == nullptr)
    hipLaunchKernelGGL((decode_gemm_kernel<FP8, true>), grid, dim3(BLOCK), 0,
                       stream, (const uint16_t *)xs.data_ptr(),
                       (const uint8_t *)ws.data_ptr(), scale,
                       (uint16_t *)y->data_ptr(), nullptr, (int)M, (int)N,
                       (int)K);
  else
    hipLaunchKernelGGL((decode_gemm_kernel<FP8, false>), grid, dim3(BLOCK), 0,
                       stream, (const uint16_t *)xs.data_ptr(),
                       (const uint8_t *)ws.data_ptr(), scale, nullptr,
                       slabs->data_ptr<float>(), (int)M, (int)N, (int)K);
}

static void combine(const at::Tensor &slabs, at::Tensor &y) {
  hipLaunchKernelGGL(decode_gemm_combine_kernel,
                     dim3(rb::rb_grid_1d(y.numel() / 4, 256)), dim3(256), 0,
                     at::cuda::getCurrentHIPStream(),
                     slabs.data_ptr<float>(), (uint16_t *)y.data_ptr(),
                     (int)slabs.size(0), y.numel());
}

// act(x W^T + bias) with up to three parameters W [N_i, K] and their biases, to a
// matrix each, or as the operand of the next product; xs as in decode_gemm.
std::vector<at::Tensor> decode_affine(
    at::Tensor xs, std::vector<at::Tensor> ws,
    std::vector<c10::optional<at::Tensor>> biases, int64_t M, int64_t act,
    bool operand) {
  TORCH_CHECK(!ws.empty() && ws.size() <= 3 && biases.size() == ws.size() &&
              (!operand || ws.size() == 1), "decode_affine: matrices");
  TORCH_CHECK(M >= 1 && M <= MMAX && act >= 0 && act <= 3,
              "decode_affine: rows, act");
  const int64_t K = ws[0].dim() == 2 ? ws[0].size(1) : 0;
  TORCH_CHECK(K > 0 && K % 32 == 0 && K < (1 << 24) && xs.is_cuda() &&
              xs.is_contiguous() && xs.scalar_type() == at::kBFloat16 &&
              xs.numel() == (K / 16) * 512, "decode_affine: operand");
  Affine a{};
  int64_t N = 0;
  std::vector<at::Tensor> out;
  for (size_t i = 0; i < ws.size(); ++i) {
    const at::Tensor &w = ws[i];
    TORCH_CHECK(w.device() == xs.device() && w.dim() == 2 && w.size(1) == K &&
                w.size(0) > 0 && w.size(0) % 32 == 0 && w.is_contiguous() &&
                w.scalar_type() == at::kBFloat16 &&
                reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
                "decode_affine: weights [32 n, 32 k] bf16");
    const auto &b = biases[i];
    TORCH_CHECK(!b.has_value() ||
                (b->device() == xs.device() && b->is_contiguous() &&
                 b->numel() == w.size(0) &&
                 b->scalar_type() == at::kBFloat16), "decode_affine: bias");
    out.push_back(operand ? at::empty({w.size(0) / 16 * 512}, xs.options())
                          : at::empty({M, w.size(0)}, xs.options()));
    a.w[i] = (const uint16_t *)w.data_ptr();
    a.bias[i] = b.has_value() ? (const uint16_t *)b->data_ptr() : nullptr;
    a.out[i] = (uint16_t *)out[i].data_ptr();
    N += w.size(0);
    TORCH_CHECK(N < (int64_t)1 << 31, "decode_affine: columns");
    a.end[i] = (int)N;
  }
  a.act = (int)act;
  a.operand = operand;
  auto go = [&](auto kernel, int rows) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(N / rows)), dim3(BLOCK), 0,
                       at::cuda::getCurrentHIPStream(),
                       (const uint16_t *)xs.data_ptr(), a, (int)M, (int)K);
  };
  if (M <= 16) go(decode_affine_kernel<1, 1>, 16);
  else if (N <= 16 * 256) go(decode_affine_kernel<1, 2>, 16);
  else go(decode_affine_kernel<2, 2>, 32);
  return out;
}

// Sum of fp32 parts [P, M, N], rounded to bf16.
at::Tensor sum_parts(at::Tensor parts) {
  TORCH_CHECK(parts.is_cuda() && parts.dim() == 3 && parts.is_contiguous() &&
              parts.scalar_type() == at::kFloat && parts.size(2) % 4 == 0 &&
              parts.size(0) > 0 &&
              reinterpret_cast<uintptr_t>(parts.data_ptr()) % 16 == 0,
              "sum_parts: fp32 [P, M, 4 n]");
  auto y = at::empty({parts.size(1), parts.size(2)},
                     parts.options().dtype(at::kBFloat16));
  if (y.numel() > 0) combine(parts, y);
  return y;
}

at::Tensor decode_gemm_raw(at::Tensor xs, at::Tensor ws, int64_t M,
                           int64_t N, int64_t K, bool f32) {
  TORCH_CHECK(xs.is_cuda() && ws.is_cuda() && xs.is_contiguous() &&
              ws.is_contiguous() && xs.scalar_type() == at::kBFloat16 &&
              ws.scalar_type() == at::kBFloat16, "decode_gemm_raw: inputs");
  TORCH_CHECK(xs.numel() == (K / 16) * 512 && ws.numel() == N * K &&
              decode_gemm_supported(M, N, K), "decode_gemm_raw: shape");
  const int split = (int)decode_gemm_split(N, K);
  if (split == 1 && !f32) {
    auto y = at::empty({M, N}, xs.options());
    launch<false>(xs, ws, nullptr, &y, nullptr, 1, M, N, K);
    return y;
  }
  auto slabs = at::empty({split, M, N}, xs.options().dtype(at::kFloat));
  launch<false>(xs, ws, nullptr, nullptr, &slabs, split, M, N, K);
  return slabs;
}

// xs from decode_swizzle_x, ws from decode_swizzle_w; M/N/K of the
// ORIGINAL y[M,N] = x[M,K] @ W[N,K]^T problem.
at::Tensor decode_gemm(at::Tensor xs, at::Tensor ws, int64_t M, int64_t N,
                       int64_t K, int64_t force_split) {
  TORCH_CHECK(xs.is_cuda() && ws.is_cuda() && xs.is_contiguous() &&
              ws.is_contiguous(), "decode_gemm: contiguous GPU tensors");
  TORCH_CHECK(xs.scalar_type() == at::kBFloat16 &&
              ws.scalar_type() == at::kBFloat16, "decode_gemm: bf16 only");
  TORCH_CHECK(xs.numel() == (K / 16) * 512, "decode_gemm: xs size");
  TORCH_CHECK(ws.numel() == N * K, "decode_gemm: ws size");
  TORCH_CHECK(decode_gemm_supported(M, N, K),
              "decode_gemm: unsupported shape ", M, "x", N, "x", K);

  auto y = at::empty({M, N}, xs.options());
  const int split = force_split > 0 ? (int)force_split
                                    : (int)decode_gemm_split(N, K);
  if (split == 1) {
    launch<false>(xs, ws, nullptr, &y, nullptr, 1, M, N, K);
    return y;
  }
  auto slabs = at::empty({split, M, N}, xs.options().dtype(at::kFloat));
  launch<false>(xs, ws, nullptr, nullptr, &slabs, split, M, N, K);
  combine(slabs, y);
  return y;
}

// The product with e4m3 weights (decode_swizzle_w8) and a scale per row:
// y [M, N] bf16, or with raw=true, where it is split, the uncombined fp32
// slabs [split, M, N].
at::Tensor decode_gemm_fp8(at::Tensor xs, at::Tensor w8s, at::Tensor scale,
                           int64_t M, int64_t N, int64_t K, bool raw) {
  TORCH_CHECK(xs.is_cuda() && w8s.is_cuda() && scale.is_cuda() &&
              xs.is_contiguous() && w8s.is_contiguous() &&
              scale.is_contiguous() && xs.scalar_type() == at::kBFloat16 &&
              w8s.scalar_type() == at::kByte &&
              scale.scalar_type() == at::kFloat, "decode_gemm_fp8: inputs");
  TORCH_CHECK(M >= 1 && M <= MMAX && N % 32 == 0 && K % 32 == 0 && K > 0 &&
              xs.numel() == (K / 16) * 512 && w8s.numel() == N * K &&
              scale.numel() == N, "decode_gemm_fp8: shape");
  const int split = (int)decode_gemm_split(N, K);
  auto y = split > 1 && raw ? at::Tensor() : at::empty({M, N}, xs.options());
  if (split == 1) {
    if (N > 0)
      launch<true>(xs, w8s, scale.data_ptr<float>(), &y, nullptr, 1, M, N, K);
    return y;
  }
  auto slabs = at::empty({split, M, N}, xs.options().dtype(at::kFloat));
  launch<true>(xs, w8s, scale.data_ptr<float>(), nullptr, &slabs, split, M, N,
               K);
  if (raw) return slabs;
  combine(slabs, y);
  return y;
}

template <int RB, int NWN, int CH>
static void launch_rows(const at::Tensor &x, const at::Tensor &ws, at::Tensor &y,
                        int split) {
  const int64_t M = x.size(0), K = x.size(1), N = y.size(1);
  constexpr int lds = 2 * (4 / NWN) * RB * 32 * CH * 32;
  static_assert(lds <= 64 * 1024, "tiles");
  TORCH_CHECK(split >= 1 && split * (4 / NWN) <= K / 16, "decode_gemm_rows");
  const dim3 grid((unsigned)((N / 32 + NWN - 1) / NWN), (unsigned)split);
  auto go = [&](auto kernel, float *slabs) {
    hipLaunchKernelGGL(kernel, grid, dim3(BLOCK), lds,
                       at::cuda::getCurrentHIPStream(),
                       (const uint16_t *)x.data_ptr(),
                       (const uint8_t *)ws.data_ptr(),
                       (uint16_t *)y.data_ptr(), slabs, (int)M, (int)N, (int)K);
  };
  if (split == 1) {
    go(decode_gemm_rows_kernel<RB, NWN, CH, true>, nullptr);
    return;
  }
  auto slabs = at::empty({split, M, N}, x.options().dtype(at::kFloat));
  go(decode_gemm_rows_kernel<RB, NWN, CH, false>, slabs.data_ptr<float>());
  combine(slabs, y);
}

// y [M, N] = x [M, K] W^T of 1 to 128 rows; ws from decode_swizzle_w.
//
// One workgroup for every CU where it can be had, as a second on some of them
// has the others wait: four blocks of W for wide weights, unsplit; else two, or
// four for long rows, of which splits to fill the CUs cost less (us with two
// and four at their best split: 4096 x 11008 of 64 rows 25 and 26, of 100 rows
// 32 and 30; 3072 x 24576 38 and 34, 50 and 41; 4096 x 4096 14 and 16, 17 and
// 20; 22016 x 4096 of 64 rows 45 and 36, 12288 x 4096 25 and 26).
at::Tensor decode_gemm_rows(at::Tensor x, at::Tensor ws, int64_t N) {
  TORCH_CHECK(x.is_cuda() && ws.is_cuda() && x.dim() == 2 &&
              x.is_contiguous() && ws.is_contiguous() &&
              x.scalar_type() == at::kBFloat16 &&
              ws.scalar_type() == at::kBFloat16 &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "decode_gemm_rows: inputs");
  const int64_t M = x.size(0), K = x.size(1);
  TORCH_CHECK(M >= 1 && M <= 128 && N > 0 && N % 32 == 0 && K % 16 == 0 &&
              K >= 1024 && K < (1 << 24) && ws.numel() == N * K,
              "decode_gemm_rows: shape");
  auto y = at::empty({M, N}, x.options());
  const bool four = N >= 20480 || K >= (M <= 64 ? 20480 : 8192);
  const int64_t wgs = (N / 32 + (four ? 3 : 1)) / (four ? 4 : 2);
  int split = 1;
  while (split < 8 && wgs * split * 2 <= 256 && K / (split * 2) >= 256)
    split *= 2;
  auto go = [&](auto rb) {
    constexpr int RB = decltype(rb)::value;
    if (four) launch_rows<RB, 4, RB == 4 ? 4 : 8>(x, ws, y, split);
    else launch_rows<RB, 2, 4>(x, ws, y, split);
  };
  if (M <= 32) go(std::integral_constant<int, 1>{});
  else if (M <= 64) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
  return y;
}
