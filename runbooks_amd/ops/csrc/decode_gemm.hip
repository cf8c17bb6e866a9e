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
#include "decode_ends.h"

namespace {

constexpr int BLOCK = 256;   // 4 waves
constexpr int MMAX = 32;

using ends::bf16x8v;
using ends::Ends;
using ends::f32x16v;
using ends::f32x4v;
using ends::fp8_to_bf16;
using ends::Kind;
using ends::load8v;
using ends::u32x4v;

// What a thread needs for its ends besides the sums; issued before the stream
// of W (begin) and behind its first loads (rest), so that their ways to memory
// lie beside its own. A thread's row m is that of its place in finish(); waves that
// have none there, of up to 16 rows, need nothing (`mine`).
template <Kind KIND> struct Early {
  static constexpr int PARTS = 8;       // of 4 squares, for up to 256 in all
  float4 squares[PARTS];
  float norm;
  float scale[4];                       // of the rows of W in finish()
  int position;
  ends::Turn<2> turn;
  RB_DEV static bool mine(int M) {
    return (__builtin_amdgcn_readfirstlane(threadIdx.x) >> 3) < M;
  }
  RB_DEV void begin(const Ends &e, int M, int base = 0) {
    const int m = min(base + ((int)threadIdx.x >> 3), M - 1);
    const int i = threadIdx.x & 7;
    if constexpr (KIND == ends::QKV) position = e.pos[m];
    if (KIND != ends::SLAB && e.squares != nullptr) {
#pragma unroll
      for (int j = 0; j < PARTS; ++j)
        squares[j] = *reinterpret_cast<const float4 *>(
            e.squares + (int64_t)m * e.parts +
            min((j * 8 + i) * 4, e.parts - 4));
    }
  }
  RB_DEV void begin_scale(const Ends &e) {
    constexpr bool PAIRS = KIND == ends::GLU || KIND == ends::QKV;
    const int c = (threadIdx.x & 7) * (PAIRS ? 2 : 4);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      scale[j] = e.scale[ends::column(
          e.half, blockIdx.x, PAIRS ? c + (j & 1) + (j >> 1) * 16 : c + j)];
  }
  RB_DEV void rest(const Ends &e, int M) {
    const int m = min((int)threadIdx.x >> 3, M - 1), i = threadIdx.x & 7;
    norm = 1.0f;
    if (KIND != ends::SLAB && e.squares != nullptr) {
      float ss = 0.0f;
#pragma unroll
      for (int j = 0; j < PARTS; ++j)
        if ((j * 8 + i) * 4 < e.parts)
          ss += (squares[j].x + squares[j].y) + (squares[j].z + squares[j].w);
#pragma unroll
      for (int off = 4; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
      norm = rsqrtf(ss * e.inv_d + e.eps);
    }
    if constexpr (KIND == ends::QKV)
      turn.load(e, m, blockIdx.x * 16 + i * 2, position);
  }
};

// Sums the four waves' parts of 32 rows of W, red[wave][row][m], times the rows'
// scales where there are any (FP8), and hands them on.
template <bool FP8, Kind KIND, int RED>
__device__ __forceinline__ void finish(const float (&red)[4][32][RED],
                                       const Ends &e, const Early<KIND> &early,
                                       int M, int N) {
  const int tid = threadIdx.x;
  const int nblk = blockIdx.x;
  __syncthreads();

  // 1024 outputs, 4 per thread, n fastest so bf16 stores coalesce 8 B.
  const int em = tid >> 3;               // 0..31
  if (em >= M) return;
  auto sum = [&](int r, int j) {
    float x = red[0][r][em] + red[1][r][em] + red[2][r][em] + red[3][r][em];
    if (KIND != ends::SLAB) x *= early.norm;
    if (FP8) x *= early.scale[j];
    return x;
  };
  if constexpr (KIND == ends::GLU || KIND == ends::QKV) {
    const int c = (tid & 7) * 2;
    float a[2] = {sum(c, 0), sum(c + 1, 1)};
    float b[2] = {sum(16 + c, 2), sum(17 + c, 3)};
    if constexpr (KIND == ends::GLU)
      ends::put_gated<2>(e, em, nblk * 16 + c, N, a, b);
    else
      ends::put_heads<2>(e, early.turn, em, nblk * 16 + c, N, a, b);
  } else {
    const int en = (tid & 7) * 4;        // 0,4,..,28
    const int n = ends::column(e.half, nblk, en);
    const float f[4] = {sum(en, 0), sum(en + 1, 1), sum(en + 2, 2),
                        sum(en + 3, 3)};
    if constexpr (KIND == ends::PLAIN) {
      ends::put<4>(e.y + (int64_t)em * N + n, f);
    } else {
      float *slab = e.slabs + ((int64_t)blockIdx.y * M + em) * N + n;
      *reinterpret_cast<float4 *>(slab) = make_float4(f[0], f[1], f[2], f[3]);
    }
  }
}

// What a lane holds of a kilobyte of W: operands of 32 rows x 16 columns, or of
// 32 rows x 32 columns in e4m3 (decode_swizzle_w, decode_swizzle_w8).
template <bool FP8> struct Step {
  static constexpr int X = FP8 ? 2 : 1;  // operands of x that go with it
  u32x4v w;
  bf16x8v x[X];
};

// Steps s0 .. s1 - 1 by two chunks of U in turn.
//
// BOTH: both are on their way before `meanwhile` waits for anything, and what is past
// the end is not loaded behind the first two; of 17 to 32 rows, whose chunks are long,
// that costs 1 to 3%. APART: loads and products stay in this order. Left to itself the
// compiler puts the loads of the loop behind all of its products, so that none is on
// its way meanwhile.
template <bool BOTH, bool APART, int U, typename Step, typename Load,
          typename Multiply, typename Meanwhile>
__device__ __forceinline__ void stream_chunks(Step (&a)[U], Step (&b)[U],
                                              int s0, int s1, Load load,
                                              Multiply multiply,
                                              Meanwhile meanwhile) {
  auto apart = [] {
    if (APART) __builtin_amdgcn_sched_barrier(0);
  };
  auto up_to_end = [&](Step (&c)[U], int s) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < s1) multiply(c[u]);
  };
  if (s0 < s1) {
    load(a, s0);
    if (BOTH) load(b, s0 + U);
  }
  meanwhile();
  if (s0 >= s1) return;
  int s = s0;
  for (; s + (BOTH ? 3 : 2) * U < s1; s += 2 * U) {
    if (!BOTH) load(b, s + U);
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(a[u]);
    apart();
    load(a, s + 2 * U);
    apart();
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(b[u]);
    apart();
    if (BOTH) load(b, s + 3 * U);
    apart();
  }
  if (BOTH && s + 2 * U < s1) {                    // three chunks are left
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(a[u]);
    apart();
    load(a, s + 2 * U);
    apart();
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(b[u]);
    up_to_end(a, s + 2 * U);
    return;
  }
  if (!BOTH) load(b, s + U);
  up_to_end(a, s);
  up_to_end(b, s + U);
}

// W nontemporal (streamed once, must not evict L2); x plain (re-read by every
// n-block: L2 is exactly where it wants to live). Columns past M read the last
// row again: their results are not stored, and x stays as short as it is.
// Loads run a chunk of U kilobytes ahead, without a branch among them (one
// makes the compiler wait for all of them); past a wave's range they read its
// last kilobyte again.
//
// Bound by the weight stream, and with 32 rows by x (as long as W, or twice as
// long as e4m3). us before -> now, weights out of cache, for N x K of
// 12288 x 4096, 22016 x 4096, 4096 x 4096 and 4096 x 11008 (up to 16 rows of such sizes
// are weight_stream16's since; of 1 and 16 rows this is what it was chosen over):
//   bf16  1 row    23.1 -> 20.0  36.9 -> 32.3  8.9 -> 8.2  21.3 -> 17.3
//         16 rows  24.3 -> 22.5  37.5 -> 33.1  9.1 -> 8.6  21.6 -> 17.7
//         32 rows  23.5 -> 23.6  37.5 -> 38.3  9.3 -> 9.3  21.9 -> 20.2
//   e4m3 (before: tiles through LDS, a slab slice per 256 columns)
//         1 row    31.9 -> 13.8  47.3 -> 20.1  17.7 -> 6.3  39.5 -> 12.4
//         16 rows  32.5 -> 14.1  49.3 -> 20.8  17.7 -> 6.5  37.7 -> 12.8
//         32 rows  34.7 -> 17.7  56.5 -> 26.4  18.1 -> 7.7  38.1 -> 16.0
template <bool FP8, typename Meanwhile>
__device__ __forceinline__ void weight_stream(
    const uint16_t *__restrict__ xs, const uint8_t *__restrict__ ws, int M,
    int K, float (&red)[4][32][MMAX], Meanwhile meanwhile) {
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
  stream_chunks<false, false>(a, b, s0, s1, load, multiply, meanwhile);
#pragma unroll
  for (int r = 0; r < 16; ++r)
    red[wid][(r & 3) + 8 * (r >> 2) + 4 * hi][col] = acc[r];
}

// The same of up to 16 rows x: products of 16 x 16, two of which share an operand of
// x, so half as many loads of x go with one of W. A step is two kilobytes of W, 32
// columns (e4m3: 64), its operands as in decode_res.hip.
//
// us in a graph with the norm left out of x and the ends, of 1 and 16 rows, by products
// of 32 x 32 with the ends behind one chunk of W, and so: 12288 x 4096 and rotation 20.1
// and 19.3, 21.0 and 20.3 (W alone takes 17.8); 6144 x 4096 11.8 and 11.2, 12.4 and 11.7;
// 22016 x 4096 and unit 32.1 and 31.0, 32.5 and 31.2 (29.3); 49152 x 3072 46.0 and 45.1,
// 46.0 and 44.4; in e4m3 12288 x 4096 14.0 and 11.6, 14.6 and 13.0 (9.5), 22016 x 4096
// 20.4 and 16.9, 19.4 and 17.7 (16).
// In e4m3, whose conversions the compiler gathers with the products, loads are kept apart
// from these (APART; 9 to 16 rows of 12288 x 3072 11.4 us by 32 x 32, 11.8 with loads
// behind the products, 10.7 apart and with nothing loaded past the end). In bf16 they
// stand behind a loop's products as compiled, 24 loads after a wait for all: apart, q, k
// and v take 1 to 6% less and heads of 128256 rows 1 to 3% more.
template <bool FP8, typename Meanwhile>
__device__ __forceinline__ void weight_stream16(
    const uint16_t *__restrict__ xs, const uint8_t *__restrict__ ws, int M,
    int K, float (&red)[4][32][17], Meanwhile meanwhile) {
  constexpr int X = FP8 ? 2 : 1, U = 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, i16 = lane & 15, grp = lane >> 4;
  const int steps = K / (32 * X), groups = gridDim.y * 4;
  const int g = blockIdx.y * 4 + wid;
  const int s0 = (int)((int64_t)steps * g / groups);
  const int s1 = (int)((int64_t)steps * (g + 1) / groups);
  const uint8_t *w = ws + (int64_t)blockIdx.x * steps * 2048 + grp * 512 +
                     i16 * 16;
  const uint8_t *x = reinterpret_cast<const uint8_t *>(xs) +
                     (FP8 ? (grp >> 1) * 2048 + (grp & 1) * 512 : grp * 512) +
                     min(i16, M - 1) * 16;
  struct Both { u32x4v w[2]; bf16x8v x[X]; };
  Both a[U], b[U];
  f32x4v acc[2] = {(f32x4v)(0.0f), (f32x4v)(0.0f)};
  auto load = [&](Both (&c)[U], int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t at = min(s + u, s1 - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        c[u].w[h] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4v *>(w + at * 2048 + h * 256));
#pragma unroll
      for (int i = 0; i < X; ++i)
        c[u].x[i] = load8v(reinterpret_cast<const uint16_t *>(
            x + at * (2048 * X) + i * 1024));
    }
  };
  auto multiply = [&](const Both &c) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (FP8) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              fp8_to_bf16(c.w[h][2 * i], c.w[h][2 * i + 1]), c.x[i], acc[h], 0,
              0, 0);
      } else {
        union { u32x4v u; bf16x8v v; } t;
        t.u = c.w[h];
        acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t.v, c.x[0], acc[h],
                                                         0, 0, 0);
      }
    }
  };
  stream_chunks<true, FP8>(a, b, s0, s1, load, multiply, meanwhile);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      red[wid][h * 16 + grp * 4 + r][i16] = acc[h][r];
}

// FEW: up to 16 rows, K a multiple of 32 (e4m3: 64).
// In bf16 the 32 x 32 kernel is kept to registers for three workgroups a CU, which it has
// without being told in e4m3 (148): left alone it takes 176, room for two (us of 17 rows
// with two and three, norm and ends included: 22016 x 4096 33.1 and 32.5, 6144 x 4096
// 12.7 and 12.5, 36864 x 2048 29.1 and 28.1, 34816 x 1024 16.9 and 15.6).
template <bool FP8, Kind KIND, bool FEW>
__global__ __launch_bounds__(BLOCK, FEW || FP8 ? 1 : 3) void decode_gemm_kernel(
    const uint16_t *__restrict__ xs, const uint8_t *__restrict__ ws, int M,
    int N, int K, Ends e) {
  __shared__ __attribute__((aligned(16))) float red[4][32][FEW ? 17 : MMAX];
  Early<KIND> early;
  const bool mine = !FEW || Early<KIND>::mine(M);
  if (mine) {
    early.begin(e, M);
    if constexpr (FP8) early.begin_scale(e);
  }
  auto meanwhile = [&] {
    if (mine) early.rest(e, M);
  };
  if constexpr (FEW) weight_stream16<FP8>(xs, ws, M, K, red, meanwhile);
  else weight_stream<FP8>(xs, ws, M, K, red, meanwhile);
  finish<FP8, KIND, FEW ? 17 : MMAX>(red, e, early, M, N);
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
// Of the ends, which took 1.3 to 3 us behind the stream where one group's wave had
// them all, every group takes a share, with its angles loaded ahead of the sums; a
// wave that shares its tile with no other waits for none. 12288 x 4096 and rotation of
// 32, 45 and 64 rows 21.8 -> 21.1, 24.5 -> 23.4, 26.4 -> 25.4 us, 6144 x 4096 of 45
// 19.1 -> 17.6, 3072 x 1024 of 64 10.0 -> 8.6. W four chunks ahead in place of two
// changes nothing: with 64 rows a CU's loads of x, all of which every workgroup needs,
// are the bound.
template <int RB, int NWN, int CH, Kind KIND>
__global__ __launch_bounds__(BLOCK, 2) void decode_gemm_rows_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ ws, int M,
    int N, int K, Ends e) {
  constexpr int KG = 4 / NWN, P = 2 * CH;          // pieces of a row
  constexpr int XL = RB * CH / NWN;                // of x, a lane and chunk
  constexpr int TILE = RB * 32 * P * 16;
  static_assert(XL * NWN == RB * CH && (KG == 1 || 2 * KG * TILE >= RB * 16384),
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
  constexpr bool NORM = RB <= 2 && KIND != ends::SLAB;
  __shared__ float norms[NORM ? RB * 32 : 1];
  Early<ends::PLAIN> early[NORM ? RB : 1];
  if constexpr (NORM)
#pragma unroll
    for (int b = 0; b < RB; ++b) early[b].begin(e, M, b * 32);
  // A sum's 8 registers 4 q .. 4 q + 3 and 8 more, of RB blocks of rows: shares of the
  // groups by turns, which end them side by side
  constexpr int SHARES = RB * 2, OWN = (SHARES + KG - 1) / KG;
  constexpr bool HEADS = KIND == ends::QKV;
  ends::Turn<4> turn[HEADS ? OWN : 1];
  int position[HEADS ? OWN : 1];
  auto row_of = [&](int i) { return min((kg + i * KG) / 2 * 32 + col, M - 1); };
  auto turns = [&] {
    if constexpr (HEADS)
#pragma unroll
      for (int i = 0; i < OWN; ++i)
        turn[i].load(e, row_of(i),
                     min(nblk, blocks - 1) * 16 + 8 * ((kg + i * KG) & 1) + 4 * hi,
                     position[i]);
  };
  if constexpr (HEADS)
#pragma unroll
    for (int i = 0; i < OWN; ++i) position[i] = e.pos[row_of(i)];

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
  auto meet = [] {                                 // those that share a tile
    if constexpr (NWN > 1) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    }
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
  // of up to 64 rows x is two chunks ahead, too, which more have no registers for
  // (us with x one and two ahead: 12288 x 4096 of 45 rows 24.8 and 24.1, of 32 23.5
  // and 22.3; 5120 x 13824 35.2 and 33.4, 37.0 and 33.0)
  constexpr int FAR = RB <= 2 ? 2 : 1;
  X x0, x1;
  W w0, w1;
  load_x(x0, s0);
  load_w(w0, s0);
  if constexpr (FAR == 2) load_x(x1, s0 + CH);
  else put_x(x0, mine);
  if constexpr (FAR == 1) load_x(x0, s0 + CH);
  load_w(w1, s0 + CH);
  if constexpr (FAR == 2) {
    put_x(x0, mine);
    load_x(x0, s0 + 2 * CH);
  }
  if constexpr (NORM) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      early[b].rest(e, M);
      if (threadIdx.x % 8 == 0) norms[b * 32 + threadIdx.x / 8] = early[b].norm;
    }
  }
  constexpr bool AHEAD = OWN <= 2;                 // more have no registers for it
  if constexpr (AHEAD) turns();
  meet();
  // chunk c, of which `w` holds W and then W of chunk c + 2; `xr` holds x of chunk
  // c + 1 and then of chunk c + 1 + FAR
  auto step = [&](W &w, X &xr, int c, auto whole) {
    const int s = s0 + c * CH;
    put_x(xr, mine + (~c & 1) * KG * TILE);
    load_x(xr, s + (1 + FAR) * CH);
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
    step(w0, FAR == 2 ? x1 : x0, c, std::true_type{});
    step(w1, x0, c + 1, std::true_type{});
  }
  for (; c < chunks; c += 2) {
    step(w0, FAR == 2 ? x1 : x0, c, std::false_type{});
    step(w1, x0, c + 1, std::false_type{});
  }
  if constexpr (!AHEAD) turns();
  if constexpr (NWN == 1) __syncthreads();         // every wave's tiles, norms
  // sum of the groups: what is another's share goes to LDS
  float *red = reinterpret_cast<float *>(smem) + wn * SHARES * KG * 512 + lane * 4;
  if constexpr (KG > 1) {
#pragma unroll
    for (int i = 0; i < SHARES; ++i)
      if (i % KG != kg)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int r = h * 8 + i % 2 * 4;
          *reinterpret_cast<float4 *>(red + (i * KG + kg) * 512 + h * 256) =
              make_float4(acc[i / 2][r], acc[i / 2][r + 1], acc[i / 2][r + 2],
                          acc[i / 2][r + 3]);
        }
    __syncthreads();
  }
  if (nblk >= blocks) return;
#pragma unroll
  for (int i = 0; i < SHARES; ++i) {
    if (i % KG != kg) continue;
    const int b = i / 2, q = i % 2, m = b * 32 + col;
    float f[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) f[h][j] = acc[b][h * 8 + q * 4 + j];
    if constexpr (KG > 1) {
      float4 other[2][KG];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < KG; ++g)
          other[h][g] = g == i % KG
              ? make_float4(f[h][0], f[h][1], f[h][2], f[h][3])
              : *reinterpret_cast<float4 *>(red + (i * KG + g) * 512 + h * 256);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float4 sum = other[h][0];
#pragma unroll
        for (int g = 1; g < KG; ++g) {
          sum.x += other[h][g].x; sum.y += other[h][g].y;
          sum.z += other[h][g].z; sum.w += other[h][g].w;
        }
        f[h][0] = sum.x; f[h][1] = sum.y; f[h][2] = sum.z; f[h][3] = sum.w;
      }
    }
    if constexpr (NORM) {
      const float norm = norms[m];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) f[h][j] *= norm;
    }
    if (m >= M) continue;
    // registers r and r + 8 of a lane are a pair, 4 neighbours at a time
    const int p = nblk * 16 + 8 * q + 4 * hi;
    if constexpr (HEADS) {
      ends::put_heads<4>(e, turn[i / KG], m, p, N, f[0], f[1]);
    } else if constexpr (KIND == ends::GLU) {
      ends::put_gated<4>(e, m, p, N, f[0], f[1]);
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = ends::column(e.half, nblk, 16 * h + 8 * q + 4 * hi);
        if constexpr (KIND == ends::PLAIN)
          ends::put<4>(e.y + (int64_t)m * N + n, f[h]);
        else
          *reinterpret_cast<float4 *>(
              e.slabs + ((int64_t)blockIdx.y * M + m) * N + n) =
              make_float4(f[h][0], f[h][1], f[h][2], f[h][3]);
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

static void check_pairs(int64_t N, int64_t half) {
  TORCH_CHECK(half == 0 ||
              (half > 0 && half % 16 == 0 && N % (2 * half) == 0),
              "decode_gemm: pairs");
}

// One-time weight swizzle (host-side tensor ops): [N,K] ->
// [N/32][K/16][2][32][8] = fragment-lane-major chunks of 1 KiB.
// With `half` its rows go in pairs (decode_ends.h).
at::Tensor decode_swizzle_w(at::Tensor w, int64_t half) {
  TORCH_CHECK(w.dim() == 2 && w.scalar_type() == at::kBFloat16 &&
              w.is_contiguous(), "decode_swizzle_w: contiguous bf16 [N,K]");
  const int64_t N = w.size(0), K = w.size(1);
  TORCH_CHECK(N % 32 == 0 && K % 16 == 0, "decode_swizzle_w: shape");
  check_pairs(N, half);
  // moved by words of 8 bytes
  const auto q = (w.storage_offset() % 4 ? w.clone() : w).view(at::kLong);
  const auto laid =
      half == 0 ? q.view({N / 32, 32, K / 16, 2, 2}).permute({0, 2, 3, 1, 4})
                : q.view({N / (2 * half), 2, half / 16, 16, K / 16, 2, 2})
                      .permute({0, 2, 4, 5, 1, 3, 6});
  return laid.contiguous().view(at::kBFloat16).view({N / 32, K / 16, 2, 32, 8});
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
at::Tensor decode_swizzle_w8(at::Tensor w8, int64_t half) {
  TORCH_CHECK(w8.dim() == 2 && w8.scalar_type() == at::kByte &&
              w8.is_contiguous(), "decode_swizzle_w8: contiguous bytes [N,K]");
  const int64_t N = w8.size(0), K = w8.size(1);
  TORCH_CHECK(N % 32 == 0 && K % 32 == 0, "decode_swizzle_w8: shape");
  check_pairs(N, half);
  const auto q = (w8.storage_offset() % 8 ? w8.clone() : w8).view(at::kLong);
  const auto laid =
      half == 0 ? q.view({N / 32, 32, K / 32, 2, 2}).permute({0, 2, 4, 1, 3})
                : q.view({N / (2 * half), 2, half / 16, 16, K / 32, 2, 2})
                      .permute({0, 2, 4, 6, 1, 3, 5});
  return laid.contiguous().view(at::kByte).view({N / 32, K / 32, 2, 32, 2, 8});
}

template <bool FP8>
static void launch(Kind kind, const at::Tensor &xs, const at::Tensor &ws,
                   const Ends &e, int split, int64_t M, int64_t N, int64_t K) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(N / 32), (unsigned)split),
                       dim3(BLOCK), 0, at::cuda::getCurrentHIPStream(),
                       (const uint16_t *)xs.data_ptr(),
                       (const uint8_t *)ws.data_ptr(), (int)M, (int)N, (int)K,
                       e);
  };
  auto of = [&](auto few) {
    constexpr bool FEW = decltype(few)::value;
    switch (kind) {
      case ends::SLAB: return go(decode_gemm_kernel<FP8, ends::SLAB, FEW>);
      case ends::PLAIN: return go(decode_gemm_kernel<FP8, ends::PLAIN, FEW>);
      case ends::GLU: return go(decode_gemm_kernel<FP8, ends::GLU, FEW>);
      case ends::QKV: return go(decode_gemm_kernel<FP8, ends::QKV, FEW>);
    }
  };
  // Of e4m3 columns a wave has one chunk of these where there are up to 1024 of them, and
  // its second one is loaded for nothing: no matter where a CU has no more than one
  // workgroup (us of the products of 16 x 16 and of 32 x 32, 1024 columns: 4096 and 8192
  // rows 4.4 and 4.6, 4.7 and 4.9; 49152 14.9 and 13.3)
  const bool few = M <= 16 && K % (FP8 ? 64 : 32) == 0 &&
                   (!FP8 || K > 1024 * split || N / 32 * split <= 256);
  if (few) of(std::true_type{});
  else of(std::false_type{});
}

// The sums of a product as slabs [split, M, N], or, unsplit, y [M, N] bf16.
template <bool FP8>
static at::Tensor sums(const at::Tensor &xs, const at::Tensor &ws, Ends e,
                       int split, bool slab, int64_t M, int64_t N, int64_t K) {
  at::Tensor out;
  if (slab) {
    out = at::empty({split, M, N}, xs.options().dtype(at::kFloat));
    e.slabs = out.data_ptr<float>();
  } else {
    out = at::empty({M, N}, xs.options());
    e.y = (uint16_t *)out.data_ptr();
  }
  if (N > 0)
    launch<FP8>(slab ? ends::SLAB : ends::PLAIN, xs, ws, e, split, M, N, K);
  return out;
}

static void combine(const at::Tensor &slabs, at::Tensor &y) {
  hipLaunchKernelGGL(decode_gemm_combine_kernel,
                     dim3(rb::rb_grid_1d(y.numel() / 4, 256)), dim3(256), 0,
                     at::cuda::getCurrentHIPStream(),
                     slabs.data_ptr<float>(), (uint16_t *)y.data_ptr(),
                     (int)slabs.size(0), y.numel());
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

// An operand [K/16][2][32][8] and W [N, K] as decode_swizzle_w or
// decode_swizzle_w8 (with the scales of its rows) lays it.
static bool check_product(const at::Tensor &xs, const at::Tensor &ws,
                          const c10::optional<at::Tensor> &scale, int64_t M,
                          int64_t N, int64_t K, int64_t half) {
  const bool fp8 = ws.scalar_type() == at::kByte;
  TORCH_CHECK(xs.is_cuda() && ws.device() == xs.device() &&
              xs.is_contiguous() && ws.is_contiguous() &&
              xs.scalar_type() == at::kBFloat16 &&
              (fp8 || ws.scalar_type() == at::kBFloat16), "decode_gemm: inputs");
  TORCH_CHECK(M >= 1 && M <= MMAX && N >= 0 && N % 32 == 0 && K > 0 &&
              K % (fp8 ? 32 : 16) == 0 && xs.numel() == (K / 16) * 512 &&
              ws.numel() == N * K &&
              (fp8 || decode_gemm_supported(M, N, K)), "decode_gemm: shape ",
              M, "x", N, "x", K);
  check_pairs(N, half);
  TORCH_CHECK(fp8 == scale.has_value() &&
              (!fp8 || (scale->device() == xs.device() &&
                        scale->is_contiguous() &&
                        scale->scalar_type() == at::kFloat &&
                        scale->numel() == N)), "decode_gemm: scales");
  return fp8;
}

// The input came without its norm's 1 / rms: `squares` [M, parts] are parts of
// the sums of squares of its rows of d.
static void set_squares(Ends &e, const c10::optional<at::Tensor> &squares,
                        int64_t M, int64_t d, double eps) {
  if (!squares.has_value()) return;
  TORCH_CHECK(squares->is_cuda() && squares->is_contiguous() &&
              squares->dim() == 2 && squares->size(0) == M &&
              squares->size(1) % 4 == 0 && squares->size(1) > 0 &&
              squares->size(1) <= 256 &&
              squares->scalar_type() == at::kFloat &&
              reinterpret_cast<uintptr_t>(squares->data_ptr()) % 16 == 0,
              "decode_gemm: squares [M, 4 n <= 256]");
  e.squares = squares->data_ptr<float>();
  e.parts = (int)squares->size(1);
  e.inv_d = 1.0f / (float)d;
  e.eps = (float)eps;
}

// Where queries, keys and values [M, N] of heads go.
static void set_heads(Ends &e, int64_t M, int64_t N, const at::Tensor &cos,
                      const at::Tensor &sin, const at::Tensor &positions,
                      const at::Tensor &k_cache, const at::Tensor &v_cache,
                      const at::Tensor &slots, int64_t hq) {
  TORCH_CHECK(k_cache.is_cuda() && k_cache.dim() == 4 && v_cache.dim() == 4 &&
              k_cache.scalar_type() == at::kBFloat16 &&
              v_cache.scalar_type() == at::kBFloat16 &&
              k_cache.is_contiguous() && v_cache.is_contiguous() &&
              reinterpret_cast<uintptr_t>(k_cache.data_ptr()) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(v_cache.data_ptr()) % 8 == 0,
              "decode_heads: caches");
  e.hq = (int)hq;
  e.hkv = (int)k_cache.size(1);
  e.bs = (int)k_cache.size(2);
  e.dh = (int)k_cache.size(3);
  const int64_t dh = e.dh;
  TORCH_CHECK(dh % 32 == 0 && dh > 0 && e.bs > 0 && hq > 0 && e.hkv > 0 &&
              (hq + 2 * e.hkv) * dh == N &&
              v_cache.numel() == k_cache.numel() &&
              v_cache.size(1) == k_cache.size(1), "decode_heads: widths");
  e.vt = v_cache.size(3) == e.bs && v_cache.size(2) == dh && dh != e.bs;
  TORCH_CHECK(positions.is_cuda() && slots.is_cuda() &&
              positions.scalar_type() == at::kInt &&
              slots.scalar_type() == at::kInt && positions.is_contiguous() &&
              slots.is_contiguous() && positions.numel() >= M &&
              slots.numel() >= M, "decode_heads: positions, slots");
  TORCH_CHECK(cos.is_cuda() && sin.is_cuda() &&
              cos.scalar_type() == at::kFloat &&
              sin.scalar_type() == at::kFloat && cos.is_contiguous() &&
              sin.is_contiguous() && cos.size(-1) == dh / 2 &&
              sin.sizes() == cos.sizes() &&
              reinterpret_cast<uintptr_t>(cos.data_ptr()) % 8 == 0 &&
              reinterpret_cast<uintptr_t>(sin.data_ptr()) % 8 == 0,
              "decode_heads: tables");
  e.half = (int)(dh / 2);
  e.cs = cos.data_ptr<float>();
  e.sn = sin.data_ptr<float>();
  e.pos = positions.data_ptr<int32_t>();
  e.slots = slots.data_ptr<int32_t>();
  e.k_cache = (uint16_t *)k_cache.data_ptr();
  e.v_cache = (uint16_t *)v_cache.data_ptr();
}

// Raw variant for fused consumers: split == 1 returns y bf16 [M, N] (with
// f32 a slab of one slice); split > 1 returns the fp32 slab [split, M, N]
// UNCOMBINED — the consumer kernel (rmsnorm_res_slab_fwd) folds the
// slices while it reads, saving the combine launch inside the decode graph.
at::Tensor decode_gemm_raw(at::Tensor xs, at::Tensor ws, int64_t M,
                           int64_t N, int64_t K, bool f32, int64_t half) {
  TORCH_CHECK(!check_product(xs, ws, c10::nullopt, M, N, K, half),
              "decode_gemm_raw: bf16");
  Ends e{};
  e.half = (int)half;
  const int split = (int)decode_gemm_split(N, K);
  return sums<false>(xs, ws, e, split, split > 1 || f32, M, N, K);
}

// xs from decode_swizzle_x, ws from decode_swizzle_w; M/N/K of the
// ORIGINAL y[M,N] = x[M,K] @ W[N,K]^T problem.
at::Tensor decode_gemm(at::Tensor xs, at::Tensor ws, int64_t M, int64_t N,
                       int64_t K, int64_t force_split, int64_t half) {
  TORCH_CHECK(!check_product(xs, ws, c10::nullopt, M, N, K, half),
              "decode_gemm: bf16 only");
  Ends e{};
  e.half = (int)half;
  const int split = force_split > 0 ? (int)force_split
                                    : (int)decode_gemm_split(N, K);
  auto out = sums<false>(xs, ws, e, split, split > 1, M, N, K);
  if (split == 1) return out;
  auto y = at::empty({M, N}, xs.options());
  combine(out, y);
  return y;
}

// The product with e4m3 weights (decode_swizzle_w8) and a scale per row:
// y [M, N] bf16, or with raw=true, where it is split, the uncombined fp32
// slabs [split, M, N].
at::Tensor decode_gemm_fp8(at::Tensor xs, at::Tensor w8s, at::Tensor scale,
                           int64_t M, int64_t N, int64_t K, bool raw,
                           int64_t half) {
  TORCH_CHECK(check_product(xs, w8s, scale, M, N, K, half),
              "decode_gemm_fp8: inputs");
  Ends e{};
  e.half = (int)half;
  e.scale = scale.data_ptr<float>();
  const int split = (int)decode_gemm_split(N, K);
  auto out = sums<true>(xs, w8s, e, split, split > 1, M, N, K);
  if (split == 1 || raw) return out;
  auto y = at::empty({M, N}, xs.options());
  combine(out, y);
  return y;
}

static void launch_ends(Kind kind, const at::Tensor &xs, const at::Tensor &ws,
                        const c10::optional<at::Tensor> &scale, Ends &e,
                        int64_t M, int64_t N, int64_t K) {
  if (scale.has_value()) {
    e.scale = scale->data_ptr<float>();
    launch<true>(kind, xs, ws, e, 1, M, N, K);
  } else {
    launch<false>(kind, xs, ws, e, 1, M, N, K);
  }
}

// Gate and unit of a gated unit in one product: act(x G^T) * (x U^T) as the
// operand of the next one. W = [G ; U], its copy paired by half its rows;
// squares: set_squares.
at::Tensor decode_glu(at::Tensor xs, at::Tensor ws,
                      c10::optional<at::Tensor> scale, int64_t M, int64_t N,
                      int64_t K, bool gelu, c10::optional<at::Tensor> squares,
                      double eps, bool rows) {
  check_product(xs, ws, scale, M, N, K, N / 2);
  TORCH_CHECK(N > 0, "decode_glu: rows");
  Ends e{};
  e.half = (int)(N / 2);
  e.gelu = gelu;
  set_squares(e, squares, M, K, eps);
  auto out = rows ? at::empty({M, N / 2}, xs.options())
                  : at::empty({N / 32 * 512}, xs.options());
  (rows ? e.y : e.operand) = (uint16_t *)out.data_ptr();
  launch_ends(ends::GLU, xs, ws, scale, e, M, N, K);
  return out;
}

// Rotated q [M, hq, dh] of one product; its rotated keys and its values go to
// the bf16 cache. W's copy is paired by half a head.
at::Tensor decode_heads(at::Tensor xs, at::Tensor ws,
                        c10::optional<at::Tensor> scale, int64_t M, int64_t N,
                        int64_t K, c10::optional<at::Tensor> squares,
                        double eps, at::Tensor cos, at::Tensor sin,
                        at::Tensor positions, at::Tensor k_cache,
                        at::Tensor v_cache, at::Tensor slots, int64_t hq) {
  Ends e{};
  set_heads(e, M, N, cos, sin, positions, k_cache, v_cache, slots, hq);
  check_product(xs, ws, scale, M, N, K, e.half);
  set_squares(e, squares, M, K, eps);
  auto q = at::empty({M, hq, e.dh}, xs.options());
  e.q = (uint16_t *)q.data_ptr();
  launch_ends(ends::QKV, xs, ws, scale, e, M, N, K);
  return q;
}

// The product with the input's norm left out of it (squares: set_squares).
at::Tensor decode_normed(at::Tensor xs, at::Tensor ws,
                         c10::optional<at::Tensor> scale, int64_t M, int64_t N,
                         int64_t K, at::Tensor squares, double eps,
                         int64_t half) {
  check_product(xs, ws, scale, M, N, K, half);
  TORCH_CHECK(N > 0, "decode_normed: rows");
  Ends e{};
  e.half = (int)half;
  set_squares(e, squares, M, K, eps);
  auto y = at::empty({M, N}, xs.options());
  e.y = (uint16_t *)y.data_ptr();
  launch_ends(ends::PLAIN, xs, ws, scale, e, M, N, K);
  return y;
}

template <int RB, int NWN, int CH>
static void launch_rows(Kind kind, const at::Tensor &x, const at::Tensor &ws,
                        const Ends &e, int64_t N, int split) {
  const int64_t M = x.size(0), K = x.size(1);
  constexpr int lds = 2 * (4 / NWN) * RB * 32 * CH * 32;
  static_assert(lds <= 64 * 1024, "tiles");
  TORCH_CHECK(split >= 1 && split * (4 / NWN) <= K / 16, "decode_gemm_rows");
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel,
                       dim3((unsigned)((N / 32 + NWN - 1) / NWN),
                            (unsigned)split), dim3(BLOCK), lds,
                       at::cuda::getCurrentHIPStream(),
                       (const uint16_t *)x.data_ptr(),
                       (const uint8_t *)ws.data_ptr(), (int)M, (int)N, (int)K,
                       e);
  };
  if (kind == ends::GLU)
    return go(decode_gemm_rows_kernel<RB, NWN, CH, ends::GLU>);
  if (kind == ends::QKV)
    return go(decode_gemm_rows_kernel<RB, NWN, CH, ends::QKV>);
  if constexpr (NWN > 1) {
    kind == ends::SLAB ? go(decode_gemm_rows_kernel<RB, NWN, CH, ends::SLAB>)
                       : go(decode_gemm_rows_kernel<RB, NWN, CH, ends::PLAIN>);
  }
}

// How a product of 1 to 128 rows is cut.
//
// One workgroup for every CU where it can be had, as a second on some of them
// has the others wait: four blocks of W for wide weights, unsplit; else two, or
// four for long rows, of which splits to fill the CUs cost less (us with two
// and four at their best split: 4096 x 11008 of 64 rows 25 and 26, of 100 rows
// 32 and 30; 3072 x 24576 38 and 34, 50 and 41; 4096 x 4096 14 and 16, 17 and
// 20; 22016 x 4096 of 64 rows 45 and 36, 12288 x 4096 25 and 26). Where four blocks
// have up to half of the CUs take a second workgroup and the others none, two are
// spread better, except that with more rows what x takes of a CU grows, the more the
// longer they are. us of a gated unit (of a product as it is) with four and two blocks,
// of 48 and 64 rows:
//   34816 x  1024   22.8  20.4 ( 23.2  20.5)   23.8  21.8 ( 24.2  21.9)
//   49152 x  2048   42.8  39.6 ( 44.1  39.8)   43.7  41.7 ( 44.8  42.8)
//   49152 x  3072   56.8  54.3 ( 57.5  55.5)   59.0  57.4 ( 60.2  59.4)
//   36864 x  4096   69.5  64.8 ( 69.8  66.0)   71.3  68.9 ( 71.7  70.5)
//   40960 x  4096   70.9  67.0 ( 71.1  68.6)   72.6  71.3 ( 73.1  73.3)
//   49152 x  4096   73.9  72.5 ( 74.6  75.1)   75.6  77.1 ( 77.0  80.9)
//   43008 x  5120   87.1  83.3 ( 87.4  85.2)   91.2  92.2 ( 91.9  95.0)
//   35840 x  6656  107.0  99.4 (107.3 100.5)  110.5 107.5 (111.2 109.9)
//   44032 x  8192  134.1 124.7 (134.8 128.5)  138.2 136.0 (139.1 140.0)
//   49152 x 12288  209.0 200.8 (212.7 206.9)  218.2 216.4 (221.5 226.1)
// Of 17 rows two blocks take 3 to 15% less, of 100 the same or more, and two workgroups
// on every CU have nothing to spread (65536 x 4096 of 45 rows 87 and 90).
struct Cut { int blocks, split; };
static Cut cut_of(int64_t M, int64_t N, int64_t K) {
  const bool spill = N > 32768 && N <= 49152 &&
                     M <= (N <= 36864 || N * K <= 40960 * 4096 ? 64 : 48);
  Cut c{(N >= 20480 && !spill) || K >= (M <= 64 ? 20480 : 8192) ? 4 : 2, 1};
  const int64_t wgs = (N / 32 + c.blocks - 1) / c.blocks;
  while (c.split < 8 && wgs * c.split * 2 <= 256 && K / (c.split * 2) >= 256)
    c.split *= 2;
  return c;
}

// The same for products with ends, which need whole sums: one block of W for a
// workgroup where two are too few workgroups (6144 x 4096 of 64 rows and its
// rotation: 25.6 us in two parts and three launches, 23.8 with two blocks whole).
static Cut whole_cut_of(int64_t M, int64_t N, int64_t K) {
  Cut c = cut_of(M, N, K);
  if (c.blocks == 2 && c.split > 1 && M <= 64) c.blocks = 1;
  c.split = 1;
  return c;
}

// Whether such a product is the faster way: of more than 64 rows, workgroups
// of one block find no registers, and parts win (6144 x 4096 of 128 rows 32.1
// and 34.7 us).
bool rows_ends_pay(int64_t M, int64_t N, int64_t K) {
  return whole_cut_of(M, N, K).blocks == 1 || cut_of(M, N, K).split == 1;
}

static void run_rows(Kind kind, const at::Tensor &x, const at::Tensor &ws,
                     const Ends &e, int64_t N, Cut c) {
  auto go = [&](auto rb) {
    constexpr int RB = decltype(rb)::value;
    if constexpr (RB < 4)
      if (c.blocks == 1) return launch_rows<RB, 1, 4>(kind, x, ws, e, N, 1);
    if (c.blocks == 2) launch_rows<RB, 2, 4>(kind, x, ws, e, N, c.split);
    else launch_rows<RB, 4, RB == 4 ? 4 : 8>(kind, x, ws, e, N, c.split);
  };
  const int64_t M = x.size(0);
  if (M <= 32) go(std::integral_constant<int, 1>{});
  else if (M <= 64) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
}

static void check_rows(const at::Tensor &x, const at::Tensor &ws, int64_t N,
                       int64_t half) {
  TORCH_CHECK(x.is_cuda() && ws.device() == x.device() && x.dim() == 2 &&
              x.is_contiguous() && ws.is_contiguous() &&
              x.scalar_type() == at::kBFloat16 &&
              ws.scalar_type() == at::kBFloat16 &&
              reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "decode_gemm_rows: inputs");
  const int64_t M = x.size(0), K = x.size(1);
  TORCH_CHECK(M >= 1 && M <= 128 && N > 0 && N % 32 == 0 && K % 16 == 0 &&
              K >= 1024 && K < (1 << 24) && ws.numel() == N * K,
              "decode_gemm_rows: shape");
  check_pairs(N, half);
}

// y [M, N] = x [M, K] W^T of 1 to 128 rows; ws from decode_swizzle_w. raw:
// where it is split, the fp32 parts [split, M, N].
at::Tensor decode_gemm_rows(at::Tensor x, at::Tensor ws, int64_t N,
                            int64_t half, bool raw) {
  check_rows(x, ws, N, half);
  const int64_t M = x.size(0), K = x.size(1);
  const Cut c = cut_of(M, N, K);
  Ends e{};
  e.half = (int)half;
  at::Tensor y, slabs;
  if (c.split > 1) {
    slabs = at::empty({c.split, M, N}, x.options().dtype(at::kFloat));
    e.slabs = slabs.data_ptr<float>();
  }
  if (c.split == 1 || !raw) {
    y = at::empty({M, N}, x.options());
    e.y = (uint16_t *)y.data_ptr();
  }
  run_rows(c.split > 1 ? ends::SLAB : ends::PLAIN, x, ws, e, N, c);
  if (c.split > 1 && raw) return slabs;
  if (c.split > 1) combine(slabs, y);
  return y;
}

// decode_glu of 1 to 128 rows x as they lie (up to 64 may come without their 1 /
// rms): the gated rows [M, N / 2], or, of up to 32 rows, an operand.
at::Tensor rows_glu(at::Tensor x, at::Tensor ws, int64_t N, bool gelu,
                    bool operand, c10::optional<at::Tensor> squares,
                    double eps) {
  check_rows(x, ws, N, N / 2);
  const int64_t M = x.size(0), K = x.size(1);
  TORCH_CHECK((M <= MMAX || !operand) &&
              (M <= 2 * MMAX || !squares.has_value()),
              "rows_glu: operand, squares");
  Ends e{};
  e.half = (int)(N / 2);
  e.gelu = gelu;
  set_squares(e, squares, M, K, eps);
  auto out = operand ? at::empty({N / 32 * 512}, x.options())
                     : at::empty({M, N / 2}, x.options());
  (operand ? e.operand : e.y) = (uint16_t *)out.data_ptr();
  run_rows(ends::GLU, x, ws, e, N, whole_cut_of(M, N, K));
  return out;
}

// decode_heads of 1 to 128 rows x as they lie (up to 64 may come without their 1 /
// rms): rotated q [M, hq, dh], or, in rows, q and k rotated and v side by side [M,
// N].
at::Tensor rows_heads(at::Tensor x, at::Tensor ws, int64_t N, at::Tensor cos,
                      at::Tensor sin, at::Tensor positions, at::Tensor k_cache,
                      at::Tensor v_cache, at::Tensor slots, int64_t hq,
                      bool rows, c10::optional<at::Tensor> squares, double eps) {
  Ends e{};
  const int64_t M = x.size(0), K = x.size(1);
  set_heads(e, M, N, cos, sin, positions, k_cache, v_cache, slots, hq);
  check_rows(x, ws, N, e.half);
  TORCH_CHECK(M <= 2 * MMAX || !squares.has_value(), "rows_heads: squares");
  set_squares(e, squares, M, K, eps);
  auto out = rows ? at::empty({M, N}, x.options())
                  : at::empty({M, hq, (int64_t)e.dh}, x.options());
  (rows ? e.y : e.q) = (uint16_t *)out.data_ptr();
  run_rows(ends::QKV, x, ws, e, N, whole_cut_of(M, N, K));
  return out;
}
