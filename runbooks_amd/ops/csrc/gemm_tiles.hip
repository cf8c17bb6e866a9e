// Products of many rows, x [M, K] times W [N, K] transposed, bf16 with fp32 sums,
// in tiles that suit their sizes, and ended by what follows them: parts of sums
// for the norm that adds them up, a gated unit, adapters; and x [M, K] times W [K,
// N], gradients of inputs, with adapters.
//
// Bound by L2, which feeds LDS at 16 TB/s (62 GB/s a CU: what is left of a
// product of 8192 x 8192 x 4096 without its matrix instructions takes 269 us in
// tiles of 256 x 256 and 554 in those of 128 x 128), and by the matrix cores
// (without loads 312 us, 1760 TFLOP/s; both together 382). So tiles are as large
// as their number allows; where it does not, for prompts of some hundred rows,
// workgroups share the sums.
//
// us in the library and here, weights out of cache: 256 x 4096 x 11008 52 and 37
// (4 parts), 512 x 4096 x 11008 78 and 48 (4), 1021 x 4096 x 11008 110 and 84 (2),
// 512 x 3072 x 24576 261 and 88 (4), 512 x 22016 x 4096 92 and 80, 1021 x 49152 x
// 3072 250 and 229, 2048 x 4096 x 14336 207 and 188, 7931 x 28672 x 4096 1292 and
// 1276 (1427 and 1306 with the gated unit).
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "decode_ends.h"

namespace tiles {

using ends::bf16x8v;
using ends::f32x4v;
using rb::buffer;
using rb::u32x4v;

typedef __attribute__((ext_vector_type(2))) uint32_t u32x2v;

__device__ __forceinline__ u32x2v packed(const float (&f)[4]) {
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4v;
  return __builtin_bit_cast(
      u32x2v, __builtin_convertvector((f32x4v){f[0], f[1], f[2], f[3]}, bf16x4v));
}

// Four columns of a lane from n on in each of two neighbouring 16 x 16 results, a
// and b, the first at column `first` of y, a row of `cols`: after an exchange
// between neighbouring fours, a lane stores eight. In pieces of 8 bytes a wave's
// store filled 32 of a line of 128 (us of zeros in these and in pieces of 16: 4096 x
// 4096 x 512 23.4 and 21.2, 8192 x 8192 x 1024 102 and 88, 2048 x 12288 x 4096 128
// and 122, 512 x 12288 x 4096 67 and 63).
__device__ __forceinline__ void put(uint16_t *y, u32x2v a, u32x2v b, int first,
                                    int fk, int cols, bool there) {
  const auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  const int n = first + (fk & 1) * 16 + (fk >> 1) * 8;
  if (!there || n >= cols) return;
  if (cols % 8 == 0) {
    *reinterpret_cast<u32x4v *>(y + n) = (u32x4v){lo[0], hi[0], lo[1], hi[1]};
  } else {
    *reinterpret_cast<u32x2v *>(y + n) = (u32x2v){lo[0], hi[0]};
    if (n + 4 < cols)
      *reinterpret_cast<u32x2v *>(y + n + 4) = (u32x2v){lo[1], hi[1]};
  }
}

// The same of one result.
__device__ __forceinline__ void put(uint16_t *y, u32x2v a, int first, int fk,
                                    int cols, bool there) {
  if (there && first + fk * 4 < cols)
    *reinterpret_cast<u32x2v *>(y + first + fk * 4) = a;
}

// As text, for the compiler copies sums between the register files otherwise.
__device__ __forceinline__ void mma(f32x4v &c, bf16x8v a, bf16x8v b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
               : "+a"(c) : "v"(a), "v"(b));
}

// The same beside a load of 16 bytes a lane into LDS at lds + MORE. Of one text, for
// the product then stands between the write of m0 and its use, which have to be an
// instruction apart: a wave issues one in four clocks, and a product takes 16.
template <unsigned MORE>
__device__ __forceinline__ void mma_load(f32x4v &c, bf16x8v a, bf16x8v b,
                                         u32x4v from, unsigned voff,
                                         unsigned soff, unsigned lds) {
  asm volatile(
      "s_add_u32 m0, %6, %7\n\t"
      "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
      "buffer_load_dwordx4 %3, %4, %5 offen lds"
      : "+a"(c)
      : "v"(a), "v"(b), "v"(voff), "s"(from), "s"(soff), "s"(lds), "n"(MORE)
      : "memory", "m0", "scc");
}

template <class F, int... Q>
__device__ __forceinline__ void each_of(F &f, std::integer_sequence<int, Q...>) {
  (f(std::integral_constant<int, Q>()), ...);
}
template <int N, class F> __device__ __forceinline__ void each(F &f) {
  each_of(f, std::make_integer_sequence<int, N>());
}

// A product by itself, outside of the matrix registers, which the sums fill.
__device__ __forceinline__ f32x4v product(bf16x8v a, bf16x8v b) {
  f32x4v c;
  asm volatile(
      "s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, 0\n\ts_nop 15"
      : "=&v"(c) : "v"(a), "v"(b));
  return c;
}

enum Kind {
  PLAIN,        // y [M, N] bf16
  PARTS,        // fp32 [P, M, N], K-tiles kt * p .. of every part
  SILU, GELU,   // act(x G^T) * (x U^T) of W = [G ; U], y [M, N / 2]
  LORA,         // y_i + scale t_i B_i^T of siblings side by side
};

// Adapters of rank 16: t [n, M, 16] and B_i [columns of i, 16], the first columns
// of the siblings multiples of 16; DOWN: A_i [16, N], start[i] elements behind b[0].
struct Adapters {
  const uint16_t *t, *b[3];
  int start[4], n;
  float scale;
};

// Of which columns of y adapters' part is: the sibling of column n.
__device__ __forceinline__ int sibling(const Adapters &a, int n) {
  return (a.n > 1 && n >= a.start[1]) + (a.n > 2 && n >= a.start[2]);
}

constexpr unsigned NOWHERE = 0x80000000;    // past the end of every such buffer

// i, known from here on: what is computed of it stays behind this.
__device__ __forceinline__ int pinned(int i) {
  asm volatile("" : "+s"(i));
  return i;
}

// Waits until the last products are in their registers, if `left` is 0. The
// compiler does not know what mma() takes, and may move sums about right behind
// the loop; this stands in it, and with a branch of its own, for otherwise the
// compiler makes a copy of the loop's body for its last round.
__device__ __forceinline__ void settle(int left) {
  asm volatile(
      "s_cmp_lg_u32 %0, 0\n\ts_cbranch_scc1 .Lsettled%=\n\t"
      "s_nop 15\n\ts_nop 15\n.Lsettled%=:" :: "s"(left) : "scc");
}

// A sum's way out of the matrix registers: as text, it stays where its use is.
__device__ __forceinline__ void take(float (&f)[4], const f32x4v &c) {
  asm volatile(
      "v_accvgpr_read_b32 %0, %4\n\tv_accvgpr_read_b32 %1, %5\n\t"
      "v_accvgpr_read_b32 %2, %6\n\tv_accvgpr_read_b32 %3, %7"
      : "=&v"(f[0]), "=&v"(f[1]), "=&v"(f[2]), "=&v"(f[3])
      : "a"(c[0]), "a"(c[1]), "a"(c[2]), "a"(c[3]));
}

// The end of LORA, in fp32 and rounded once: a product more, of 16 columns (and
// 16 absent ones), for each of 16 x 16 sums, from rows m0 and columns n0 on. In a
// pass of its own over y it took 42 us of 2048 x 22016 (lora_group.hip).
template <int FM, int FN>
__device__ __forceinline__ void end_lora(const Adapters &a,
                                         const f32x4v (&acc)[FM][FN],
                                         uint16_t *y, int m0, int n0, int fr,
                                         int fk, int M, int N) {
  const bf16x8v none = (bf16x8v)(__bf16)0.0f;
  auto start = [&](int s) {
    return s == 0 ? 0 : s == 1 ? a.start[1] : a.start[2];
  };
  const int at = (fk & 1) * 8;
  bf16x8v bw[FN], tx[FM];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = __builtin_amdgcn_readfirstlane(min(n0 + j * 16, N - 16));
    const int s = sibling(a, n);
    const uint16_t *b = s == 0 ? a.b[0] : s == 1 ? a.b[1] : a.b[2];
    const bf16x8v v = ends::load8v(
        b + (int64_t)(n - start(s) + fr) * 16 + at);
    bw[j] = fk < 2 ? v : none;
  }
  // of these and those below, where the compiler sees it: otherwise it waits
  // for all loads in the loop over K that follows
  constexpr int loaded = 0x0f70;        // vmcnt(0)
  __builtin_amdgcn_s_waitcnt(loaded);
  int of = -1;
  u32x2v held[FM];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = __builtin_amdgcn_readfirstlane(n0 + j * 16);
    if (n >= N) continue;
    const int s = sibling(a, n);
    if (s != of) {
      of = s;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const bf16x8v v = ends::load8v(
            a.t + ((int64_t)s * M + min(m0 + i * 16 + fr, M - 1)) * 16 + at);
        tx[i] = fk < 2 ? v : none;
      }
      __builtin_amdgcn_s_waitcnt(loaded);
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + i * 16 + fr;
      const f32x4v d = product(bw[j], tx[i]);
      float f[4];
      take(f, acc[i][j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] += a.scale * d[e];
      const u32x2v now = packed(f);
      if (j % 2 == 0)
        held[i] = now;
      else
        put(y + (int64_t)m * N, held[i], now, n - 16, fk, N, m < M);
      if (j % 2 == 0 && (j + 1 == FN || n + 16 >= N))
        put(y + (int64_t)m * N, now, n, fk, N, m < M);
    }
  }
}

// Four waves, each a quarter of a tile of BM rows of x and BN rows of W: one wave
// a SIMD, whose 512 registers hold the sums and two sets of operands. K goes by
// 64 columns (a K-tile), through SX buffers of x and SW of W in LDS, straight
// from memory. A row of a buffer has 128 bytes; its pieces of 16 lie at their
// index ^ (row / 2) % 8, so that the operands of 16 rows spread over the banks.
//
// A K-tile is 2 F slots of a matrix instruction and what is issued beside it,
// so that no unit gets a burst (loads all at once, in half of the slots, took
// 103 us where these take 79, of 512 x 22016 x 4096): in the first half the
// operands of the second are read; from slot B1, when all waves have read theirs
// and the buffer is free, it is filled for the K-tile SX (SW) on; from slot B2,
// when the next K-tile is there, that one's first operands are read.
//
// A slot is 16 clocks, in which a wave issues three instructions beside the product.
// So a load has one beside it (mma_load), and what its addresses take, some 30
// scalar instructions a K-tile, is spread over the slots in front of B1 instead of
// standing before the first (pinned(); us of normal data and of zeros, before and
// now: 2048 x 12288 x 4096 165 and 162, 132 and 128; 7931 x 28672 x 4096 with the
// gated unit 1334 and 1305, 1044 and 1005; 2048 x 22016 x 4096 279 and 273, 227 and
// 219). With wider stores a step of llama2-7b, 4 x 512 tokens, takes 59.0 ms, 60.5
// before.
//
// Workgroups stay for all of their tiles, and the buffers are filled for the
// next one during the end of the one before. Tiles go to XCDs in runs, down
// bands of 8, so that those that run together share rows in its L2 (7931 x 28672
// x 4096: 1432 us down all rows and one tile a workgroup, 1330 so).
//
// DOWN: W is [K, N] and lies in LDS as it does in memory, a row of BN columns for
// each of a K-tile's 64; ds_read_b64_tr takes operands out of it, four of a column
// each. Pieces of 32 bytes lie at their index ^ (row % 4 + row / 8 % 2 * 4), so that
// the eight rows that half a wave reads spread over the banks.
//
// Its adapters are one K-tile more, the columns of t_i and the rows of A_i side by
// side (and zeros): no pass over y, and sums that are rounded once. With the pass
// (8 to 20 us), the library took 359 us for 2048 x 22016 to 4096 columns in its best
// form, two fp32 halves and their sum, and this takes 297 (1245 TFLOP/s; two parts
// of 256 x 256, bound by power: 1.7 GHz); a step of llama2-7b, 4 x 512 tokens, 67.0 ms
// before and 63.3 now.
template <int BM, int BN, int WR, int WC, int SX, int SW, Kind KIND, bool DOWN>
__global__ __launch_bounds__(WR * WC * 64, 1) void gemm_tiles_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ w,
    void *__restrict__ y, int M, int N, int K, int tm, int tn, int kt, int first,
    Adapters lora) {
  constexpr bool GLU = KIND == SILU || KIND == GELU;
  static_assert(!DOWN || KIND == PLAIN || KIND == PARTS, "ends");
  static_assert(!DOWN || ((BN == 128 || BN == 256) && WR * WC == 4),
                "siblings of a load");
  constexpr int WAVES = WR * WC, FM = BM / WR / 16, FN = BN / WC / 16;
  constexpr int LOADS = (BM + BN) / 8 / WAVES;      // of a wave and K-tile
  constexpr int XL = BM / 8 / WAVES, WL = LOADS - XL;
  constexpr int XS = BM * 128, WS = BN * 128;       // bytes of a buffer
  static_assert(SW == SX || SW == SX + 1, "buffers");
  static_assert(!GLU || FN % 2 == 0, "pairs");
  static_assert(BN % (8 * WAVES) == 0 && BM % (8 * WAVES) == 0, "loads");
  extern __shared__ __attribute__((aligned(128))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid / WC, wn = wid % WC;

  // this workgroup's tiles: every per-th of its XCD's
  const int nwg = tm * tn, xcd = blockIdx.x % 8;
  const int q8 = nwg / 8, r8 = nwg % 8;
  const int begin = xcd * q8 + min(xcd, r8);
  const int end = begin + q8 + (xcd < r8);
  const int per = (gridDim.x + 7 - xcd) / 8;
  int at = begin + blockIdx.x / 8;
  if (at >= end) return;
  // K-tiles of this part, and of them those of x and W
  const int kb = blockIdx.y * kt, kw = min(kt, K / 64 - kb);
  const int kn =
      kw + (DOWN && lora.n > 0 && blockIdx.y + 1 == gridDim.y ? 1 : 0);

  struct Place { int m0, n0; u32x4v rx, rw; unsigned sx, sw; };
  auto place = [&](int at) {
    Place p;
    const int band = at / (8 * tn), in = at % (8 * tn);
    const int rows = min(8, tm - band * 8);
    p.m0 = (band * 8 + in % rows) * BM;
    p.n0 = first + in / rows * BN;
    auto rows_of = [&](const uint16_t *base, int row, int rows) {
      return buffer(base + (int64_t)row * K, (uint32_t)rows * (uint32_t)K * 2);
    };
    p.rx = rows_of(x, p.m0, min(M - p.m0, BM));
    if constexpr (!DOWN)
      p.rw = GLU ? rows_of(w, p.n0 / 2, N - p.n0 / 2)
                 : rows_of(w, p.n0, min(N - p.n0, BN));
    return p;
  };
  Place here = place(at);

  unsigned voff[LOADS];
  auto row_of = [&](int i) { return (i * WAVES + wid) * 8 + (lane >> 3); };
  auto offsets_x = [&] {
#pragma unroll
    for (int i = 0; i < XL; ++i)
      voff[i] = (unsigned)row_of(i) * (unsigned)(K * 2) +
                ((lane & 7) ^ ((row_of(i) >> 1) & 7)) * 16;
  };
  // DOWN: a wave's load is of 64 / PR rows of PR pieces
  constexpr int PR = BN / 8;
  auto down_row = [&](int i) {
    return ((i - XL) * WAVES + wid) * (64 / PR) + lane / PR;
  };
  auto down_column = [&](int i) {
    const int k = down_row(i);
    return ((lane % PR) ^ ((k & 3) << 1 | (k >> 3 & 1) << 3)) * 8;
  };
  auto offsets_w = [&] {
#pragma unroll
    for (int i = XL; i < LOADS; ++i) {
      if (DOWN) {
        voff[i] = (unsigned)(down_row(i) * N + down_column(i)) * 2;
        continue;
      }
      const int row = row_of(i), c = (lane & 7) ^ ((row >> 1) & 7);
      int from = row - BM;
      if (GLU) {                        // a wave's gates, then its units
        const int in = from % (FN * 16);
        from = from / (FN * 16) * (FN * 8) + in % (FN * 8) +
               (in < FN * 8 ? 0 : N / 2);
      }
      voff[i] = (unsigned)from * (unsigned)(K * 2) + c * 16;
    }
  };
  offsets_x();
  offsets_w();
  // What K-tile t of x and of W is loaded from: by its first column; W, DOWN, as a
  // buffer of its rows, what is past them being past the buffer.
  auto aim_x = [&](Place &p, int t) {
    p.sx = (unsigned)(kb + t) * 128;
    if constexpr (DOWN) {
      if (t == kw) {
        p.sx = 0;
        p.rx = buffer(lora.t + (int64_t)p.m0 * 16,
                      (uint32_t)(lora.n * M - p.m0) * 32);
#pragma unroll
        for (int i = 0; i < XL; ++i) {
          const int row = row_of(i), c = (lane & 7) ^ ((row >> 1) & 7);
          voff[i] = (c >> 1) < lora.n
                        ? (unsigned)((c >> 1) * M + row) * 32 + (c & 1) * 16
                        : NOWHERE;
        }
      } else if (t == 0) {
        offsets_x();
      }
    }
  };
  auto aim_w = [&](Place &p, int t) {
    p.sw = (unsigned)(kb + t) * 128;
    if constexpr (DOWN) {
      p.sw = 0;
      p.rw = buffer(w + (int64_t)(kb + t) * 64 * N + p.n0,
                    (uint32_t)(64 * N - p.n0) * 2);
      if (t == kw) {
        p.rw = buffer(lora.b[0], NOWHERE);
#pragma unroll
        for (int i = XL; i < LOADS; ++i) {
          const int k = down_row(i), n = p.n0 + down_column(i), s = k >> 4;
          // selects, no branches, which would cut the loop in pieces
          const int from = ((s == 0) * lora.start[0] + (s == 1) * lora.start[1] +
                            (s == 2) * lora.start[2] + (k & 15) * N + n) * 2;
          const bool there = (s < lora.n) & (n < N);
          voff[i] = there ? (unsigned)from : NOWHERE;
        }
      } else if (t == 0) {
        offsets_w();
      }
    }
  };
  auto load = [&](const Place &p, int b, int i) {
    const unsigned at = (i * WAVES + wid) * 1024;
    if (i < XL)
      rb::lds_load(p.rx, voff[i], p.sx, b * XS + at);
    else
      rb::lds_load(p.rw, voff[i], p.sw, SX * XS + b * WS + at - XS);
  };
  f32x4v acc[FM][FN];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = (f32x4v)(0.0f);
  };
  clear();

  const int fr = lane & 15, fk = lane >> 4, sw = (fr >> 1) & 7;
  const int xa = (wm * FM * 16 + fr) * 128;
  const int wa = SX * XS + (wn * FN * 16 + fr) * 128;
  const int c0 = (fk ^ sw) * 16, c1 = ((fk + 4) ^ sw) * 16;
  bf16x8v fx[2][FM], fw[2][FN];
  // DOWN: this lane's 8 bytes of row 8 fk + fr / 4, by fragment
  int dw[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
    dw[j] = SX * XS + (fk * 8 + (fr >> 2)) * BN * 2 + (fr & 3) * 8 +
            ((wn * FN + j) ^ (fr >> 2 | (fk & 1) << 2)) * 32;
  auto frag = [&](int set, int bx, int bw, int i) {
    const char *b = smem + (set ? c1 : c0);
    if (DOWN && i < FN) {
      const char *p = smem + (dw[i] + bw * WS) + set * 32 * BN * 2;
      fw[set][i] = rb::lds_column8(p, p + 4 * BN * 2);
    } else if (i < FN)
      fw[set][i] =
          *reinterpret_cast<const bf16x8v *>(b + bw * WS + wa + i * 2048);
    else
      fx[set][i - FN] = *reinterpret_cast<const bf16x8v *>(
          b + bx * XS + xa + (i - FN) * 2048);
  };
  auto wait = [](auto n) {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(decltype(n)::value)
                 : "memory");
  };
#pragma unroll
  for (int u = -SW; u < 0; ++u) {
    Place p = here;
    aim_w(p, u + SW);
    if (u + SX >= 0) aim_x(p, u + SX);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      if (i >= XL) load(p, u + SW, i);
      else if (u + SX >= 0) load(p, u + SX, i);
  }
  constexpr int AHEAD = (SX - 2) * LOADS + (SW > SX ? WL : 0);
  wait(std::integral_constant<int, AHEAD + LOADS>());
#pragma unroll
  for (int i = 0; i < FM + FN; ++i) frag(0, 0, 0, i);

  constexpr int F = FM * FN, R = FM + FN;
  constexpr int B1 = F / 2 > R + 1 ? F / 2 : (R + 2 < F ? R + 2 : F - 1);
  constexpr int B2 = F + (F - 2 - F * 6 / 16 >= R ? F * 6 / 16
                          : F - R > 2 ? (F - R) / 2 : 1);
  constexpr int R1 = (B1 - 2) / R > 0 ? (B1 - 2) / R : 1;
  constexpr int R2 = (2 * F - B2 - 1) / R > 0 ? (2 * F - B2 - 1) / R : 1;
  constexpr int D = (2 * F - B1) / LOADS;
  constexpr int BEFORE =
      (B2 - B1 + D - 1) / D < LOADS ? (B2 - B1 + D - 1) / D : LOADS;
  // slots for what the loads' addresses take
  constexpr int A = 1, AD = (B1 - 1 - A) / 5;
  static_assert(D > 0 && AD > 0 && (R - 1) * R1 < B1 && B2 + 1 + (R - 1) * R2 < 2 * F,
                "slots");
  int bx = 0, bw = 0;
  while (true) {
    const int then = at + per;
    const bool more = then < end;
    const Place next = more ? place(then) : here;
    for (int t = 0; t < kn; ++t) {
      int nx, nw;
      unsigned lx, lw;
      Place p;                        // of the K-tiles that are fetched now
      auto slot = [&](auto at) __attribute__((always_inline)) {
        constexpr int q = decltype(at)::value;
        constexpr int set = q / F, i = q / FN % FM, j = q % FN;
        if constexpr (q == A) {
          const int u = pinned(t + SX);
#pragma unroll
          for (int e = 0; e < 3; ++e) p.rx[e] = u < kn ? here.rx[e] : next.rx[e];
          p.rx[3] = here.rx[3];
          p.m0 = u < kn ? here.m0 : next.m0;
        }
        if constexpr (q == A + AD) {
          const int u = pinned(t + SX);
          aim_x(p, u < kn ? u : u - kn);
        }
        if constexpr (q == A + 2 * AD) {
          lx = pinned(bx) * XS + wid * 1024;
          lw = SX * XS - XS + bw * WS + wid * 1024;
        }
        if constexpr (q == A + 3 * AD) {
          const int u = pinned(t + SW);
#pragma unroll
          for (int e = 0; e < 3; ++e) p.rw[e] = u < kn ? here.rw[e] : next.rw[e];
          p.rw[3] = here.rw[3];
          p.n0 = u < kn ? here.n0 : next.n0;
        }
        if constexpr (q == A + 4 * AD) {
          const int u = pinned(t + SW);
          aim_w(p, u < kn ? u : u - kn);
        }
        if constexpr (q == A + 5 * AD) {
          nx = pinned(bx + 1), nw = pinned(bw + 1);
          nx = nx == SX ? 0 : nx;
          nw = nw == SW ? 0 : nw;
        }
        if constexpr (q == B1)
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if constexpr (q == B2) wait(std::integral_constant<int, AHEAD + BEFORE>());
        if constexpr (q >= B1 && (q - B1) % D == 0 && (q - B1) / D < LOADS) {
          constexpr int l = (q - B1) / D;
          mma_load<l * WAVES * 1024>(
              acc[i][j], fw[set][j], fx[set][i], l < XL ? p.rx : p.rw,
              voff[l], l < XL ? p.sx : p.sw, l < XL ? lx : lw);
        } else {
          mma(acc[i][j], fw[set][j], fx[set][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (q % R1 == 0 && q / R1 < R) frag(1, bx, bw, q / R1);
        if constexpr (q > B2 && (q - B2 - 1) % R2 == 0 && (q - B2 - 1) / R2 < R)
          frag(0, nx, nw, (q - B2 - 1) / R2);
        __builtin_amdgcn_sched_barrier(0);
      };
      each<2 * F>(slot);
      bx = nx;
      bw = nw;
      settle(__builtin_amdgcn_readfirstlane(kn - 1 - t));
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (KIND == LORA)
      end_lora<FM, FN>(lora, acc, (uint16_t *)y, here.m0 + wm * FM * 16,
                       here.n0 + wn * FN * 16, fr, fk, M, N);
    else
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = here.m0 + (wm * FM + i) * 16 + fr;
      __builtin_amdgcn_sched_barrier(0);
      constexpr int RESULTS = GLU ? FN / 2 : FN;
      const int n0 = (GLU ? here.n0 / 2 : here.n0) + wn * RESULTS * 16;
      const int cols = GLU ? N / 2 : N;
      u32x2v held = {};
#pragma unroll
      for (int j = 0; j < RESULTS; ++j) {
        float f[4];
        take(f, acc[i][j]);
        if constexpr (KIND == PARTS) {
          const int n = n0 + j * 16 + fk * 4;
          if (m < M && n < N)
            *reinterpret_cast<f32x4v *>(
                (float *)y + ((int64_t)blockIdx.y * M + m) * N + n) =
                (f32x4v){f[0], f[1], f[2], f[3]};
        } else {
          if constexpr (GLU) {
            float u[4];
            take(u, acc[i][j + FN / 2]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              f[e] = ends::gate(f[e], u[e], KIND == GELU);
          }
          uint16_t *row = (uint16_t *)y + (int64_t)m * cols;
          if (j % 2 == 1)
            put(row, held, packed(f), n0 + j * 16 - 16, fk, cols, m < M);
          else if (j + 1 == RESULTS)
            put(row, packed(f), n0 + j * 16, fk, cols, m < M);
          held = packed(f);
        }
      }
    }
    if (!more) break;
    clear();
    asm volatile("s_nop 7" ::: "memory");
    at = then;
    here = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace tiles

namespace {

using tiles::Kind;

// What a tile takes in us, fitted to products of 129 to 8192 rows: a K-tile, and
// begin and end. Small ones are bound by L2, at 32 and 40 kB a K-tile.
struct Tile {
  int bm, bn;
  double step, rest;
};

constexpr Tile TILES[] = {{256, 256, 1.40, 7.0}, {192, 256, 1.12, 6.5},
                          {256, 192, 1.13, 6.5}, {256, 128, 0.78, 6.0},
                          {128, 256, 0.80, 6.0}, {128, 192, 0.74, 5.0},
                          {128, 128, 0.54, 5.0}};
constexpr int N_TILES = sizeof(TILES) / sizeof(TILES[0]), MAX_PARTS = 4;

// Columns (of W's rows) up to `split` in tiles of `tile`, the others in `rest`;
// split 0: all in `tile`.
struct Choice {
  int tile = -1, parts = 1, rest = -1;
  int64_t split = 0;
  double us = 1e30;
};

// Whether each of `parts` has K-tiles enough for the buffers.
bool divides(int64_t K, int parts) {
  const int64_t all = K / 64, each = (all + parts - 1) / parts;
  return all - (parts - 1) * each >= 4;
}

// The fastest by these times: rounds of 256 workgroups, and fp32 parts written
// and read at 5 TB/s.
Choice choose(int64_t M, int64_t N, int64_t K, int max_parts, int only) {
  Choice best;
  for (int v = 0; v < N_TILES; ++v) {
    if (only >= 0 && v != only) continue;
    const Tile &t = TILES[v];
    const int64_t n = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn);
    for (int p = 1; p <= max_parts; ++p) {
      if (!divides(K, p)) continue;
      const int64_t rounds = (n * p + 255) / 256;
      const double steps = (double)((K / 64 + p - 1) / p);
      double us = rounds * steps * t.step + t.rest * (1 + 0.3 * (rounds - 1));
      if (p > 1) us += p * M * N * 8 / 5e6;
      if (us < best.us) best = {v, p, -1, 0, us};
    }
  }
  return best;
}

// choose(), or whole rounds of a tile and the rest in a launch of its own, where
// a round that is nearly empty would follow (us with the gated unit, in one, in
// two, and the library's product and the unit: 700 x 22016 x 4096 134, 125 and
// 151, 2200 x 22016 x 4096 362, 309 and 330, 1800 x 28672 x 4096 387, 337 and 354,
// 6500 x 28672 x 4096 1127, 1093 and 1283).
Choice choose_two(int64_t M, int64_t N, int64_t K) {
  Choice best = choose(M, N, K, 1, -1);
  for (int v = 0; v < N_TILES; ++v) {
    const Tile &t = TILES[v];
    const int64_t tm = (M + t.bm - 1) / t.bm, tn = (N + t.bn - 1) / t.bn;
    const int64_t rounds = tm * tn / 256, cols = rounds * 256 / tm;
    if (rounds == 0 || cols >= tn) continue;
    const Choice rest = choose(M, N - cols * t.bn, K, 1, -1);
    const double us = rounds * (K / 64) * t.step +
                      t.rest * (1 + 0.3 * (rounds - 1)) + rest.us;
    if (us + 3 < best.us) best = {v, 1, rest.tile, cols * t.bn, us + 3};
  }
  return best;
}

// The same for W [K, N], in a fine-tune's steps, whose products keep the chip so
// busy that it lowers its clock (2.4 GHz to 1.7): a K-tile takes `few` us where up
// to half of the CUs have a workgroup, `all` where each has one. Fitted to 64 to
// 8192 rows. Parts are added up by a launch of their own.
struct DownTile { double few, all; };
constexpr DownTile DOWN_TILES[N_TILES] = {{1.29, 1.54}, {1.09, 1.24}, {}, {.79, .91},
                                          {.83, .94}, {}, {.57, .585}};

double down_us(int v, int64_t M, int64_t N, int64_t K, int p) {
  const Tile &t = TILES[v];
  const int64_t n = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn) * p;
  const int64_t rounds = (n + 255) / 256;
  const double fill = (double)n / (rounds * 256);
  const DownTile &d = DOWN_TILES[v];
  const double step = d.few + (d.all - d.few) * std::max(0.0, 2 * fill - 1);
  const double us = rounds * (double)((K / 64 + p - 1) / p + 1) * step +
                    t.rest * (1 + 0.3 * (rounds - 1));
  return p == 1 ? us : us + M * N * (p * 8 + 2) / 5e6 + 5.0;
}

Choice choose_down(int64_t M, int64_t N, int64_t K, int max_parts, int only) {
  Choice best;
  auto all = [&](int64_t cols, int most, auto &&take) {
    for (int v = 0; v < N_TILES; ++v) {
      if (TILES[v].bn == 192 || (only >= 0 && v != only)) continue;
      for (int p = 1; p <= most; ++p)
        if (divides(K, p)) take(v, p, down_us(v, M, cols, K, p));
    }
  };
  all(N, max_parts, [&](int v, int p, double us) {
    if (us < best.us) best = {v, p, -1, 0, us};
  });
  if (only >= 0) return best;
  // whole rounds of a tile, and the rest in a launch of its own
  all(N, 1, [&](int v, int, double) {
    const Tile &t = TILES[v];
    const int64_t tm = (M + t.bm - 1) / t.bm, tn = (N + t.bn - 1) / t.bn;
    const int64_t cols = tm * tn / 256 * 256 / tm;
    if (cols == 0 || cols >= tn) return;
    const double first = down_us(v, M, cols * t.bn, K, 1);
    all(N - cols * t.bn, 1, [&](int r, int, double us) {
      if (first + us + 3 < best.us)
        best = {v, 1, r, cols * t.bn, first + us + 3};
    });
  });
  return best;
}

template <int BM, int BN, int SX, int SW, Kind KIND, bool DOWN>
void launch(const at::Tensor &x, const at::Tensor &w, at::Tensor &y, int parts,
            int64_t first, int64_t last, const tiles::Adapters &lora) {
  auto kernel = tiles::gemm_tiles_kernel<BM, BN, 2, 2, SX, SW, KIND, DOWN>;
  constexpr int lds = (SX * BM + SW * BN) * 128;
  static const bool once =
      hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds) ==
      hipSuccess;
  TORCH_CHECK(once, "tile_gemm: LDS size");
  const int M = (int)x.size(0), K = (int)x.size(1);
  const int N = (int)w.size(DOWN ? 1 : 0);
  const int tm = (M + BM - 1) / BM, tn = (int)((last - first + BN - 1) / BN);
  const int kt = (K / 64 + parts - 1) / parts;
  hipLaunchKernelGGL(kernel, dim3(std::min(tm * tn, 256), parts), dim3(256),
                     lds, at::cuda::getCurrentHIPStream(),
                     (const uint16_t *)x.data_ptr(),
                     (const uint16_t *)w.data_ptr(), y.data_ptr(), M, N, K, tm,
                     tn, kt, (int)first, lora);
  C10_CUDA_KERNEL_LAUNCH_CHECK();
}

template <Kind KIND, bool DOWN = false>
void run(int tile, const at::Tensor &x, const at::Tensor &w, at::Tensor &y,
         int parts, int64_t first, int64_t last,
         const tiles::Adapters &lora = {}) {
  auto go = [&](auto bm, auto bn, auto sx, auto sw) {
    if constexpr (!DOWN || bn() != 192)
      launch<bm(), bn(), sx(), sw(), KIND, DOWN>(x, w, y, parts, first, last,
                                                 lora);
  };
  using std::integral_constant;
#define TILE(bm, bn, sx, sw)                                             \
  return go(integral_constant<int, bm>(), integral_constant<int, bn>(), \
            integral_constant<int, sx>(), integral_constant<int, sw>())
  switch (tile) {
    case 0: TILE(256, 256, 2, 2);
    case 1: TILE(192, 256, 2, 2);
    case 2: TILE(256, 192, 2, 2);
    case 3: TILE(256, 128, 3, 3);
    case 4: TILE(128, 256, 2, 3);
    case 5: TILE(128, 192, 3, 4);
    default: TILE(128, 128, 3, 4);
  }
#undef TILE
}

bool fits(const at::Tensor &t) {
  return t.is_cuda() && t.dim() == 2 && t.is_contiguous() &&
         t.scalar_type() == at::kBFloat16 && t.size(0) > 0 &&
         t.size(0) < (1 << 24) &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

}  // namespace

// Whether tile_gemm takes x and W (with `glu`, W = [G ; U]).
bool tile_gemm_takes(at::Tensor x, at::Tensor w, bool glu) {
  return fits(x) && fits(w) && x.size(1) == w.size(1) &&
         x.device() == w.device() && x.size(1) % 64 == 0 &&
         x.size(1) >= 256 && x.size(1) <= (1 << 20) &&
         w.size(0) % (glu ? 8 : 4) == 0 &&
         (!glu || w.size(0) * w.size(1) * 2 < ((int64_t)1 << 32));
}

// Whether a product of more than 320 rows is as good in tiles as in the library, which
// has tiles of 256 x 256 and others, is slow at columns that are no multiple of 256,
// and takes short sums (up to 512) long to begin and end.
//
// Up to one round of 256 x 256: where columns are a multiple, tiles that fill the CUs
// (85% of a round; small ones 70%), or whole bands of rows (1, 2, 4, 8) of which the
// library pads more than a tenth. us there and in tiles: 1021 x 12288 x 3072 65 and 59,
// 400 x 10240 x 4096 48 and 42, 512 x 12288 x 4096 55 and 53; not: 1280 x 4096 x 4096
// 47 and 49, 640 x 8192 x 3072 38 and 40, 330 x 8192 x 4096 33 and 35.
//
// More rounds: not where they are whole or nearly whole for the library (7931 x 6144 x
// 4096 275 and 283, 2048 x 8192 x 2560 65 and 69), nor of sums past 6144, which it
// takes as fast (mean 1.00 of 641 sizes).
//
// Of 15098 sizes, 321 to 24576 rows, 256 to 20480 columns and sums of 256 to 8192, 12347
// go by tiles: the mean is 0.87 of the library's time, 414 are slower by more than 3%
// and 106 by more than 6%. Of the others the mean would be 0.99, 917 and 414.
bool tile_gemm_pays(int64_t M, int64_t N, int64_t K) {
  const int64_t down = (M + 255) / 256, across = (N + 255) / 256;
  const int64_t all = down * across;
  if (M <= 320 || M > 24576 || N < 256 || N > 20480 || K < 256 || K > 8192 ||
      all < (K > 2048 ? 64 : 40))
    return false;
  if (K <= 512) return true;
  const bool padded = N % 256 != 0;
  const Choice c = choose_two(M, N, K);
  const Tile &t = TILES[c.tile];
  const bool large = t.bm == 256 && t.bn == 256;
  if (all <= 256) {
    if (c.rest >= 0 || padded || large) return c.rest < 0 && padded;
    const int64_t tm = (M + t.bm - 1) / t.bm, tn = (N + t.bn - 1) / t.bn;
    const int64_t slots = (tm * tn + 255) / 256 * 256;
    const double fill = (double)(M * N) / (double)(slots * t.bm * t.bn);
    if (t.bm == 128 && t.bn == 128) return K <= 2048 || fill >= 0.7;
    return fill >= 0.85 || (t.bm != 192 && 8 % tm == 0 &&
                            M * 10 < down * 2304 && tm * tn * 4 >= slots * 3);
  }
  if (all % 256 == 0) return padded && K <= 6144;
  if (down <= 5) return true;
  if (K > 6144) return false;
  const int64_t step = 256 / down;      // columns of tiles in a round
  if (c.rest >= 0) return down * step < 256;
  return padded || !large || down * step < 230 || across % step != 0;
}

// Parts that tile_gemm makes of sums where it may.
int64_t tile_gemm_parts(int64_t M, int64_t N, int64_t K) {
  return choose(M, N, K, MAX_PARTS, -1).parts;
}

// What tile_gemm and tile_lora run: tile, parts, the tile of the columns from
// `split` on (-1: none) and split.
std::vector<int64_t> tile_gemm_choice(int64_t M, int64_t N, int64_t K,
                                      int64_t max_parts) {
  const Choice c = max_parts > 1 ? choose(M, N, K, (int)max_parts, -1)
                                 : choose_two(M, N, K);
  return {c.tile, c.parts, c.rest, c.split};
}

// x W^T: bf16 [M, N]; where max_parts > 1, possibly fp32 parts [P, M, N] of the
// sums. glu 1 (SiLU) or 2 (tanh-GELU): act(x G^T) * (x U^T) of W = [G ; U]. tile
// and parts: the choice of a test.
at::Tensor tile_gemm(at::Tensor x, at::Tensor w, int64_t max_parts, int64_t glu,
                     int64_t tile, int64_t parts) {
  TORCH_CHECK(tile_gemm_takes(x, w, glu != 0) && glu >= 0 && glu <= 2 &&
              (glu == 0 || (max_parts <= 1 && parts <= 1)) &&
              tile < N_TILES && max_parts <= MAX_PARTS && parts <= MAX_PARTS,
              "tile_gemm: x ", x.sizes(), ", W ", w.sizes());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  Choice c = max_parts > 1 || tile >= 0 ? choose(M, N, K, (int)max_parts,
                                                 (int)tile)
                                        : choose_two(M, N, K);
  if (parts > 0) c.parts = (int)parts;
  TORCH_CHECK(divides(K, c.parts), "tile_gemm: parts");
  if (c.parts > 1) {
    auto y = at::empty({c.parts, M, N}, x.options().dtype(at::kFloat));
    run<tiles::PARTS>(c.tile, x, w, y, c.parts, 0, N);
    return y;
  }
  auto y = at::empty({M, glu ? N / 2 : N}, x.options());
  auto go = [&](int t, int64_t first, int64_t last) {
    if (glu == 1) run<tiles::SILU>(t, x, w, y, 1, first, last);
    else if (glu == 2) run<tiles::GELU>(t, x, w, y, 1, first, last);
    else run<tiles::PLAIN>(t, x, w, y, 1, first, last);
  };
  if (c.split > 0) {
    go(c.tile, 0, c.split);
    go(c.rest, c.split, N);
  } else {
    go(c.tile, 0, N);
  }
  return y;
}

// Adapters of rank 16 as the tiles read them: t [n, M, 16], and matrices whose
// dimension `wide` is 16.
static tiles::Adapters tile_adapters(const at::Tensor &x, const at::Tensor &t,
                                     const std::vector<at::Tensor> &ms,
                                     int wide) {
  tiles::Adapters a{};
  a.n = (int)ms.size();
  a.scale = 1.0f;
  TORCH_CHECK(a.n <= 3, "tiles: at most 3 adapters");
  auto adapter = [&](const at::Tensor &m, int d) {
    TORCH_CHECK(m.is_contiguous() && m.device() == x.device() &&
                m.scalar_type() == at::kBFloat16 && m.size(d) == 16 &&
                reinterpret_cast<uintptr_t>(m.data_ptr()) % 16 == 0,
                "tiles: adapters of rank 16, bf16");
    return (const uint16_t *)m.data_ptr();
  };
  if (a.n == 0) return a;
  TORCH_CHECK(t.dim() == 3 && t.size(0) == a.n && t.size(1) == x.size(0) &&
              a.n * t.size(1) * 32 < (int64_t)tiles::NOWHERE,
              "tiles: t [n, M, 16]");
  a.t = adapter(t, 2);
  for (int i = 0; i < a.n; ++i) {
    TORCH_CHECK(ms[i].dim() == 2, "tiles: adapters' matrices");
    a.b[i] = adapter(ms[i], wide);
  }
  return a;
}

// x W^T + scale t_i B_i^T of one to three siblings side by side: t [n, M, 16], B_i
// [columns of i, 16].
at::Tensor tile_lora(at::Tensor x, at::Tensor w, at::Tensor t,
                     std::vector<at::Tensor> bs, double scale, int64_t tile) {
  const int64_t M = x.size(0), N = w.size(0);
  TORCH_CHECK(tile_gemm_takes(x, w, false) && tile < N_TILES && !bs.empty(),
              "tile_lora: x ", x.sizes(), ", W ", w.sizes());
  tiles::Adapters a = tile_adapters(x, t, bs, 1);
  int64_t at = 0;
  for (int i = 0; i < a.n; ++i) {
    TORCH_CHECK(bs[i].size(0) % 16 == 0 && bs[i].size(0) > 0,
                "tile_lora: columns");
    a.start[i] = (int)at;
    at += bs[i].size(0);
  }
  TORCH_CHECK(at == N, "tile_lora: columns of the siblings");
  a.scale = (float)scale;
  const Choice c = tile >= 0 ? choose(M, N, x.size(1), 1, (int)tile)
                             : choose_two(M, N, x.size(1));
  auto y = at::empty({M, N}, x.options());
  if (c.split > 0) {
    run<tiles::LORA>(c.tile, x, w, y, 1, 0, c.split, a);
    run<tiles::LORA>(c.rest, x, w, y, 1, c.split, N, a);
  } else {
    run<tiles::LORA>(c.tile, x, w, y, 1, 0, N, a);
  }
  return y;
}

// Whether tile_gemm_down takes x [M, K] and W [K, N].
bool tile_gemm_down_takes(at::Tensor x, at::Tensor w) {
  return fits(x) && fits(w) && x.size(1) == w.size(0) &&
         x.device() == w.device() && x.size(1) % 64 == 0 &&
         x.size(1) >= 256 && x.size(1) <= (1 << 20) && w.size(1) % 8 == 0 &&
         w.size(1) < (1 << 22);
}

// Whether tile_gemm_down, with the parts' sum, is as good as the library and a pass
// for the adapters: 300 rows of 12288 to 4096 columns 56 us, 118 there, 2048 rows 172
// and 198; of 22016 to 4096 512 rows 99 and 202, 2048 297 and 359; of 4096 to 11008
// 2048 rows 168 and 179. It is not (us there and here)
//  - of a few rows, and of results of less than 64K in narrow columns, whose sums the
//    library splits further (33 x 768 of 8192 19 and 23, 129 x 256 of 4096 13 and 17);
//  - of small results and short sums, where begin and end count (300 x 1024 of 1024
//    12.2 and 13.6, 400 x 2048 of 2048 17.5 and 19.5);
//  - where one launch leaves CUs idle, of sums that are not much longer than the result
//    is wide (2500 x 4096 of 12288 213 and 238, 1100 x 4096 of 4096 51 and 56, 2500 x
//    2048 of 5632 68 and 75, 1100 x 8192 of 8192 139 and 148).
// Of 17362 other sizes, 33 to 24576 rows of 64 to 20480 columns and sums of 256 to 57344,
// with one adapter, the mean is 0.69 of the library's time; 196 are slower by more than
// 3%, and of those of 2048 columns and more 73 of 9476: long sums whose tiles are as many
// and as large as the library's (3001 x 4096 of 28672 556 and 579), which it makes up
// for in a step (two adapters, lower clocks: mistral-7b, 3001 tokens, 96.3 ms and 97.1
// with the library there).
bool tile_gemm_down_pays(int64_t M, int64_t N, int64_t K) {
  if (M <= 32 || M > 24576 || N < 64 || K > 57344) return false;
  const Choice c = choose_down(M, N, K, MAX_PARTS, -1);
  if (c.tile < 0) return false;
  const Tile &t = TILES[c.tile];
  const int64_t tiles = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn);
  const int64_t rounds = (tiles + 255) / 256, all = M * N;
  const bool one = c.parts == 1 && c.rest < 0;
  if (N < 2048 && all < 65536 && K > 1024) return false;
  if (one && K > 512 && K <= 1024 && all >= 20000 && all < 500000) return false;
  if (K > 1024 && K <= 2048 && all >= 250000 && all < 1000000) return false;
  return !(M >= 1024 && one && tiles * 10 < rounds * 2304 && N <= K &&
           (N <= 4096 || K < 2 * N));
}

std::vector<int64_t> tile_gemm_down_choice(int64_t M, int64_t N, int64_t K,
                                           int64_t max_parts) {
  const Choice c = choose_down(M, N, K, (int)max_parts, -1);
  return {c.tile, c.parts, c.rest, c.split};
}

// x W + sum_i t_i A_i, W [K, N] and up to three adapters A_i [16, N], t [n, M, 16]:
// bf16 [M, N], or, where max_parts > 1, possibly fp32 parts [P, M, N] of the sums.
at::Tensor tile_gemm_down(at::Tensor x, at::Tensor w, at::Tensor t,
                          std::vector<at::Tensor> as, int64_t max_parts,
                          int64_t tile, int64_t parts) {
  TORCH_CHECK(tile_gemm_down_takes(x, w) && tile < N_TILES &&
              max_parts >= 1 && max_parts <= MAX_PARTS && parts <= MAX_PARTS &&
              (tile < 0 || TILES[tile].bn != 192),
              "tile_gemm_down: x ", x.sizes(), ", W ", w.sizes());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(1);
  tiles::Adapters a = tile_adapters(x, t, as, 0);
  for (const auto &m : as)
    TORCH_CHECK(m.size(1) == N, "tile_gemm_down: columns of A");
  // the kernel reads all A_i from the first in memory on, within 2 GiB
  at::Tensor near;
  if (a.n > 1) {
    int order[3] = {0, 1, 2};
    std::sort(order, order + a.n,
              [&](int i, int j) { return a.b[i] < a.b[j]; });
    if (a.b[order[a.n - 1]] + 16 * N - a.b[order[0]] >= (1 << 30)) {
      near = at::cat(as);
      for (int i = 0; i < a.n; ++i)
        a.b[i] = (const uint16_t *)near.data_ptr() + i * 16 * N;
      order[0] = 0;
    }
    const uint16_t *base = a.b[order[0]];
    for (int i = 0; i < a.n; ++i) a.start[i] = (int)(a.b[i] - base);
    a.b[0] = base;
  }
  Choice c = choose_down(M, N, K, (int)max_parts, (int)tile);
  if (parts > 0) c.parts = (int)parts;
  TORCH_CHECK(divides(K, c.parts), "tile_gemm_down: parts");
  if (c.parts > 1) {
    auto y = at::empty({c.parts, M, N}, x.options().dtype(at::kFloat));
    run<tiles::PARTS, true>(c.tile, x, w, y, c.parts, 0, N, a);
    return y;
  }
  auto y = at::empty({M, N}, x.options());
  if (c.split > 0) {
    run<tiles::PLAIN, true>(c.tile, x, w, y, 1, 0, c.split, a);
    run<tiles::PLAIN, true>(c.rest, x, w, y, 1, c.split, N, a);
  } else {
    run<tiles::PLAIN, true>(c.tile, x, w, y, 1, 0, N, a);
  }
  return y;
}
