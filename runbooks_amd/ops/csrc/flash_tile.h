// LDS tiles of the flash attention kernels (attention_prefill.hip,
// attention_bwd.hip): rows of DH bf16 values, loaded straight from memory
// (global_load_lds, 16 bytes a lane) and read both ways, by rows as MFMA
// operands along DH and by columns (ds_read_b64_tr_b16) as operands along the
// rows.
//
// Row r's 16-byte chunk c stands at chunk c ^ mix(r). A load writes 64
// consecutive chunks, so the mixing is done on the address it reads. With it
// the 16 rows of one chunk, which a row read takes, and the 4 rows of 4
// chunks, which a column read takes, fall on all 64 banks once.
#pragma once

#include <torch/extension.h>

#include <type_traits>
#include <utility>

#include "common.h"

namespace flash {

// Contiguous values may start anywhere; the kernels load 16 bytes at a time.
static inline at::Tensor aligned16(const at::Tensor &t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t;
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8v;
typedef __attribute__((ext_vector_type(16))) float f32x16v;
using rb::u32x4v;

constexpr int ROWS = 64;               // of a tile

// one v_cvt_pk_bf16_f32 (two scalar conversions take four instructions)
RB_DEV unsigned pack2(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2v;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2v;
  union { bf16x2v b; unsigned u; } c;
  c.b = __builtin_convertvector((f32x2v){lo, hi}, bf16x2v);
  return c.u;
}

// The order of a block's instructions: N products, an operand of each read from LDS
// AHEAD products before it. Left to itself the compiler has every product wait for a
// read of its own. us, 32 heads of 128, with that and without: 1021 tokens 21.5 and
// 22.9, 2000 (four waves of whole keys) 50 and 55.
template <int N, int AHEAD> RB_DEV void reads_ahead() {
  __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
  for (int i = 0; i < N - AHEAD; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
}

// f of 0 .. N - 1, known where it is compiled.
template <class F, int... Q>
RB_DEV void each_of(F &f, std::integer_sequence<int, Q...>) {
  (f(std::integral_constant<int, Q>()), ...);
}
template <int N, class F> RB_DEV void each(F &f) {
  each_of(f, std::make_integer_sequence<int, N>());
}

template <int DH> RB_DEV constexpr int mix(int row) {
  return DH == 64 ? ((row >> 1 & 1) << 2) | (row >> 2 & 3)
                  : ((row & 3) << 2) | (row >> 2 & 3);
}

template <int DH> constexpr int tile_bytes() { return ROWS * DH * 2; }

// Loads of a tile by NW waves: piece i of wave w is the kilobyte (1024 bytes
// of LDS) i * NW + w of the tile, STEP rows after the one before; mix() is
// linear in the bits of a row. Rows `stride` elements apart.
template <int DH, int NW> struct TileLoad {
  static constexpr int PIECES = tile_bytes<DH>() / 1024 / NW;
  static constexpr int CHUNKS = DH / 8;          // of a row
  static constexpr int STEP = NW * 64 / CHUNKS;
  unsigned at[PIECES];                           // bytes from a tile's first row
  int64_t stride;

  RB_DEV TileLoad(int wid, int lane, int64_t stride) : stride(stride) {
    const int piece = wid * 64 + lane;
    const int row = piece / CHUNKS, off = piece % CHUNKS ^ mix<DH>(row);
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      at[i] = (unsigned)(row + i * STEP) * (unsigned)(stride * 2) +
              (off ^ mix<DH>(i * STEP)) * 16;
  }

  // Rows r0 .. r0 + 63 of `rows` rows from `base` on; rows past the end are zeros.
  // `tile` is uniform. The caller waits (vmcnt): the compiler, which would wait for
  // all loads to LDS before the next read of it, does not see these. Addresses are
  // the tile's, in scalar registers, and these. us before, with loads that it saw
  // and addresses of each lane, and now: the forward of 7931 tokens, 16 heads of
  // 256 714 and 682, 5000 tokens, 16 heads of 64 81 and 79.
  RB_DEV void operator()(const uint16_t *base, int r0, int rows, char *tile,
                         int wid) const {
    const int n = min(rows - r0, ROWS);
    const u32x4v from = rb::buffer(
        base + r0 * stride, n > 0 ? (uint32_t)((n - 1) * stride + DH) * 2 : 0);
    const unsigned to = __builtin_amdgcn_readfirstlane(
        (unsigned)(size_t)(__attribute__((address_space(3))) char *)tile);
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      rb::lds_load(from, at[i], 0, to + (i * NW + wid) * 1024);
  }
};

// How a wave of 32 query rows from `wrow` on walks the tiles of its workgroup,
// all of which it waits for with the others: `full` tiles that all its rows see
// whole, then those up to key `last`. Rows past the end see none.
struct Walk { int full, last; };
__host__ __device__ constexpr Walk walk(int wrow, int rows) {
  return wrow < rows ? Walk{wrow / ROWS, wrow + 31} : Walk{0, -1};
}

// Operand of rows r0 .. r0 + 31 along columns 16 ks .. 16 ks + 15: element e
// of lane (hi, col) is row r0 + col, column 16 ks + 8 hi + e. r0 % 16 == 0.
template <int DH>
RB_DEV bf16x8v row_frag(const char *tile, int r0, int ks, int col, int hi) {
  return *reinterpret_cast<const bf16x8v *>(
      tile + (r0 + col) * (DH * 2) + ((ks * 2 + hi) ^ mix<DH>(col)) * 16);
}

// Operand of columns 32 dt .. 32 dt + 31 along rows r0 .. r0 + 15, in the order
// of a score tile's registers: element e of lane (hi, col) is column
// 32 dt + col, row r0 + 8 (e / 4) + 4 hi + e % 4; PLAIN: row r0 + 8 hi + e.
// r0 % 16 == 0.
template <int DH, bool PLAIN = false>
RB_DEV bf16x8v column_frag(const char *tile, int r0, int dt, int lane) {
  const int i = lane & 15, hi = lane >> 5;
  const int r = (PLAIN ? 8 : 4) * hi + (i >> 2), r2 = r + (PLAIN ? 4 : 8);
  const int chunk = dt * 4 + (lane >> 4 & 1) * 2 + (i >> 1 & 1);
  const char *lo = tile + (r0 + r) * (DH * 2) +
                   (chunk ^ mix<DH>(r)) * 16 + (i & 1) * 8;
  const char *up = tile + (r0 + r2) * (DH * 2) +
                   (chunk ^ mix<DH>(r2)) * 16 + (i & 1) * 8;
  return rb::lds_column8(lo, up);
}

// Eight values of a score tile's registers -> the other operand: rows in the order
// of the registers, as column_frag takes them; PLAIN: in their own, for which
// the halves of the wave exchange the middle ones of 16.
template <bool PLAIN = false>
RB_DEV bf16x8v score_frag(const f32x16v &p, int ks) {
  union { unsigned u[4]; bf16x8v v; } c;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    c.u[i] = pack2(p[ks * 8 + 2 * i], p[ks * 8 + 2 * i + 1]);
  if constexpr (PLAIN) {
    const auto a = __builtin_amdgcn_permlane32_swap(c.u[0], c.u[2], false,
                                                    false);
    const auto b = __builtin_amdgcn_permlane32_swap(c.u[1], c.u[3], false,
                                                    false);
    c.u[0] = a[0]; c.u[1] = b[0]; c.u[2] = a[1]; c.u[3] = b[1];
  }
  return c.v;
}

// Workgroup -> (tile, head, batch). Tiles of a causal triangle differ in
// length: the longest come first. The heads of one key/value head stay on one
// XCD, whose L2 then holds their keys, when those heads divide by the XCDs.
struct Place { int tile, head, batch; };
RB_DEV Place place(int id, int tiles, int heads, int kv, int batch,
                   bool longest_is_last) {
  const int per_tile = heads * batch;
  int t = id / per_tile, j = id % per_tile;
  if (longest_is_last) t = tiles - 1 - t;
  const int group = heads / kv;
  if (kv * batch % 8 == 0) {
    const int xcd = j % 8, k = j / 8;        // consecutive ids: next XCD
    const int pair = k / group * 8 + xcd;    // (batch, kv head)
    return {t, pair % kv * group + k % group, pair / kv};
  }
  return {t, j % heads, j / heads};
}

}  // namespace flash
