// Paged decode attention (one query token per sequence) for CDNA4 (gfx950).
//
// The serving hot loop: memory-bound on the KV read (HBM3E gives 6.6 TB/s to
// long reads that pass L2's older lines, 5.9 to others). Design, MI355X-first:
//  * wave64 split into lane groups, each of which owns one kv token at 16 bytes
//    a lane and load: 16 lanes for rows of 256 and 512 bytes (heads of 128 and
//    256), 8 for rows of 128 (heads of 64, up to two query heads a kv head) and
//    for e4m3, so every wave streams 4 or 8 contiguous KV rows at a time. (Heads
//    of 64 with four query heads or more keep 16 lanes of 8 bytes, for registers.)
//  * GQA/MQA-native: a workgroup handles one (seq, kv_head); its G query
//    heads share each K/V read (falcon-40b MQA G=16, llama2-70b G=8,
//    llama2-7b MHA G=1).
//  * flash-style online softmax entirely in registers; group partials
//    merged by lane permutations, wave partials via LDS.
//  * kv-split ("flash-decoding") for long sequences / small batch: grid z
//    = nsplit partitions, fp32 partials (m, l, acc) merged by a tiny
//    second kernel — sized so batch*Hkv*nsplit >> 256 CUs.
//
// q:       [B, Hq, Dh] bf16     out: [B, Hq, Dh] bf16
// caches:  [num_blocks, Hkv, BS, Dh] bf16 (see kvcache.hip)
// block_tables: [B, max_blocks] int32;  seq_lens: [B] int32
// partial: [B, Hq, nsplit, Dh + 2] fp32 workspace when nsplit > 1

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>
#include <type_traits>

#include "common.h"

int64_t paged_decode_parts(int64_t nsplit, int64_t longest, int64_t dh,
                           int64_t group, bool transposed);

namespace {

constexpr int BLOCK = 256;    // 4 waves
constexpr int NW = 4;

typedef __attribute__((ext_vector_type(8))) __bf16 rb_bf16x8v;
typedef __attribute__((ext_vector_type(2))) __bf16 rb_bf16x2v;
typedef __attribute__((ext_vector_type(4))) float rb_f32x4v;

RB_DEV unsigned rb_pack_bf16(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2v;
  union { rb_bf16x2v v; unsigned u; } c;
  c.v = __builtin_convertvector((f32x2v){lo, hi}, rb_bf16x2v);
  return c.u;
}

// one v_dot2_f32_bf16: c += a_pair . b_pair (packed bf16 pairs)
RB_DEV float rb_dot2(unsigned a, unsigned b, float c) {
  union { unsigned u; rb_bf16x2v v; } x, y;
  x.u = a;
  y.u = b;
  return __builtin_amdgcn_fdot2_f32_bf16(x.v, y.v, c, false);
}

// VE outputs of sequence b from column kk0 of a row (a multiple of VE, as VE is
// of 4) in the decode GEMM's operand layout, [K/16][2][32][8].
template <int VE>
RB_DEV void store_operand(uint16_t *swz, int kk0, int b, const float *v,
                          float scale) {
  constexpr int W = VE < 8 ? VE : 8;
#pragma unroll
  for (int e0 = 0; e0 < VE; e0 += W) {
    const int kk = kk0 + e0;
    uint16_t *p =
        swz + (kk >> 4) * 512 + ((kk >> 3) & 1) * 256 + b * 8 + (kk & 7);
#pragma unroll
    for (int e = 0; e < W; ++e) p[e] = rb::f32_to_bf16(v[e0 + e] * scale);
  }
}

// What a workgroup of a grid (B, Hkv, splits) takes. Workgroups 256 apart in launch
// order share a CU; in plain order those would be heads of one sequence wherever
// the batch divides 256, and the CUs of the longest ones would run long after the
// others.
struct Place { int b, h, split, len, start; };

// The sequences are shifted with head and split, once around over the whole grid:
// a CU gets sequences spread evenly over the batch.
RB_DEV int shifted() {
  const unsigned y = blockIdx.y + gridDim.y * blockIdx.z;
  return (int)((blockIdx.x + y * gridDim.x / (gridDim.y * gridDim.z)) %
               gridDim.x);
}

RB_DEV Place shifted_place(const int32_t *lens, const int32_t *starts) {
  const int b = shifted();
  return {b, (int)blockIdx.y, (int)blockIdx.z, lens[b],
          starts != nullptr ? starts[b] : 0};
}

// The longest sequences first, so that none is begun late, and every other 256
// workgroups the other way round, so that a CU that has a long one gets a short one
// with it. Up to 64 sequences, whose lengths one wave compares for all (B steps of
// three instructions; all waves of a CU together took 0.8 us).
//
// us by shifts and sorted, 32 heads of 128: 32 sequences of 129 to 2015 tokens 101
// and 94 (6.0 TB/s), 16 of 800 to 3900 in e4m3 66 and 62, 64 of 100 to 1200 120 and 113,
// 32 of 1072 each 93.5 and 93.1; 8 kv heads of 128 with four queries each: 64 of 1000 to
// 4003 122 and 106 (6.2 TB/s), 32 of 100 to 4000 in two parts 63 and 52; 16 heads of 256:
// 7 of 90 to 1801 in parts 27.4 and 26.2, 16 of 100 to 2000 57.8 and 58.1.
// Where nothing is uneven that cost 0.3 to 0.8 us, so lengths within 128 tokens of the
// first one's go by shifts, and what a wave has loaded is not loaded again (us of a
// table of 4096 by shifts alone, sorted, and so: 32 of 100 13.7, 14.4 and 13.9, 64 of
// 500 with 8 kv heads 26.9, 27.7 and 26.8, 16 of 100 with 12 heads of 64 9.0, 9.8 and
// 9.2; 32 of 20 to 500 31.2, 29.7 and 29.5). Tables of up to 512 tokens go by shifts,
// as do up to four sequences, whose parts are all begun at once (of two and three
// within 1% either way), and more than 64, for which a wave has no lanes.
RB_DEV Place sorted_place(const int32_t *lens, const int32_t *starts) {
  const int B = gridDim.x, hkv = gridDim.y, of_each = hkv * gridDim.z;
  const int lane = threadIdx.x & 63;
  int len = 0, start = 0;
  if (lane < B) {
    len = lens[lane];
    if (starts != nullptr) start = starts[lane];
  }
  const int sees = max(0, len - start);
  const int off = sees - __builtin_amdgcn_readfirstlane(sees);
  if (!__any(lane < B && (off > 128 || off < -128))) {
    const int b = shifted();
    return {b, (int)blockIdx.y, (int)blockIdx.z,
            __builtin_amdgcn_readlane(len, b),
            __builtin_amdgcn_readlane(start, b)};
  }
  __shared__ int found;
  const int all = B * of_each;
  const int id = blockIdx.x + B * (blockIdx.y + hkv * blockIdx.z);
  const int round = id & ~255;
  const int at = id & 256 ? round + min(256, all - round) - 1 - (id & 255) : id;
  if (threadIdx.x < 64) {
    // all of them different
    const int key = lane < B ? sees * 64 + lane : -1;
    int longer = 0;
#pragma unroll
    for (int i0 = 0; i0 < 64; i0 += 8)
      if (i0 < B)
#pragma unroll
        for (int i = i0; i < i0 + 8; ++i)
          longer += __builtin_amdgcn_readlane(key, i) > key;
    if (lane < B && longer == at / of_each) found = lane;
  }
  __syncthreads();
  const int b = __builtin_amdgcn_readfirstlane(found), rest = at % of_each;
  return {b, rest % hkv, rest / hkv, __builtin_amdgcn_readlane(len, b),
          __builtin_amdgcn_readlane(start, b)};
}

// Blocks of sequence b, from the first one of its part on, that another sequence of the
// batch reads too (a prefix that their requests share): those stay in L2 for the
// others, while what one sequence reads goes past L2's older lines.
//
// For a workgroup that has own[i] = block lo + i of its part's `n` blocks on their way
// to LDS. A wave asks for the other sequences' block lo ahead of these (Ask), and looks
// at them behind these and ahead of the barrier that these need anyway (before). Only
// where there is another one are the two rows compared (after).
//
// us of 32 sequences, 512 shared tokens and 100 of their own, all read past L2, none, and
// so; 3600 and 100: 32 heads of 128 44.2, 31.4 and 28.6; 257, 142 and 120; in e4m3 27.5,
// 23.9 and 20.2; 137, 105 and 78; 8 kv heads of 128 with four queries each 18.9, 15.4 and
// 14.8; 74.6, 43.7 and 43.4; 16 heads of 256 42.0, 29.6 and 27.9; 238, 115 and 112. Where
// nothing is shared it takes up to 0.5 us (32 of 100 tokens 13.4 and 13.9), so parts of
// up to four blocks, whose loads are little, are not looked at.
struct Shared {
  int other, same;
  RB_DEV static bool asked(int n) { return n > 4 && gridDim.x > 1; }
  RB_DEV static bool first_wave() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x) < 64;
  }
  // of one wave: what it compares, asked for ahead of `own`
  struct Ask {
    int mine = 0, len = 0, block = 0;
    RB_DEV Ask(const int32_t *tables, const int32_t *lens, int max_blocks, int b,
               int lo, int n) {
      if (!asked(n) || !first_wave()) return;
      const int i = min((int)threadIdx.x & 63, (int)gridDim.x - 1);
      mine = tables[(int64_t)b * max_blocks + lo];
      len = lens[i];
      block = tables[(int64_t)i * max_blocks + lo];
    }
  };
  RB_DEV void before(const Ask &ask, const int32_t *tables, const int32_t *lens,
                     int max_blocks, int bs, int b, int lo, int n) {
    const int B = gridDim.x, lane = threadIdx.x & 63;
    if (!asked(n) || !first_wave()) return;
    int found = -1, len = ask.len, block = ask.block;
    for (int i0 = 0;;) {
      const unsigned long long those =
          __ballot(i0 + lane < B && i0 + lane != b && len > lo * bs &&
                   block == ask.mine);
      if (those != 0) found = i0 + __builtin_ctzll(those);
      i0 += 64;
      if (found >= 0 || i0 >= B) break;
      const int i = min(i0 + lane, B - 1);
      len = lens[i];
      block = tables[(int64_t)i * max_blocks + lo];
    }
    if (lane == 0) {
      other = found;
      same = n;
    }
  }
  template <int THREADS>
  RB_DEV int after(const int32_t *tables, const int32_t *lens, int max_blocks,
                   int bs, int lo, int n, const int32_t *own) {
    if (!asked(n)) return 0;
    const int who = __builtin_amdgcn_readfirstlane(other);
    if (who < 0) return 0;
    const int32_t *at = tables + (int64_t)who * max_blocks + lo;
    const int theirs = (lens[who] + bs - 1) / bs - lo;
    for (int i = threadIdx.x; i < n; i += THREADS)
      if (i >= theirs || at[i] != own[i]) {
        atomicMin(&same, i);
        break;
      }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(same);
  }
};

// load(true) or load(false), whose instructions differ in what they say to L2 alone:
// taken for the same ones, they would become one that says nothing.
template <typename Load> RB_DEV void by_policy(bool past, Load load) {
  if (past) {
    asm volatile("; past L2" ::: "memory");
    load(std::true_type{});
    asm volatile("; past L2" ::: "memory");
  } else {
    load(std::false_type{});
  }
}

// FP8: caches are e4m3 rows of fp8_row_bytes(DH) = DH bytes + f32
// scale (+pad): decode attention is KV-bandwidth bound at long context,
// so halving cache bytes halves the dominant stream AND doubles KV
// capacity within 288 GB. Dequant rides
// v_cvt_pk_f32_fp8 in the inner loop.
//
// BS: tokens of a block, where that is known (0: any number). With it the first form's
// two kinds of loads fit the 64 registers of eight waves a SIMD.
template <int DH, int G, bool SPLIT, bool FP8 = false, int WAVES = NW,
          int PER_SIMD = 1, bool ONCE = false, int BS = 0>
__global__ __launch_bounds__(WAVES * 64, PER_SIMD) void paged_decode_kernel(
    const uint16_t *__restrict__ q, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache, const int32_t *__restrict__ block_tables,
    const int32_t *__restrict__ seq_lens,
    const int32_t *__restrict__ seq_starts, uint16_t *__restrict__ out,
    uint16_t *__restrict__ out_swz,
    float *__restrict__ partial, int hkv, int block_size, int max_blocks,
    int nsplit, float scale, bool sorted) {
  const int bs = BS != 0 ? BS : block_size;
  // Lane-group geometry: GL lanes cover one token's Dh, with 16 B a lane and
  // load (8 B accesses run 0.54-0.70x on gfx950 — the first fp8 cut used
  // 16-lane groups and showed ZERO long-context win): 16 lanes for bf16 rows of
  // heads of 128 and, by two loads, 256; 8 lanes for e4m3 rows, of 1 B an
  // element, and for bf16 rows of heads of 64, of 128 B.
  // (More query heads keep 16-lane groups, G > 4 for fp8 and G >= NW for heads
  // of 64: qreg[G][VE]+acc[G][VE] of twice the VE would spill past 256 VGPRs)
  constexpr int GL = (FP8 && G <= 4) || (DH == 64 && G < NW) ? 8 : 16;
  constexpr int VE = DH / GL;              // elems per lane
  constexpr int TPW = 64 / GL;             // tokens per wave pass
  // Head-split mode (G >= NW): each wave owns GW = G/NW query heads
  // over ALL tokens — the waves re-read the same K/V rows (L1/L2-
  // served; HBM bytes unchanged) — instead of all G heads over a
  // quarter of the tokens. Cuts per-wave state (qreg+acc = 2*G*VE
  // floats) by NW, unlocking occupancy 2 -> 4-5 on the GQA/MQA
  // kernels, shortens the serial dot->reduce->exp chain per
  // iteration, and removes the cross-wave LDS merge entirely.
  constexpr bool HS = (G >= NW);
  constexpr int GW = HS ? G / NW : G;
  const Place place =
      sorted ? sorted_place(seq_lens, seq_starts)
             : shifted_place(seq_lens, seq_starts);
  const int b = place.b, h_kv = place.h, split = place.split;
  const int hq0 = h_kv * G;
  const int Hq = hkv * G;

  const int seq_len = place.len;
  // Strict sliding windows: seq_starts[b] (0 when null) is the first
  // VIRTUAL position this query attends to — mistral attends to exactly
  // W trailing tokens, not the engine's retained block-aligned W..W+15.
  // Index math pre-validated on CPU: tests/test_decode_sim_cpu.py
  // (simulate_decode seq_starts).
  const int start = place.start;
  int t_begin = start, t_end = seq_len;
  if (SPLIT) {
    const int len = seq_len - start;
    const int chunk = (len + nsplit - 1) / nsplit;
    t_begin = start + split * chunk;
    t_end = min(seq_len, t_begin + chunk);
  }

  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int grp = lane / GL;               // lane group: token sub-index
  const int gl = lane % GL;                // lane within group
  // This lane's columns: pieces of 16 bytes, those of a group side by side, so
  // that a load takes whole lines of memory (16 heads of 256, whose rows are two
  // pieces a lane, us with a lane's pieces side by side and so: 32 sequences of 100
  // to 2000 tokens 100 and 91, 7 of 90 to 1801 29.5 and 27.3).
  constexpr int CH = VE < (FP8 ? 16 : 8) ? VE : (FP8 ? 16 : 8);
  const int d0 = gl * CH;
  auto column = [&](int e) { return d0 + e / CH * (GL * CH) + e % CH; };

  // Q for this wave's GW heads. bf16 caches keep Q as PACKED bf16 pairs: the
  // K dot then runs on v_dot2_f32_bf16 straight from the raw K words — no
  // per-element convert+FMA chain — and is scaled in fp32.
  const int hq_base = hq0 + (HS ? wid * GW : 0);
  float qreg[GW][VE];
  unsigned qpk[GW][VE / 2];
#pragma unroll
  for (int g = 0; g < GW; ++g) {
    const uint16_t *qp = q + ((int64_t)b * Hq + hq_base + g) * DH;
#pragma unroll
    for (int e = 0; e < VE; ++e) qreg[g][e] = 0.f;
    {
      float tmp[VE];
#pragma unroll
      for (int e8 = 0; e8 < VE; e8 += 8) {
        if (VE - e8 >= 8) rb::VIO<uint16_t>::load(qp + column(e8), tmp + e8);
        else {
#pragma unroll
          for (int e = 0; e < VE % 8; ++e)
            tmp[e8 + e] = rb::bf16_to_f32(qp[column(e8 + e)]);
        }
      }
      if (FP8) {
#pragma unroll
        for (int e = 0; e < VE; ++e) qreg[g][e] = tmp[e] * scale;
      } else {
#pragma unroll
        for (int e2 = 0; e2 < VE / 2; ++e2)
          qpk[g][e2] = rb_pack_bf16(tmp[2 * e2], tmp[2 * e2 + 1]);
      }
    }
  }

  float m[GW], l[GW], acc[GW][VE];
#pragma unroll
  for (int g = 0; g < GW; ++g) {
    m[g] = -INFINITY; l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < VE; ++e) acc[g][e] = 0.f;
  }

  const int32_t *bt = block_tables + (int64_t)b * max_blocks;

  // Stage this WG's slice of the block table through LDS: all four
  // waves walk the same row, and a per-iteration global bt[] read
  // sits on the K/V address chain (its vmcnt gates the row loads).
  // 512 entries cover 8K tokens at bs=16; longer ranges fall back to
  // global reads past the staged prefix.
  constexpr int BT_LDS = 512;
  __shared__ int32_t bt_lds[BT_LDS];
  const int blk0 = t_begin / bs;
  const int nbt =
      t_begin < t_end ? min((t_end - 1) / bs - blk0 + 1, BT_LDS) : 0;
  __shared__ Shared shared;
  auto numbers = [&] {
    for (int i = (int)threadIdx.x; i < nbt; i += WAVES * 64)
      bt_lds[i] = bt[blk0 + i];
  };
  if constexpr (ONCE) {
    const Shared::Ask ask(block_tables, seq_lens, max_blocks, b, blk0,
                          nbt);
    numbers();
    shared.before(ask, block_tables, seq_lens, max_blocks, bs, b, blk0, nbt);
  } else {
    numbers();
  }
  __syncthreads();
  int alone = 0;                           // from this token on
  if constexpr (ONCE)
    alone = (blk0 + shared.after<WAVES * 64>(block_tables, seq_lens, max_blocks,
                                             bs, blk0, nbt, bt_lds)) * bs;

  // Software-pipelined KV stream: the K/V rows of later steps are issued as
  // RAW bytes while one is computed. (Converting at load time puts an
  // s_waitcnt vmcnt(0) between every row and its dot product.) Tail steps clamp
  // to the last row; the duplicate rows are masked out of the softmax with
  // s = -inf, so the trip count is wave-uniform and the prefetch is
  // branch-free inside.
  //
  // A step is TPS tokens of every lane group, TPS * TPW consecutive ones of a
  // wave. With few query heads the chain dot -> reduce -> exp -> accumulate is
  // what a step takes, and two tokens share it; the longest sequence of a batch
  // is one workgroup's chain.
  // us, 32 heads of 128, before (plain order of the sequences, one token a
  // step) and now: 32 sequences of 129 to 2015 tokens 141 -> 119 (4.7 TB/s),
  // of 1072 each 102 -> 106 (5.3); one of 701 in one split 35 -> 23, with 16
  // splits and their merge 13.2 -> 11.2; 16 of 800 to 3900 from an e4m3 cache
  // 93 -> 79.
  constexpr int KBPL = FP8 ? VE : VE * 2;  // K/V bytes per lane
  constexpr int RW = KBPL / 4;             // u32 words of that
  constexpr int TPS = GW == 1 || (GW == 2 && !FP8) ? 2 : 1;
  constexpr int DEPTH = (G >= 4) ? 4 : 2;
  const int stride = (HS ? 1 : WAVES) * TPW * TPS;    // tokens of a step
  const int tw0 = t_begin + (HS ? 0 : wid * TPW * TPS);  // wave's first token
  const int t_base = tw0 + grp;            // this lane group's first
  const int niter = (t_end > tw0) ? (t_end - tw0 + stride - 1) / stride : 0;

  uint32_t kraw[DEPTH][TPS][RW], vraw[DEPTH][TPS][RW];
  float kscale[DEPTH][TPS], vscale[DEPTH][TPS];

  const int uw = __builtin_amdgcn_readfirstlane(wid);
  auto fetch = [&](int i, int slot) {
    auto load = [&](auto past) {
      constexpr bool PAST = decltype(past)::value;
#pragma unroll
      for (int u = 0; u < TPS; ++u) {
        const int tt = min(t_base + i * stride + u * TPW, t_end - 1);
        const int bi = (unsigned)tt / (unsigned)bs - blk0;
        int blk = bt_lds[min(bi, BT_LDS - 1)];
        if (bi >= BT_LDS) {
          blk = bt[blk0 + bi];
          asm volatile("" : "+v"(blk));
        }
        const unsigned head = (unsigned)blk * (unsigned)hkv + h_kv;
        const int64_t row = (int64_t)head * bs + (unsigned)tt % (unsigned)bs;
        const uint8_t *k = reinterpret_cast<const uint8_t *>(k_cache);
        const uint8_t *v = reinterpret_cast<const uint8_t *>(v_cache);
        if constexpr (FP8) {
          const int64_t at = row * (DH + 16);
#pragma unroll
          for (int c = 0; c < VE; c += CH) {
            rb::ld_words<CH / 4>(kraw[slot][u] + c / 4, k + at + column(c));
            rb::ld_words<CH / 4>(vraw[slot][u] + c / 4, v + at + column(c));
          }
          kscale[slot][u] = *reinterpret_cast<const float *>(k + at + DH);
          vscale[slot][u] = *reinterpret_cast<const float *>(v + at + DH);
        } else {
          const int64_t at = (row * DH + d0) * 2;
#pragma unroll
          for (int c = 0; c < VE; c += CH)
            rb::ld_words<CH / 2, PAST>(kraw[slot][u] + c / 2,
                                       k + at + c * GL * 2);
#pragma unroll
          for (int c = 0; c < VE; c += CH)
            rb::ld_words<CH / 2, PAST>(vraw[slot][u] + c / 2,
                                       v + at + c * GL * 2);
        }
      }
    };
    const int first = t_begin + (HS ? 0 : uw * TPW * TPS) + i * stride;
    if constexpr (ONCE) by_policy(first >= alone, load);
    else load(std::false_type{});
  };

  // cur is a compile-time constant at every call site below, so the
  // ring buffer stays in registers (no dynamic indexing).
  auto step = [&](int i, int cur) {
    if (i + DEPTH - 1 < niter) fetch(i + DEPTH - 1, (cur + DEPTH - 1) % DEPTH);
#pragma unroll
    for (int g = 0; g < GW; ++g) {
      float sc[TPS], mn = m[g];
#pragma unroll
      for (int u = 0; u < TPS; ++u) {
        float x = 0.f;
        if (FP8) {
          float kf[VE];
#pragma unroll
          for (int w = 0; w < RW; ++w)
            rb::fp8w_to_f32(kraw[cur][u][w], kf + w * 4);
#pragma unroll
          for (int e = 0; e < VE; ++e) x += qreg[g][e] * kf[e];
          x *= kscale[cur][u];
        } else {
          // the K dot runs packed, straight from the raw words
#pragma unroll
          for (int e2 = 0; e2 < VE / 2; ++e2)
            x = rb_dot2(kraw[cur][u][e2], qpk[g][e2], x);
          x *= scale;
        }
        sc[u] = x;
      }
      // reduce across the lane group
      rb::lane_sums<GL>(sc);
#pragma unroll
      for (int u = 0; u < TPS; ++u) {
        if (t_base + i * stride + u * TPW >= t_end) sc[u] = -INFINITY;
        mn = fmaxf(mn, sc[u]);
      }
      if (mn != -INFINITY) {
        const float alpha = __expf(m[g] - mn);
        m[g] = mn;
        l[g] *= alpha;
#pragma unroll
        for (int e = 0; e < VE; ++e) acc[g][e] *= alpha;
#pragma unroll
        for (int u = 0; u < TPS; ++u) {
          float p = __expf(sc[u] - mn);
          l[g] += p;
          float vf[VE];
          if (FP8) {
#pragma unroll
            for (int w = 0; w < RW; ++w)
              rb::fp8w_to_f32(vraw[cur][u][w], vf + w * 4);
            p *= vscale[cur][u];
          } else {
            const uint16_t *vr =
                reinterpret_cast<const uint16_t *>(vraw[cur][u]);
#pragma unroll
            for (int e = 0; e < VE; ++e) vf[e] = rb::bf16_to_f32(vr[e]);
          }
#pragma unroll
          for (int e = 0; e < VE; ++e) acc[g][e] += p * vf[e];
        }
      }
    }
  };

#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (d < niter) fetch(d, d);
  for (int i = 0; i < niter; i += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (i + d < niter) step(i + d, d);
  }

  // Merge the TPW groups inside each wave: lanes l^GL ... l^32 hold the
  // same d0 slice, so lanes apart by a bit merge matching
  // elements.
  auto merge = [&](auto bit) {
    constexpr int OFF = decltype(bit)::value;
#pragma unroll
    for (int g = 0; g < GW; ++g) {
      const float mo = rb::lane_xor<OFF>(m[g]);
      const float lo = rb::lane_xor<OFF>(l[g]);
      const float mn = fmaxf(m[g], mo);
      // lanes without a key yet keep their zeros
      const float a1 = mn == -INFINITY ? 1.0f : __expf(m[g] - mn);
      const float a2 = mn == -INFINITY ? 0.0f : __expf(mo - mn);
#pragma unroll
      for (int e = 0; e < VE; ++e)
        acc[g][e] = acc[g][e] * a1 + rb::lane_xor<OFF>(acc[g][e]) * a2;
      l[g] = l[g] * a1 + lo * a2;
      m[g] = mn;
    }
  };
  if constexpr (GL == 8) merge(std::integral_constant<int, 8>{});
  merge(std::integral_constant<int, 16>{});
  merge(std::integral_constant<int, 32>{});

  if constexpr (HS) {
    // Head-split: each wave owns its GW heads outright — write out
    // (or the split partial) straight from registers, no LDS merge.
    if (grp == 0) {
#pragma unroll
      for (int g = 0; g < GW; ++g) {
        const int h = hq_base + g;
        if (SPLIT) {
          float *pp =
              partial + (((int64_t)b * Hq + h) * nsplit + split) * (DH + 2);
#pragma unroll
          for (int e = 0; e < VE; ++e) pp[column(e)] = acc[g][e];
          if (gl == 0) { pp[DH] = m[g]; pp[DH + 1] = l[g]; }
        } else {
          const float inv_l = (l[g] > 0.f) ? 1.0f / l[g] : 0.f;
          uint16_t *op = out + ((int64_t)b * Hq + h) * DH;
#pragma unroll
          for (int e = 0; e < VE; ++e)
            op[column(e)] = rb::f32_to_bf16(acc[g][e] * inv_l);
          if (out_swz != nullptr)
#pragma unroll
            for (int c = 0; c < VE; c += CH)
              store_operand<CH>(out_swz, h * DH + column(c), b, acc[g] + c,
                                inv_l);
        }
      }
    }
    return;
  }

  // Merge across the waves via LDS. Layout per (wave, head):
  // [DH acc][m][l] floats.
  __shared__ float lds[HS ? 1 : WAVES][HS ? 1 : G][DH + 2];
  if (grp == 0) {   // lanes 0..GL-1 of each wave hold the wave's merged state
#pragma unroll
    for (int g = 0; g < GW; ++g) {
#pragma unroll
      for (int e = 0; e < VE; ++e) lds[wid][g][column(e)] = acc[g][e];
      if (gl == 0) { lds[wid][g][DH] = m[g]; lds[wid][g][DH + 1] = l[g]; }
    }
  }
  __syncthreads();

  // Wave `wid` finalizes heads g = wid, wid+WAVES, ... (lanes 0..15 active).
  for (int g = wid; g < G; g += WAVES) {
    if (grp != 0) continue;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, lds[w][g][DH]);
    float ll = 0.f, av[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) av[e] = 0.f;
    if (mm != -INFINITY) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const float a = __expf(lds[w][g][DH] - mm);
        ll += lds[w][g][DH + 1] * a;
#pragma unroll
        for (int e = 0; e < VE; ++e) av[e] += lds[w][g][column(e)] * a;
      }
    }
    if (SPLIT) {
      float *pp = partial + (((int64_t)b * Hq + hq0 + g) * nsplit + split) * (DH + 2);
#pragma unroll
      for (int e = 0; e < VE; ++e) pp[column(e)] = av[e];
      if (gl == 0) { pp[DH] = mm; pp[DH + 1] = ll; }
    } else {
      const float inv_l = (ll > 0.f) ? 1.0f / ll : 0.f;
      uint16_t *op = out + ((int64_t)b * Hq + hq0 + g) * DH;
#pragma unroll
      for (int e = 0; e < VE; ++e)
        op[column(e)] = rb::f32_to_bf16(av[e] * inv_l);
      if (out_swz != nullptr)
#pragma unroll
        for (int c = 0; c < VE; c += CH)
          store_operand<CH>(out_swz, (hq0 + g) * DH + column(c), b, av + c,
                            inv_l);
    }
  }
}

// e4m3 caches of blocks of 16, up to two query heads a kv head: whole blocks of a head,
// which are contiguous, go to LDS past the registers, and their rows of DH + 16 bytes
// (values, scale) are read there. Loaded by rows, which begin and end within lines of
// memory, scales apart, a line was asked for up to three times and could not pass L2.
// A wave has a ring of its own and waits for no other, nor for more of its blocks than
// the one it reads; a lane group of eight takes a row, 16 tokens a step. Keys are
// multiplied as bf16 pairs, which they are exactly.
//
// Bound by memory. us by rows and so, whole sequences, 32 heads of 128: 16 of 800 to
// 3900 tokens 68.9 and 59.5 (5.8 TB/s), 32 of 1000 59.1 and 51.8, 64 of 1000 111 and
// 96, 32 of 50 to 1000 34.0 and 30.3, of 100 11.7 and 10.3, of 20 6.9 and 6.9, one of 50
// 4.8 and 4.3; where few CUs have anything to do, 4000 and 15 of 100 39.5 and 30.6, 4000
// and 31 of 100 58.0 and 40.9 (40.1 and 69.7 where a step waited for every block that was
// on its way). Two queries each: 32 of 50 to 1000 51 and 34. 12 heads of 64: 64 of 500
// 17.5 and 15.6. Four workgroups of four waves fill a CU, as two of eight do; the longer
// ring that two of four have room for is slower.
template <int DH, int WAVES> struct Blocks8 {
  static constexpr int PART = (DH + 16) * 16, STAGE = 2 * PART;   // K, then V
  static constexpr int FULL = PART / 1024, LOADS = 2 * FULL + 1;
  static constexpr int PER_CU = WAVES == 8 || DH == 256 ? 2 : 4;
  static constexpr int AHEAD = (160 / PER_CU - 3) * 1024 / STAGE / WAVES;
  static constexpr int LDS = WAVES * AHEAD * STAGE;
  static_assert(PART % 1024 == 256 && AHEAD >= 2, "pieces, ring");
};

template <int DH, int G, bool SPLIT, int WAVES, bool ONCE>
__global__ __launch_bounds__(WAVES * 64, DH == 256 ? 2 : 4) void paged_decode8_kernel(
    const uint16_t *__restrict__ q, const uint8_t *__restrict__ k_cache,
    const uint8_t *__restrict__ v_cache,
    const int32_t *__restrict__ block_tables,
    const int32_t *__restrict__ seq_lens,
    const int32_t *__restrict__ seq_starts, uint16_t *__restrict__ out,
    uint16_t *__restrict__ out_swz, float *__restrict__ partial, int hkv,
    int max_blocks, int nsplit, float scale, bool sorted) {
  using R = Blocks8<DH, WAVES>;
  constexpr int BS = 16, GL = 8, VE = DH / GL, TPW = 64 / GL, U = BS / TPW;
  constexpr int CH = VE < 16 ? VE : 16, RW = VE / 4;
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr float RISE = 8.0f;          // of a maximum before it is moved
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const Place place =
      sorted ? sorted_place(seq_lens, seq_starts)
             : shifted_place(seq_lens, seq_starts);
  const int b = place.b, h_kv = place.h, split = place.split;
  const int hq0 = h_kv * G, Hq = hkv * G;
  int t_begin = place.start, t_end = place.len;
  if (SPLIT) {
    const int chunk = (place.len - place.start + nsplit - 1) / nsplit;
    t_begin = place.start + split * chunk;
    t_end = min(place.len, t_begin + chunk);
  }
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = lane / GL, gl = lane % GL;
  // this lane's columns, as in paged_decode_kernel
  auto column = [&](int e) { return e / CH * (GL * CH) + gl * CH + e % CH; };

  const int32_t *bt = block_tables + (int64_t)b * max_blocks;
  constexpr int BT_LDS = 512;
  __shared__ int32_t bt_lds[BT_LDS];
  const int lo = t_begin / BS, hi = t_end > t_begin ? (t_end - 1) / BS : lo - 1;
  const int staged = min(hi - lo + 1, BT_LDS);
  __shared__ Shared shared;
  auto numbers = [&] {
    for (int i = (int)threadIdx.x; i < staged; i += WAVES * 64)
      bt_lds[i] = bt[lo + i];
  };
  if constexpr (ONCE) {
    const Shared::Ask ask(block_tables, seq_lens, max_blocks, b, lo,
                          staged);
    numbers();
    shared.before(ask, block_tables, seq_lens, max_blocks, BS, b, lo, staged);
  } else {
    numbers();
  }

  unsigned qpk[G][VE / 2];              // the rows' own bits; scaled in fp32
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int c = 0; c < VE; c += CH)
#pragma unroll
      for (int e = 0; e < CH; e += 8) {
        const uint4 w = *reinterpret_cast<const uint4 *>(
            q + ((int64_t)b * Hq + hq0 + g) * DH + column(c + e));
        qpk[g][(c + e) / 2] = w.x;
        qpk[g][(c + e) / 2 + 1] = w.y;
        qpk[g][(c + e) / 2 + 2] = w.z;
        qpk[g][(c + e) / 2 + 3] = w.w;
      }
  // where the compiler sees it: otherwise it waits for these in the loop, and with them
  // for the blocks that are on their way
  __builtin_amdgcn_s_waitcnt(0x0f70);             // vmcnt(0)
  __syncthreads();
  int alone = 0;                                  // from this block on
  if constexpr (ONCE)
    alone = lo + shared.after<WAVES * 64>(block_tables, seq_lens, max_blocks, BS,
                                          lo, staged, bt_lds);

  const unsigned mine = wid * (R::AHEAD * R::STAGE);
  const unsigned ring =
      mine + (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem;
  // a block's number, from LDS alone where it lies there: of a pointer to either place
  // the load would wait for all blocks that are on their way
  auto block_of = [&](int bi) {
    int blk = bt_lds[min(bi - lo, BT_LDS - 1)];
    if (bi - lo >= BT_LDS) {
      blk = bt[bi];
      asm volatile("" : "+v"(blk));
    }
    return __builtin_amdgcn_readfirstlane(blk);
  };
  auto send = [&](int bi, int stage, auto past) {
    constexpr bool PAST = decltype(past)::value;
    const int64_t at = ((int64_t)block_of(bi) * hkv + h_kv) * R::PART;
    const uint8_t *k = k_cache + at, *v = v_cache + at;
    const unsigned to =
        __builtin_amdgcn_readfirstlane(ring + stage * R::STAGE);
#pragma unroll
    for (int i = 0; i < R::FULL; ++i)
      rb::lds_load_from<PAST>(k + i * 1024 + lane * 16, to + i * 1024);
    // the last 16 pieces of K and the first of V
    if (lane < 32)
      rb::lds_load_from<PAST>(
          (lane < 16 ? k + R::FULL * 1024 : v - 256) + lane * 16,
          to + R::FULL * 1024);
#pragma unroll
    for (int i = 0; i < R::FULL; ++i)
      rb::lds_load_from<PAST>(v + 256 + i * 1024 + lane * 16,
                              to + R::PART + 256 + i * 1024);
  };
  auto fetch = [&](int bi, int stage) {
    if (ONCE && bi >= alone) send(bi, stage, std::true_type{});
    else send(bi, stage, std::false_type{});
  };

  float m[G], l[G], acc[G][VE];         // maxima in exponents of 2
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.0f;
#pragma unroll
    for (int e = 0; e < VE; ++e) acc[g][e] = 0.0f;
  }
  const float to2 = scale * LOG2E;
#pragma unroll
  for (int j = 0; j < R::AHEAD; ++j)
    if (lo + wid + j * WAVES <= hi) fetch(lo + wid + j * WAVES, j);
  int stage = 0;
  for (int bi = lo + wid; bi <= hi; bi += WAVES) {
    if (bi + (R::AHEAD - 1) * WAVES <= hi)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R::AHEAD - 1) * R::LOADS)
                   : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t kw[U][RW], vw[U][RW];
    float ks[U], vs[U];
    const char *at = smem + mine + stage * R::STAGE + grp * (DH + 16);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const char *k = at + u * TPW * (DH + 16), *v = k + R::PART;
#pragma unroll
      for (int c = 0; c < VE; c += CH) {
        rb::ld_words<CH / 4>(kw[u] + c / 4, (const uint8_t *)k + column(c));
        rb::ld_words<CH / 4>(vw[u] + c / 4, (const uint8_t *)v + column(c));
      }
      ks[u] = *reinterpret_cast<const float *>(k + DH);
      vs[u] = *reinterpret_cast<const float *>(v + DH);
    }
    // read before it is written again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (bi + R::AHEAD * WAVES <= hi) fetch(bi + R::AHEAD * WAVES, stage);
    stage = stage + 1 == R::AHEAD ? 0 : stage + 1;
    if (bi * BS < t_begin || (bi + 1) * BS > t_end) {
      // rows that are not the sequence's may hold anything
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = bi * BS + u * TPW + grp;
        const bool there = t >= t_begin && t < t_end;
        vs[u] = there ? vs[u] : 0.0f;
#pragma unroll
        for (int w = 0; w < RW; ++w) vw[u][w] = there ? vw[u][w] : 0;
      }
    }

    float x[G][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int g = 0; g < G; ++g) x[g][u] = 0.0f;
#pragma unroll
      for (int w = 0; w < RW; ++w) {
        const unsigned a = rb::fp8_pair_bf16<false>(kw[u][w]);
        const unsigned c = rb::fp8_pair_bf16<true>(kw[u][w]);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          x[g][u] = rb_dot2(a, qpk[g][2 * w], x[g][u]);
          x[g][u] = rb_dot2(c, qpk[g][2 * w + 1], x[g][u]);
        }
      }
    }
    float p[G][U];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      rb::lane_sums<GL>(x[g]);
      float mx = -INFINITY;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = bi * BS + u * TPW + grp;
        x[g][u] = t >= t_begin && t < t_end ? x[g][u] * (ks[u] * to2)
                                            : -INFINITY;
        mx = fmaxf(mx, x[g][u]);
      }
      if (__any(mx > m[g] + RISE)) {
        const float mn = fmaxf(m[g], mx);
        // groups that have seen no key keep a finite reference
        const float alpha =
            __builtin_amdgcn_exp2f(m[g] - (mn == -INFINITY ? 0.0f : mn));
        l[g] *= alpha;
#pragma unroll
        for (int e = 0; e < VE; ++e) acc[g][e] *= alpha;
        m[g] = mn;
      }
      const float ref = m[g] == -INFINITY ? 0.0f : m[g];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p[g][u] = __builtin_amdgcn_exp2f(x[g][u] - ref);
        l[g] += p[g][u];
        p[g][u] *= vs[u];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int w = 0; w < RW; ++w) {
        float f[4];
        rb::fp8w_to_f32(vw[u][w], f);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int g = 0; g < G; ++g) acc[g][w * 4 + e] += p[g][u] * f[e];
      }
  }

  // the lane groups of a wave, then the waves
  auto merge = [&](auto bit) {
    constexpr int OFF = decltype(bit)::value;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float mo = rb::lane_xor<OFF>(m[g]), lo = rb::lane_xor<OFF>(l[g]);
      const float mn = fmaxf(m[g], mo), ref = mn == -INFINITY ? 0.0f : mn;
      const float a1 = __builtin_amdgcn_exp2f(m[g] - ref);
      const float a2 = __builtin_amdgcn_exp2f(mo - ref);
#pragma unroll
      for (int e = 0; e < VE; ++e)
        acc[g][e] = acc[g][e] * a1 + rb::lane_xor<OFF>(acc[g][e]) * a2;
      l[g] = l[g] * a1 + lo * a2;
      m[g] = mn;
    }
  };
  merge(std::integral_constant<int, 8>{});
  merge(std::integral_constant<int, 16>{});
  merge(std::integral_constant<int, 32>{});
  static_assert(WAVES * G * (DH + 2) * 4 <= R::LDS, "merge buffer");
  float *ex = reinterpret_cast<float *>(smem);      // [wave][head][DH + 2]
  __syncthreads();                      // the last blocks have been read
  if (grp == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float *r = ex + (wid * G + g) * (DH + 2);
#pragma unroll
      for (int e = 0; e < VE; ++e) r[column(e)] = acc[g][e];
      if (gl == 0) {
        r[DH] = m[g];
        r[DH + 1] = l[g];
      }
    }
  }
  __syncthreads();
  // a wave a head, a lane DH / 64 columns
  constexpr int V = DH / 64;
  const int d0 = lane * V;
  for (int g = wid; g < G; g += WAVES) {
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
      mm = fmaxf(mm, ex[(w * G + g) * (DH + 2) + DH]);
    const float ref = mm == -INFINITY ? 0.0f : mm;
    float ll = 0.0f, o[V];
#pragma unroll
    for (int e = 0; e < V; ++e) o[e] = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float *r = ex + (w * G + g) * (DH + 2);
      const float a = __builtin_amdgcn_exp2f(r[DH] - ref);
      ll += r[DH + 1] * a;
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] += r[d0 + e] * a;
    }
    const int h = hq0 + g;
    if (SPLIT) {
      float *pp = partial +
                  (((int64_t)b * Hq + h) * nsplit + split) * (DH + 2);
#pragma unroll
      for (int e = 0; e < V; ++e) pp[d0 + e] = o[e];
      if (lane == 0) {
        pp[DH] = mm / LOG2E;
        pp[DH + 1] = ll;
      }
    } else {
      const float inv_l = ll > 0.0f ? 1.0f / ll : 0.0f;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const int kk = h * DH + d0 + e;
        const uint16_t y = rb::f32_to_bf16(o[e] * inv_l);
        out[(int64_t)b * Hq * DH + kk] = y;
        if (out_swz != nullptr)
          out_swz[(kk >> 4) * 512 + (kk >> 3 & 1) * 256 + b * 8 + (kk & 7)] = y;
      }
    }
  }
}

// Second pass for SPLIT mode: a workgroup of one wave merges the nsplit partials of one
// (b, hq) row. Maxima and sums are one load of the wave (a lane a partial), and the rows
// (VE = dh / 64 values a lane) are loaded 16 at a time beside it: one round trip to memory
// up to 16 splits. us of both kernels, one sequence of 701 tokens, 32 heads, 12 splits:
// 10.2 with rows loaded by eights behind their weights, 8.6 with rows beside them and
// four rows of the output a workgroup of four waves, 8.0 so.
template <int VE>
__global__ __launch_bounds__(64) void decode_combine_kernel(
    const float *__restrict__ partial, uint16_t *__restrict__ out,
    uint16_t *__restrict__ out_swz, int Hq, int nsplit) {
  constexpr int DH = VE * 64, CHUNK = 16;
  const int row = blockIdx.x;           // b * Hq + hq
  const int lane = threadIdx.x, d0 = lane * VE;
  const float *p = partial + (int64_t)row * nsplit * (DH + 2);
  float x[CHUNK][VE];
  auto load = [&](int s0) {             // past the end: the last one again
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
      const float *r = p + min(s0 + i, nsplit - 1) * (DH + 2) + d0;
#pragma unroll
      for (int e = 0; e < VE; ++e) x[i][e] = r[e];
    }
  };
  auto weights_of = [&](int s) {        // (m, l) of this lane's partial
    return *reinterpret_cast<const float2 *>(
        p + min(s + lane, nsplit - 1) * (DH + 2) + DH);
  };
  float2 ml = weights_of(0);
  load(0);
  float mm = lane < nsplit ? ml.x : -INFINITY;
  for (int s = 64; s < nsplit; s += 64)
    if (s + lane < nsplit) mm = fmaxf(mm, weights_of(s).x);
  mm = rb::wave_reduce_max(mm);
  float ll[1] = {0.f}, o[VE];
#pragma unroll
  for (int e = 0; e < VE; ++e) o[e] = 0.f;
  for (int s0 = 0; s0 < nsplit; s0 += CHUNK) {
    if (s0 % 64 == 0 && s0 > 0) ml = weights_of(s0);
    if (s0 > 0) load(s0);
    // partials of no keys have a maximum of minus infinity
    const int here = s0 / 64 * 64 + lane;
    const float w = here < nsplit && ml.x != -INFINITY ? __expf(ml.x - mm) : 0.f;
    if (s0 % 64 == 0) ll[0] += ml.y * w;
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
      const float by = __uint_as_float(__builtin_amdgcn_readlane(
          __float_as_uint(w), s0 % 64 + i));
#pragma unroll
      for (int e = 0; e < VE; ++e)
        if (by != 0.f) o[e] += x[i][e] * by;
    }
  }
  rb::lane_sums<64>(ll);
  const float inv_l = (ll[0] > 0.f) ? 1.0f / ll[0] : 0.f;
  auto put = [&](uint16_t *at) {
    if constexpr (VE == 1) *at = rb::f32_to_bf16(o[0] * inv_l);
#pragma unroll
    for (int e = 0; e + 1 < VE; e += 2)
      *reinterpret_cast<uint32_t *>(at + e) =
          rb::pack_bf16x2(o[e] * inv_l, o[e + 1] * inv_l);
  };
  put(out + (int64_t)row * DH + d0);
  if (out_swz != nullptr) {
    const int b = row / Hq, kk = row % Hq * DH + d0;
    put(out_swz + (kk >> 4) * 512 + ((kk >> 3) & 1) * 256 + b * 8 + (kk & 7));
  }
}

// ---------------------------------------------------------------------------
// MFMA decode for GQA/MQA (G >= 4), bf16 cache, DH in {64, 128}, bs == 16.
//
// The scalar formulation above spends ~30 VALU ops per (token, head) on
// dot -> shfl-reduce -> exp -> acc; at G >= 4 that serial chain is the
// bind (PMC: 57% WAIT_ANY / 28% VALU at 2 waves/SIMD pre-head-split,
// and the head-split variant re-reads K/V NW times through L2). Here
// scores and O^T are mfma_f32_16x16x32_bf16 chains — each K/V row is
// read once, and per-block VALU drops ~60x.
//
//  * a wave takes pairs of 16-token cache blocks, a step each: the chain scores
//    -> maximum -> exp -> product, which is what a step takes, is shared by 32
//    tokens. us, 32 query and 8 kv heads of 128, before (a block a step, P
//    through shuffles, 32-column products of G columns) and now: 64 sequences
//    of 1000 to 4003 tokens 139 -> 126 (5.2 TB/s), of 2500 each 122 -> 121;
//    8 of them with 8 splits 29 -> 23, one of 4000 with 16 splits 23 -> 12.
//    Two waves per SIMD: with one (280 registers) the first takes 137.
//  * two score tiles S[16][G], whose rows are tokens in an order of our own
//    choice: tile T's row 4 h + r is token 8 (h % 2) + 4 T + r of block h / 2.
//    A lane's scores of both tiles are then 8 consecutive tokens of one block,
//    and, rounded, the operand P[32 tok][G] as they are.
//  * K is read DIRECTLY in A-fragment order from the [BS, Dh] block
//    layout: 16 B per lane, 64 B segments, no staging.
//  * V comes from the TRANSPOSED cache layout ([Dh, BS] per block,
//    alloc_kv_cache v_transposed — the framework owns the layout, so
//    the PV A-fragment is a direct 16 B/lane read too. The first cut
//    staged the transpose through per-wave LDS; PMC showed 26-43% of
//    wave cycles burned in LDS bank conflicts (the b16 scatter's 8-row
//    lane stride lands on 2 of 64 banks at any 16-aligned row pitch).
//  * fragment maps (guide + mfma_probe_16x16x32 GPU test):
//      16x16x32: A[i=l&15][k=(l>>4)*8+e]; B[k][j=l&15]; C[j=l&15][i=(l>>4)*4+r]
// ---------------------------------------------------------------------------
// FP8 mode: K rows stay the scalar-path e4m3 layout ([BS][DH bytes +
// f32 scale + pad], fp8_row_bytes); V blocks are TRANSPOSED e4m3
// ([DH+4][BS] bytes — the 4 tail "rows" are 64 B = the 16 per-token
// f32 scales). Fragments are 8 B/lane raw loads dequanted at use; the
// per-token K scale folds into the S rows after the score MFMA and the
// V scale into P before the PV MFMA (softmax l/m stay on unscaled P).
template <int DH, int G, bool SPLIT, bool FP8 = false>
__global__ __launch_bounds__(BLOCK, 2) void paged_decode_mfma_kernel(
    const uint16_t *__restrict__ q, const uint16_t *__restrict__ k_cache,
    const uint16_t *__restrict__ v_cache,
    const int32_t *__restrict__ block_tables,
    const int32_t *__restrict__ seq_lens,
    const int32_t *__restrict__ seq_starts, uint16_t *__restrict__ out,
    uint16_t *__restrict__ out_swz, float *__restrict__ partial, int hkv,
    int max_blocks, int nsplit, float scale, bool sorted) {
  constexpr int BS = 16;                  // cache block = one S tile
  constexpr int KS32 = DH / 32;           // QK^T contraction steps
  constexpr int DT = DH / 16;             // O^T 16-row d-tiles
  constexpr int FRW = FP8 ? 2 : 4;        // u32 words per raw fragment

  const Place place =
      sorted ? sorted_place(seq_lens, seq_starts)
             : shifted_place(seq_lens, seq_starts);
  const int b = place.b, h_kv = place.h, split = place.split;
  const int hq0 = h_kv * G;
  const int Hq = hkv * G;

  const int seq_len = place.len;
  const int start = place.start;
  int t_begin = start, t_end = seq_len;
  if (SPLIT) {
    const int len = seq_len - start;
    const int chunk = (len + nsplit - 1) / nsplit;
    t_begin = start + split * chunk;
    t_end = min(seq_len, t_begin + chunk);
  }

  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int i16 = lane & 15;
  const int h16 = lane >> 4;              // 0..3

  const int32_t *bt = block_tables + (int64_t)b * max_blocks;

  // block-table staging (shared by all waves; same scheme as scalar)
  constexpr int BT_LDS = 512;
  __shared__ int32_t bt_lds[BT_LDS];
  const int blk0 = t_begin / BS;
  const int nbt =
      t_begin < t_end ? min((t_end - 1) / BS - blk0 + 1, BT_LDS) : 0;
  __shared__ Shared shared;
  auto numbers = [&] {
    for (int i = tid; i < nbt; i += BLOCK) bt_lds[i] = bt[blk0 + i];
  };
  if constexpr (!FP8) {
    const Shared::Ask ask(block_tables, seq_lens, max_blocks, b, blk0,
                          nbt);
    numbers();
    shared.before(ask, block_tables, seq_lens, max_blocks, BS, b, blk0, nbt);
  } else {
    numbers();
  }
  // cross-wave merge region
  __shared__ float mlds[NW][G][DH + 2];
  __syncthreads();
  int alone = 0;                          // from this block on
  if constexpr (!FP8)
    alone = blk0 + shared.after<BLOCK>(block_tables, seq_lens, max_blocks, BS,
                                       blk0, nbt, bt_lds);

  // Q fragments (B of the swapped QK^T); head = i16.
  rb_bf16x8v qf[KS32];
  {
    const bool hv = i16 < G;
    const uint16_t *qp =
        q + ((int64_t)b * Hq + hq0 + (hv ? i16 : 0)) * DH + h16 * 8;
#pragma unroll
    for (int ks = 0; ks < KS32; ++ks)
      qf[ks] = hv ? *reinterpret_cast<const rb_bf16x8v *>(qp + ks * 32)
                  : (rb_bf16x8v)(__bf16)0.0f;
  }

  rb_f32x4v acc_o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc_o[dt] = (rb_f32x4v)(0.0f);
  float m_run = -INFINITY, l_run = 0.0f;  // l_run: of this lane's tokens

  const int blk_lo = t_begin / BS;
  const int blk_hi = (t_end > t_begin) ? (t_end - 1) / BS : blk_lo - 1;
  // this lane's tokens within a pair of blocks, as scores and as V columns
  const int half = h16 >> 1, tok0 = (h16 & 1) * 8;
  // the K row that this lane loads for tile 0 (tile 1: four rows on)
  const int khalf = i16 >> 3, krow = (i16 >> 2 & 1) * 8 + (i16 & 3);

  // two pairs' raw fragments: the next one's are issued while one is computed
  uint32_t kfr[2][2][KS32][FRW], vfr[2][DT][FRW];
  float ksc[2][8], vsc[2][8];            // fp8 per-token scales

  auto block_of = [&](int bi) {          // the last one again past the end
    bi = min(bi, blk_hi);
    const int bi_l = bi - blk0;
    return (bi_l < BT_LDS) ? bt_lds[bi_l] : bt[bi];
  };
  auto fetch = [&](int bi, int slot) {
    const int blk_a = block_of(bi), blk_b = block_of(bi + 1);
    const int64_t kblk = (int64_t)(khalf ? blk_b : blk_a) * hkv + h_kv;
    const int64_t vblk = (int64_t)(half ? blk_b : blk_a) * hkv + h_kv;
    if (FP8) {
      constexpr int RB8 = DH + 16;       // fp8 K row bytes
      const uint8_t *k8 = reinterpret_cast<const uint8_t *>(k_cache);
      const uint8_t *kb = k8 + kblk * BS * RB8;
      const uint8_t *vb =
          reinterpret_cast<const uint8_t *>(v_cache) + vblk * (DH + 4) * BS;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ks = 0; ks < KS32; ++ks)
          rb::ld_words<2>(kfr[slot][t][ks],
                          kb + (krow + 4 * t) * RB8 + ks * 32 + h16 * 8);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        rb::ld_words<2>(vfr[slot][dt], vb + (dt * 16 + i16) * BS + tok0);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        ksc[slot][e] = *reinterpret_cast<const float *>(
            k8 + (vblk * BS + tok0 + e) * RB8 + DH);
        vsc[slot][e] = *reinterpret_cast<const float *>(
            vb + DH * BS + (tok0 + e) * 4);
      }
    } else {
      const uint8_t *kb = reinterpret_cast<const uint8_t *>(
          k_cache + kblk * BS * DH);
      // v block is [DH][BS] (transposed layout)
      const uint8_t *vb = reinterpret_cast<const uint8_t *>(
          v_cache + vblk * DH * BS);
      auto load = [&](auto past) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int ks = 0; ks < KS32; ++ks)
            rb::ld_words<4, decltype(past)::value>(
                kfr[slot][t][ks],
                kb + ((krow + 4 * t) * DH + ks * 32 + h16 * 8) * 2);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          rb::ld_words<4, decltype(past)::value>(
              vfr[slot][dt], vb + ((dt * 16 + i16) * BS + tok0) * 2);
      };
      by_policy(bi >= alone, load);
    }
  };

  // raw fragment -> bf16 MFMA operand (fp8: dequant UNSCALED — scales
  // fold into S / P outside the MFMA)
  auto frag = [&](const uint32_t *raw) -> rb_bf16x8v {
    union { unsigned u[4]; rb_bf16x8v v; } c;
    if (FP8) {
      float f[8];
      rb::fp8w_to_f32(raw[0], f);
      rb::fp8w_to_f32(raw[1], f + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        c.u[e] = rb_pack_bf16(f[2 * e], f[2 * e + 1]);
    } else {
      c.u[0] = raw[0]; c.u[1] = raw[1]; c.u[2] = raw[2]; c.u[3] = raw[3];
    }
    return c.v;
  };

  constexpr int PAIR = 2 * NW;            // blocks of a step
  auto step = [&](int bi, int cur) {
    if (bi + PAIR <= blk_hi) fetch(bi + PAIR, cur ^ 1);

    // ---- scores of two tiles: element 4 T + r is token tok0 + 4 T + r ----
    float p[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      rb_f32x4v s4 = (rb_f32x4v)(0.0f);
#pragma unroll
      for (int ks = 0; ks < KS32; ++ks)
        s4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(kfr[cur][t][ks]),
                                                     qf[ks], s4, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) p[t * 4 + r] = s4[r] * scale;
    }
    if (FP8) {
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] *= ksc[cur][e];
    }

    // ---- mask + online softmax (state per head = per col = per lane) --
    const int t0 = (bi + half) * BS + tok0;
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (t0 + e < t_begin || t0 + e >= t_end) p[e] = -INFINITY;
      mx = fmaxf(mx, p[e]);
    }
    mx = fmaxf(mx, rb::lane_xor<16>(mx));
    mx = fmaxf(mx, rb::lane_xor<32>(mx));
    if (__any(mx > m_run)) {
      const float mn = fmaxf(m_run, mx);
      const float alpha = mn == -INFINITY ? 1.0f : __expf(m_run - mn);
      l_run *= alpha;
      m_run = mn;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc_o[dt][r] *= alpha;
    }
    // heads that have seen no finite score keep a finite reference
    const float ref = m_run == -INFINITY ? 0.0f : m_run;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = __expf(p[e] - ref);
      l_run += p[e];
      // fp8: the per-token V scale rides on P here (l stays on the unscaled
      // softmax numerators)
      if (FP8) p[e] *= vsc[cur][e];
    }
    union { unsigned u[4]; rb_bf16x8v v; } pf;
#pragma unroll
    for (int e = 0; e < 4; ++e) pf.u[e] = rb_pack_bf16(p[2 * e], p[2 * e + 1]);

    // ---- O^T[d][head] += V^T @ P ----------------------------------------
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      acc_o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          frag(vfr[cur][dt]), pf.v, acc_o[dt], 0, 0, 0);
  };

  const int bi0 = blk_lo + 2 * __builtin_amdgcn_readfirstlane(wid);
  if (bi0 <= blk_hi) fetch(bi0, 0);
  for (int bi = bi0; bi <= blk_hi; bi += 2 * PAIR) {
    step(bi, 0);
    if (bi + PAIR <= blk_hi) step(bi + PAIR, 1);
  }
  l_run += rb::lane_xor<16>(l_run);
  l_run += rb::lane_xor<32>(l_run);

  // ---- cross-wave merge via LDS (same scheme as the scalar kernel) ----
  // acc_o lane map: head = i16, d = dt*16 + 4*h16 + r.
  if (i16 < G) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        mlds[wid][i16][dt * 16 + 4 * h16 + r] = acc_o[dt][r];
  }
  if (lane < 16 && i16 < G) {
    mlds[wid][i16][DH] = m_run;
    mlds[wid][i16][DH + 1] = l_run;
  }
  __syncthreads();

  constexpr int VE = DH / 16;             // elems per merge lane
  const int gl = lane & 15;
  const int d0 = gl * VE;
  for (int g = wid; g < G; g += NW) {
    if (lane >= 16) continue;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) mm = fmaxf(mm, mlds[w][g][DH]);
    float ll = 0.f, av[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) av[e] = 0.f;
    if (mm != -INFINITY) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float a = __expf(mlds[w][g][DH] - mm);
        ll += mlds[w][g][DH + 1] * a;
#pragma unroll
        for (int e = 0; e < VE; ++e) av[e] += mlds[w][g][d0 + e] * a;
      }
    }
    if (SPLIT) {
      float *pp =
          partial + (((int64_t)b * Hq + hq0 + g) * nsplit + split) * (DH + 2);
#pragma unroll
      for (int e = 0; e < VE; ++e) pp[d0 + e] = av[e];
      if (gl == 0) { pp[DH] = mm; pp[DH + 1] = ll; }
    } else {
      const float inv_l = (ll > 0.f) ? 1.0f / ll : 0.f;
      uint16_t *op = out + ((int64_t)b * Hq + hq0 + g) * DH + d0;
#pragma unroll
      for (int e = 0; e < VE; ++e) op[e] = rb::f32_to_bf16(av[e] * inv_l);
      if (out_swz != nullptr)
        store_operand<VE>(out_swz, (hq0 + g) * DH + d0, b, av, inv_l);
    }
  }
}

template <int DH, int G, bool FP8>
void launch_decode(const at::Tensor &q, const at::Tensor &k_cache,
                   const at::Tensor &v_cache, const at::Tensor &block_tables,
                   const at::Tensor &seq_lens,
                   const c10::optional<at::Tensor> &seq_starts,
                   at::Tensor &out, const c10::optional<at::Tensor> &out_swz,
                   int nsplit,
                   float scale, hipStream_t stream) {
  const int32_t *starts = seq_starts.has_value()
      ? seq_starts->data_ptr<int32_t>() : nullptr;
  const int B = (int)q.size(0);
  const int hkv = (int)k_cache.size(1);
  const int bs = (int)k_cache.size(2);
  const int max_blocks = (int)block_tables.size(1);
  uint16_t *swz = out_swz.has_value() ? (uint16_t *)out_swz->data_ptr()
                                      : nullptr;
  const int64_t longest = (int64_t)max_blocks * bs;
  const bool sorted = B > 4 && B <= 64 && longest > 512;
  // MFMA route: keyed on the TRANSPOSED V layout (bf16 [Dh, BS] /
  // fp8 [Dh+4, BS] blocks) the allocator chooses for MFMA-eligible
  // models (G >= 4, DH <= 128, 16-token blocks — RB_DECODE_MFMA=0 at
  // alloc reverts). The layout is the single source of truth: a
  // transposed cache can only be read by the MFMA kernel and vice
  // versa.
  const bool vt = v_cache.size(3) == bs &&
      v_cache.size(2) == (int64_t)(FP8 ? DH + 4 : DH);
  nsplit = (int)paged_decode_parts(nsplit, longest, DH, G, vt);
  if constexpr (G >= 4 && DH <= 128) {
    if (vt && bs == 16) {
      if (nsplit <= 1) {
        hipLaunchKernelGGL((paged_decode_mfma_kernel<DH, G, false, FP8>),
                           dim3(B, hkv, 1), dim3(BLOCK), 0, stream,
                           (const uint16_t *)q.data_ptr(),
                           (const uint16_t *)k_cache.data_ptr(),
                           (const uint16_t *)v_cache.data_ptr(),
                           block_tables.data_ptr<int32_t>(),
                           seq_lens.data_ptr<int32_t>(), starts,
                           (uint16_t *)out.data_ptr(), swz, nullptr, hkv,
                           max_blocks, 1, scale, sorted);
      } else {
        const int Hq = hkv * G;
        auto partial = at::empty({B, Hq, nsplit, DH + 2},
                                 q.options().dtype(at::kFloat));
        hipLaunchKernelGGL((paged_decode_mfma_kernel<DH, G, true, FP8>),
                           dim3(B, hkv, nsplit), dim3(BLOCK), 0, stream,
                           (const uint16_t *)q.data_ptr(),
                           (const uint16_t *)k_cache.data_ptr(),
                           (const uint16_t *)v_cache.data_ptr(),
                           block_tables.data_ptr<int32_t>(),
                           seq_lens.data_ptr<int32_t>(), starts,
                           nullptr, nullptr, partial.data_ptr<float>(), hkv,
                           max_blocks, nsplit, scale, sorted);
        hipLaunchKernelGGL((decode_combine_kernel<DH / 64>),
                           dim3(B * Hq), dim3(64), 0, stream,
                           partial.data_ptr<float>(),
                           (uint16_t *)out.data_ptr(), swz, Hq,
                           nsplit);
      }
      return;
    }
  }
  TORCH_CHECK(!vt, "paged_decode: transposed V cache requires the MFMA "
              "path (bf16, G>=4, Dh<=128, bs==16); got G=", G, " Dh=", DH);
  const int Hq = hkv * G;
  auto go = [&](auto kernel, int waves, int splits, float *partial) {
    hipLaunchKernelGGL(kernel, dim3(B, hkv, splits), dim3(waves * 64), 0,
                       stream, (const uint16_t *)q.data_ptr(),
                       (const uint16_t *)k_cache.data_ptr(),
                       (const uint16_t *)v_cache.data_ptr(),
                       block_tables.data_ptr<int32_t>(),
                       seq_lens.data_ptr<int32_t>(), starts,
                       splits > 1 ? nullptr : (uint16_t *)out.data_ptr(),
                       splits > 1 ? nullptr : swz, partial, hkv, bs, max_blocks,
                       splits, scale, sorted);
  };
  // Keys and values go past L2's older lines, as in a step a sequence's are read once
  // (ONCE; us of caches that lie in memory, without and with it: 32 sequences of 129 to
  // 2015 tokens, 32 heads of 128 104 and 92, 4 of 4000 54 and 49, one of 701 10.9 and
  // 10.2, of 37 4.8 and 4.5; 64 of 37 to 1400, 12 heads of 64 30.9 and 28.0). What
  // sequences share does not (Shared). Heads of 64 are those of small models, whose
  // caches a few sequences leave in L2 from step to step: there not, as far as a
  // layer's table has room for no more than L2's 32 MB (one of 37 tokens, 12 heads 3.6
  // and 3.9).
  const bool once = DH != 64 || (int64_t)B * hkv * longest *
                                        (FP8 ? DH + 16 : DH * 2) * 2 >
                                    ((int64_t)32 << 20);
  if constexpr (FP8 && G < NW) {
    // (loads to LDS take addresses that are multiples of their 16 bytes; a cache that
    // begins anywhere, or has other blocks, is read through registers)
    const auto begin = reinterpret_cast<uintptr_t>(k_cache.data_ptr()) |
                       reinterpret_cast<uintptr_t>(v_cache.data_ptr());
    if (bs == 16 && begin % 16 == 0) {
      const int splits = std::max(nsplit, 1);
      at::Tensor partial;
      if (splits > 1)
        partial = at::empty({B, Hq, splits, DH + 2},
                            q.options().dtype(at::kFloat));
      auto go8 = [&](auto part, auto waves, auto past) {
        constexpr int WAVES = decltype(waves)::value;
        constexpr int lds = Blocks8<DH, WAVES>::LDS;
        auto kernel = paged_decode8_kernel<DH, G, decltype(part)::value, WAVES,
                                           decltype(past)::value>;
        static const bool ready =
            hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                lds) == hipSuccess;
        TORCH_CHECK(ready, "paged_decode: LDS size");
        hipLaunchKernelGGL(kernel, dim3(B, hkv, splits), dim3(WAVES * 64), lds,
                           stream, (const uint16_t *)q.data_ptr(),
                           (const uint8_t *)k_cache.data_ptr(),
                           (const uint8_t *)v_cache.data_ptr(),
                           block_tables.data_ptr<int32_t>(),
                           seq_lens.data_ptr<int32_t>(), starts,
                           splits > 1 ? nullptr : (uint16_t *)out.data_ptr(),
                           splits > 1 ? nullptr : swz,
                           splits > 1 ? partial.data_ptr<float>() : nullptr,
                           hkv, max_blocks, splits, scale, sorted);
      };
      auto by_cache = [&](auto part, auto waves) {
        if constexpr (DH == 64)
          if (!once) return go8(part, waves, std::false_type{});
        go8(part, waves, std::true_type{});
      };
      // By 8 waves where two workgroups a CU are all there are. With more the others
      // would be begun when these end, and four of 4 waves fit a CU (us by 4 and 8, 12
      // heads of 64: 64 sequences of 100 tokens 7.1 and 9.2, of 300 11.1 and 13.1, of 50 to
      // 1000 17.0 and 19.5, 2000 and 63 of 100 20.7 and 14.7; by rows 7.8, 11.7, 18.6, 19.2;
      // 43 sequences 6.6 8.6, 10.1 11.4, 13.9 14.2, 20.3 14.4 and 7.3, 10.4, 14.4, 17.6).
      using Four = std::integral_constant<int, 4>;
      using Most = std::integral_constant<int, DH == 256 ? 4 : 8>;
      if (splits > 1) by_cache(std::true_type{}, Four{});
      else if (longest > 64 && (int64_t)B * hkv <= 512)
        by_cache(std::false_type{}, Most{});
      else by_cache(std::false_type{}, Four{});
      if (splits > 1)
        hipLaunchKernelGGL((decode_combine_kernel<DH / 64>),
                           dim3(B * Hq), dim3(64), 0, stream,
                           partial.data_ptr<float>(),
                           (uint16_t *)out.data_ptr(), swz, Hq, splits);
      return;
    }
  }
  // blocks of 16 tokens, as caches have them, or any
  auto by_block = [&](auto launch) {
    using Any = std::integral_constant<int, 0>;
    using Sixteen = std::integral_constant<int, 16>;
    if constexpr (!FP8 && G < NW) {
      if (bs == 16 && once) return launch(std::true_type{}, Sixteen{});
      if constexpr (DH == 64)
        if (bs == 16) return launch(std::false_type{}, Sixteen{});
    }
    // (eight query heads read a block's number often: us with any number of tokens in a
    // block and with 16, 64 heads of 128, 64 sequences of 50 to 1000 tokens 77.7 and 62.5,
    // 32 of 2000 131 and 114; 32 heads of 64 30.4 and 28.9, 51.5 and 48.1)
    if constexpr (!FP8 && G == 8)
      if (bs == 16) return launch(std::false_type{}, Sixteen{});
    launch(std::false_type{}, Any{});
  };
  if constexpr (G < NW) {
    // Whole sequences by 8 waves: of a short one more have nothing to do, and a CU
    // has room for more workgroups (which is why one query head a kv head keeps
    // to 64 registers, of 68). By 16 where long tables and few workgroups leave
    // the longest sequences to the end; by 4 where there are workgroups enough and
    // 8 waves take too many registers (two query heads).
    // us by 4, 8 and 16 waves, caches out of L2, 32 heads of 128 in bf16: 32 sequences of
    // 100 tokens 13.9, 14.0 and 17.5, of 300 30.7, 30.6 and 33.1, of 129 to 2015 100, 94
    // and 97, 4000 and 31 of 100 112, 64 and 49; 16 of 100 9.2, 9.3 and 9.6, of 800 to
    // 3900 129, 103 and 102, 4000 and 15 of 100 109, 61 and 47; one of 100 6.1, 5.2 and
    // 5.9, of 512 16.2, 10.6 and 10.1. By 4 and 8 waves: 12 heads of 64, 64 of 37 to 1400
    // 32.0 and 28.5; 32 kv heads with two queries each, 64 of 100 25.3 and 31.5, of 50 to
    // 1000 93 and 99; 16 heads of 256, 40 of 100 16.2 and 18.6, of 50 to 1000 62.4 and
    // 59.3. e4m3 by whole blocks (above): 32 heads of 128, 32 of 100 10.7 and 14.4, of 50
    // to 1000 31.6 and 34.5, 64 of 300 33.8 and 39.6, of 1000 99.9 and 98.1, 16 of 1000
    // 29.3 and 28.9, 4000 and 15 of 100 41.1 and 30.3.
    constexpr int ROOM = !FP8 && G == 1 && DH <= 128 ? 8 : 1;
    const int64_t base = (int64_t)B * hkv;
    if constexpr (ROOM == 8 && DH == 128)
      if (nsplit <= 1 && longest > 512 && base <= 512)
        return by_block([&](auto past, auto block) {
          go(paged_decode_kernel<DH, G, false, FP8, 16, ROOM,
                                 decltype(past)::value, decltype(block)::value>,
             16, 1, nullptr);
        });
    const bool many = (FP8 || G > 1) && base > (DH == 64 ? 1023 : 512);
    if (nsplit <= 1 && longest > 64 && !many)
      return by_block([&](auto past, auto block) {
        go(paged_decode_kernel<DH, G, false, FP8, 8, ROOM, decltype(past)::value,
                               decltype(block)::value>,
           8, 1, nullptr);
      });
  }
  if (nsplit <= 1)
    return by_block([&](auto past, auto block) {
      go(paged_decode_kernel<DH, G, false, FP8, NW, 1, decltype(past)::value,
                             decltype(block)::value>,
         NW, 1, nullptr);
    });
  auto partial = at::empty({B, Hq, nsplit, DH + 2},
                           q.options().dtype(at::kFloat));
  by_block([&](auto past, auto block) {
    go(paged_decode_kernel<DH, G, true, FP8, NW, 1, decltype(past)::value,
                           decltype(block)::value>,
       NW, nsplit, partial.data_ptr<float>());
  });
  hipLaunchKernelGGL((decode_combine_kernel<DH / 64>),
                     dim3(B * Hq), dim3(64), 0, stream,
                     partial.data_ptr<float>(), (uint16_t *)out.data_ptr(), swz,
                     Hq, nsplit);
}

}  // namespace

// Parts that a sequence of a kv head is taken in, of the nsplit that there are
// workgroups of 4 waves for; `longest` is what a block table has room for, the only
// bound on the lengths that is known here.
//
// Parts of fewer than 64 tokens cost more than they save (one sequence of 37
// tokens, 32 heads of 128: 16 parts 8.2 us, one 4.1; matrix instructions take 32:
// 32 query heads, one of 500, 16 parts 7.5, 10 7.9). One workgroup of more waves
// takes all of a sequence in place of two parts, or where the table is short: then
// the launch that adds up the parts goes, and the longest sequence of an uneven
// batch takes about as long. In place of more parts it does not, and an engine's
// tables are wide whatever the lengths.
//
// us whole and in parts, caches out of L2, 32 heads of 128 in bf16, and in e4m3:
//   one (16 parts at most)  100 tokens  5.2  7.0   5.4  6.8   256   7.3  7.2   6.2  6.8
//                           384         9.0  7.4   7.1  7.1   512  10.6  7.6   7.8  7.2
//                           768        12.7  8.3   9.3  8.2  1024  15.0  8.6  10.8  8.2
//   two (16)                256         7.6  7.8   6.4  7.2   384   9.5  8.6   7.4  8.4
//                           512        11.2  9.1   8.1  8.5  1024  16.1 11.8  11.2 10.7
//   4 (8)                   256         8.1  9.2   6.9  8.6   512  12.1 11.8   8.6 10.6
//                          1024        18.8 18.2  12.2 13.4
//     1024 and 3 of 50                 15.6 11.0  11.1 10.6
//   8 (4)                   256        10.0 11.7   8.2 10.9   512  15.3 17.6  10.9 13.6
//                          1024        26.9 28.1  17.8 20.0
//     129 to 2015                      31.8 30.0  21.4 21.6
//     4000 and 7 of 100                45.5 35.6  29.5 17.6
//   16 (2)                  256        15.5 17.6  11.3 13.8   512  26.2 28.8  17.4 20.2
//     800 to 3900                       104  111  62.7 64.8
//     4000 and 15 of 100               47.1 61.7  30.5 26.9
// 16 heads of 256:
//   one (16)                256         9.8  8.2   8.3  8.4   384  11.9  8.5  10.0  8.5
//   8 (8)                   256        11.7 12.4   9.1 11.6   384  15.6 15.3  10.6 15.1
//     512 and 7 of 50                  14.9 10.2  12.2 15.1
//   16 (4)  4000 and 15 of 100         77.7 41.0  60.1 23.5
//   32 (2)  100 to 2000                93.1 94.7  54.6 60.6
//           4000 and 31 of 100         82.9 73.5  62.1 37.6
// The lines lie where even batches of four and more have them. One or two sequences in
// bf16 would gain 1 to 3 us in parts in tables of 384 to 512 tokens (256: 192 to 256).
int64_t paged_decode_parts(int64_t nsplit, int64_t longest, int64_t dh,
                           int64_t group, bool transposed) {
  const int64_t parts =
      std::min(nsplit, (longest + 63) / (transposed ? 32 : 64));
  const bool whole =
      group < NW && (parts <= 2 || longest <= (dh > 128 ? 256 : 512));
  return whole ? 1 : std::max<int64_t>(parts, 1);
}

std::vector<at::Tensor> paged_decode_swz(at::Tensor q, at::Tensor k_cache,
                                         at::Tensor v_cache,
                                         at::Tensor block_tables,
                                         at::Tensor seq_lens, int64_t nsplit,
                                         double scale,
                                         c10::optional<at::Tensor> seq_starts);

at::Tensor paged_decode(at::Tensor q, at::Tensor k_cache, at::Tensor v_cache,
                        at::Tensor block_tables, at::Tensor seq_lens,
                        int64_t nsplit, double scale,
                        c10::optional<at::Tensor> seq_starts) {
  return paged_decode_swz(q, k_cache, v_cache, block_tables, seq_lens,
                          nsplit, scale, seq_starts)[0];
}

// Variant also returning the decode-GEMM operand layout of the output
// (o_proj input swizzle fused into the attention epilogue).
std::vector<at::Tensor> paged_decode_swz(at::Tensor q, at::Tensor k_cache,
                                         at::Tensor v_cache,
                                         at::Tensor block_tables,
                                         at::Tensor seq_lens, int64_t nsplit,
                                         double scale,
                                         c10::optional<at::Tensor> seq_starts) {
  if (seq_starts.has_value()) {
    TORCH_CHECK(seq_starts->scalar_type() == at::kInt &&
                seq_starts->is_contiguous(), "paged_decode: seq_starts");
  }
  TORCH_CHECK(q.is_cuda() && q.is_contiguous(), "paged_decode: q");
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "paged_decode: bf16 only");
  TORCH_CHECK(block_tables.scalar_type() == at::kInt && seq_lens.scalar_type() == at::kInt,
              "paged_decode: int32 metadata");
  const int Hq = (int)q.size(1);
  const int dh = (int)q.size(2);
  const int hkv = (int)k_cache.size(1);
  TORCH_CHECK(Hq % hkv == 0, "paged_decode: Hq % Hkv");
  const int G = Hq / hkv;
  auto out = at::empty_like(q);
  // emit the o_proj operand layout only for decode-batch shapes
  c10::optional<at::Tensor> out_swz;
  const int B0 = (int)q.size(0);
  if (B0 <= 32 && (Hq * dh) % 16 == 0) {
    out_swz = at::empty({(int64_t)(Hq * dh / 16) * 512}, q.options());
  }
  auto stream = at::hip::getCurrentHIPStream();

  const bool fp8 = k_cache.scalar_type() == at::kByte;
  if (fp8) {
    TORCH_CHECK((int)k_cache.size(3) == dh + 16 &&
                v_cache.scalar_type() == at::kByte,
                "paged_decode: fp8 cache rows must be dh+16 bytes");
  }
#define RB_DEC(DHV, GV)                                                        \
  do {                                                                         \
    if (fp8)                                                                   \
      launch_decode<DHV, GV, true>(q, k_cache, v_cache, block_tables,         \
                                   seq_lens, seq_starts, out, out_swz,        \
                                   (int)nsplit, (float)scale, stream);        \
    else                                                                       \
      launch_decode<DHV, GV, false>(q, k_cache, v_cache, block_tables,        \
                                    seq_lens, seq_starts, out, out_swz,       \
                                    (int)nsplit, (float)scale, stream);       \
  } while (0)
  if (dh == 128) {
    switch (G) {
      case 1: RB_DEC(128, 1); break;
      case 2: RB_DEC(128, 2); break;
      case 4: RB_DEC(128, 4); break;
      case 8: RB_DEC(128, 8); break;
      default: TORCH_CHECK(false, "paged_decode: unsupported G=", G);
    }
  } else if (dh == 64) {
    switch (G) {
      case 1: RB_DEC(64, 1); break;
      case 2: RB_DEC(64, 2); break;
      case 4: RB_DEC(64, 4); break;
      case 8: RB_DEC(64, 8); break;
      case 16: RB_DEC(64, 16); break;
      default: TORCH_CHECK(false, "paged_decode: unsupported G=", G);
    }
  } else if (dh == 256) {
    // gemma-7b (wide heads, MHA). VE=16 -> ~70 VGPRs at G=1.
    switch (G) {
      case 1: RB_DEC(256, 1); break;
      case 2: RB_DEC(256, 2); break;
      default: TORCH_CHECK(false, "paged_decode: unsupported G=", G);
    }
  } else {
    TORCH_CHECK(false, "paged_decode: Dh must be 64/128/256, got ", dh);
  }
#undef RB_DEC
  if (out_swz.has_value()) return {out, *out_swz};
  return {out};
}
