// Flash-attention prefill (causal, GQA/MQA, bf16) for CDNA4 (gfx950).
//
// A workgroup is NW waves of 32 query rows each; tiles of 64 keys and values
// (flash_tile.h) stand in two LDS buffers, the next one on its way while one
// is worked on: one barrier per tile.
//
//  * S^T = K Q^T: a lane pair (l, l ^ 32) holds the scores of one query, so a
//    row's maximum is an in-lane reduction and one shuffle.
//  * Online softmax in base 2; the running maximum moves only when a row
//    exceeds it by a factor of 2^8, so the accumulators are rarely rescaled
//    (sums and result refer to the same maximum, whichever it is).
//  * O^T += V^T P^T: the transposed reads of V take the keys in the order of
//    the scores' registers, which are then the other operand as they are.
//
// What bounds it: the matrix cores and the softmax's vector instructions in
// turn (per 64 x 32 scores of 128 columns 32 MFMA of 32 cycles, and about as
// long in vector instructions); two waves per SIMD overlap them. Measured, one
// prompt, before (tiles staged through registers between two barriers) and now:
//   7931 tokens, 32 query and 8 kv heads of 128    1554 -> 484 us, 1065 TF/s
//   3001 tokens, the same                           331 ->  88 us,  842 TF/s
//   512 tokens, 32 heads of 128                      43 ->  13 us
//   1021 tokens, 16 heads of 256                    133 ->  36 us
//   4000 tokens, 32 heads of 64                     288 ->  89 us,  737 TF/s
// Since then, with loads to LDS that the compiler does not wait for, operands read
// ahead (flash_tile.h) and, of heads of 256, sums that stay in the matrix registers, on
// another card: 7931 tokens 510 -> 491, 2048 of 32 heads 54 -> 49, 1021 of 32 heads
// 22.7 -> 21.5; 16 heads of 256, 7931 713 -> 632, 1021 36 -> 33 (add_products). What is
// left: the two waves of a SIMD do the same at the same time, so that products and
// vector instructions take turns (48% of the time each). Two groups of waves a half-step
// apart, a barrier between half-steps, took as long: a half-step of products then waits
// for LDS (1860 clocks, 1024 of products).
//
// mfma_f32_32x32x16_bf16 layouts:
//   A[i][k]: i = lane&31, k = (lane>>5)*8 + e (e = 0..7)
//   C[i][j]: j = lane&31, i = (reg&3) + 8*(reg>>2) + 4*(lane>>5)
//
// q,k,v,out: [B, S, H, DH] bf16 token-major (tokens of q, and of k and v, at a
// stride of their own). DH in {64, 128, 256}.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>
#include <type_traits>

#include "flash_tile.h"

namespace {

using namespace flash;

constexpr float LOG2E = 1.4426950408889634f;
constexpr float RISE = 8.0f;           // of a maximum before it is moved

// c[i] += a[i] b, c in the matrix registers: as text, for with more sums than there are
// vector registers the compiler moves them back and forth in every step. It does not see
// these products, so what it would wait for ahead of one is in the text: a and b may
// have just been computed, moved or put together (up to 4 wait states; behind the first
// product nothing comes in between). Whoever else reads or writes c settles it first.
//
// Four at a time share the wait. us of 16 heads of 256 with products by themselves, a
// wait in each (of four and of two states) and so: 7931 tokens 731, 704 and 632, 1021
// 37.3, 35.7 and 33.3; and with a wait in the first of eight only, which what the
// compiler puts ahead of the others would have broken, 688 and 36.2.
constexpr int TEXT_PRODUCTS = 4;
RB_DEV void add_products(f32x16v *c, const bf16x8v *a, bf16x8v b) {
  asm volatile(
      "s_nop 3\n\t"
      "v_mfma_f32_32x32x16_bf16 %0, %4, %8, %0\n\t"
      "v_mfma_f32_32x32x16_bf16 %1, %5, %8, %1\n\t"
      "v_mfma_f32_32x32x16_bf16 %2, %6, %8, %2\n\t"
      "v_mfma_f32_32x32x16_bf16 %3, %7, %8, %3"
      : "+a"(c[0]), "+a"(c[1]), "+a"(c[2]), "+a"(c[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b));
}

RB_DEV void scale_sum(float &c, float by) {
  float t;
  asm volatile(
      "v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %2, %1\n\t"
      "v_accvgpr_write_b32 %0, %1" : "+a"(c), "=&v"(t) : "v"(by));
}

// SPLIT 2: two waves share 32 query rows, one takes the lower and one the upper
// 32 keys of every tile; their results meet in LDS at the end.
//
// ORDERED (SPLIT 1): 32 keys at a time in their own order, the maximum moved by
// every score above it, natural exponentials. The forward of training with
// ReLU keeps this one order of its roundings, for its gradient is not a
// continuous function of them: units that stand at zero pass all of a gradient
// or none, and of two orders, each 6% (2-norm) from the gradient of opt-125m in
// 64 bits, one is 4 to 6% from the other. Only heads of 64, whose factor of 1/8
// rounds nothing. us, 12 heads, 4 x 512 and 2047 tokens: 15 and 45, otherwise 10
// and 23.
template <int DH, int NW, int SPLIT, bool ORDERED = false>
__global__ __launch_bounds__(NW * 64, DH == 256 ? 1 : 2) void flash_prefill_kernel(
    const uint16_t *__restrict__ qp, const uint16_t *__restrict__ kp,
    const uint16_t *__restrict__ vp, uint16_t *__restrict__ op,
    float *__restrict__ lsep,  // [B, Hq, S] log-sum-exp for training bwd
    int B, int S, int Hq, int Hkv, int64_t q_stride, int64_t kv_stride,
    float scale) {
  constexpr int KSTEPS = DH / 16;       // QK^T contraction steps
  constexpr int DTILES = DH / 32;       // O column tiles
  constexpr int QT = NW / SPLIT * 32;
  constexpr int TILE = tile_bytes<DH>();

  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int hi = lane >> 5;
  const int col = lane & 31;                // qrow within the wave tile

  const Place at = place(blockIdx.x, (S + QT - 1) / QT, Hq, Hkv, B, true);
  const int q0 = at.tile * QT, h = at.head, b = at.batch;
  const int h_kv = h / (Hq / Hkv);
  const int group = wid / SPLIT, part = wid % SPLIT;
  const int wrow = q0 + group * 32;
  const int qrow = wrow + col;              // this lane's query row
  const bool q_valid = qrow < S;

  const uint16_t *kb = kp + (int64_t)b * S * kv_stride + h_kv * DH;
  const uint16_t *vb = vp + (int64_t)b * S * kv_stride + h_kv * DH;
  const TileLoad<DH, NW> load(wid, lane, kv_stride);
  const int kv_end = min(S, q0 + QT);       // causal upper bound for this WG
  const int n_tiles = (kv_end + ROWS - 1) / ROWS;
  load(kb, 0, S, smem, wid);
  load(vb, 0, S, smem + TILE, wid);

  // ---- Q fragments (B operand of K Q^T); a factor below zero goes into
  // their signs, so that scores and their maxima have one order, and a factor
  // of zero clears them, so that hidden scores stay at minus infinity --------
  bf16x8v qf[KSTEPS];
  {
    const uint16_t *src =
        qp + ((int64_t)b * S + (q_valid ? qrow : 0)) * q_stride + h * DH +
        hi * 8;
    const unsigned flip = scale < 0.0f ? 0x80008000u : 0u;
    const unsigned keep = scale == 0.0f ? 0u : ~0u;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      union { uint4 u; bf16x8v v; } c;
      c.u = *reinterpret_cast<const uint4 *>(src + ks * 16);
      c.u.x = (c.u.x ^ flip) & keep;
      c.u.y = (c.u.y ^ flip) & keep;
      c.u.z = (c.u.z ^ flip) & keep;
      c.u.w = (c.u.w ^ flip) & keep;
      qf[ks] = c.v;
    }
  }
  // scores -> exponents of 2
  const float to2 = scale == 0.0f ? 1.0f : fabsf(scale) * LOG2E;

  f32x16v acc_o[DTILES];
#pragma unroll
  for (int dt = 0; dt < DTILES; ++dt) acc_o[dt] = (f32x16v)(0.0f);
  float m_run = -INFINITY;                  // in exponents of 2 (ORDERED: of e)
  float l_run = 0.0f;

  // Wide heads have more sums than there is room for among the vector registers. Where
  // anything but a product reads or writes them, this is ahead of it and behind it, as
  // the compiler waits for neither (20 wait states at most).
  constexpr bool TEXT = DH == 256;
  auto settle = [&] {
    if constexpr (TEXT)
      asm volatile("s_nop 15\n\ts_nop 15"
                   : "+a"(acc_o[0]), "+a"(acc_o[1]), "+a"(acc_o[2]),
                     "+a"(acc_o[3]), "+a"(acc_o[4]), "+a"(acc_o[5]),
                     "+a"(acc_o[6]), "+a"(acc_o[7]));
  };
  settle();

  // Keys kbase .. kbase + 32 SUB - 1 of the tile, from row r0 on; `masked`:
  // some of them are hidden from some row
  constexpr int SUB = DH == 256 || SPLIT == 2 || ORDERED ? 1 : 2;
  constexpr int AT_ONCE = TEXT ? TEXT_PRODUCTS : 1;
  auto keys = [&](const char *kt, const char *vt, int kbase, int r0,
                  auto masked) {
    f32x16v s[SUB];
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
      s[u] = (f32x16v)(0.0f);
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
        s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            row_frag<DH>(kt, r0 + u * 32, ks, col, hi), qf[ks], s[u], 0, 0, 0);
    }
    // (of heads of 64 it changes nothing, of 256 it costs 4%)
    if constexpr (DH == 128) reads_ahead<SUB * KSTEPS, 8>();
    if constexpr (decltype(masked)::value) {
#pragma unroll
      for (int u = 0; u < SUB; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kbase + u * 32 + (r & 3) + 8 * (r >> 2) + 4 * hi;
          if (key > qrow) s[u][r] = -INFINITY;
        }
    }
    float mx = s[0][0];
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[u][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if constexpr (ORDERED) {
      const float by = scale == 0.0f ? 1.0f : fabsf(scale);
      const float mn = fmaxf(m_run, mx * by);
      if (mn == -INFINITY) return;
      const float alpha = m_run == -INFINITY ? 0.0f : __expf(m_run - mn);
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[0][r] = s[0][r] == -INFINITY ? 0.0f : __expf(s[0][r] * by - mn);
        sum += s[0][r];
      }
      l_run = l_run * alpha + sum;
      m_run = mn;
      if (alpha != 1.0f) {
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc_o[dt][r] *= alpha;
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8v pf = score_frag<true>(s[0], ks);
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt)
          acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              column_frag<DH, true>(vt, r0 + ks * 16, dt, lane), pf,
              acc_o[dt], 0, 0, 0);
      }
      return;
    }
    mx *= to2;
    if (__any(mx > m_run + RISE)) {
      const float mn = fmaxf(m_run, mx);
      // rows that have seen no finite score keep a finite reference
      const float alpha = __builtin_amdgcn_exp2f(
          m_run - (mn == -INFINITY ? 0.0f : mn));
      l_run *= alpha;
      // (TEXT: three instructions a sum, 0.9 us, where the others take one. The first
      // time there is nothing to scale; us of 16 heads of 256, 33 tokens 9.6 and 8.6,
      // 100 11.4 and 10.4, 250 15.3 and 14.1)
      if (!TEXT || __any(m_run != -INFINITY)) {
        settle();
#pragma unroll
        for (int dt = 0; dt < DTILES; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            if constexpr (TEXT) {
              float c = acc_o[dt][r];
              scale_sum(c, alpha);
              acc_o[dt][r] = c;
            } else {
              acc_o[dt][r] *= alpha;
            }
          }
        settle();
      }
      m_run = mn;
    }
    const float ref = m_run == -INFINITY ? 0.0f : m_run;
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[u][r] = __builtin_amdgcn_exp2f(fmaf(s[u][r], to2, -ref));
        l_run += s[u][r];
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8v pf = score_frag(s[u], ks);
#pragma unroll
        for (int dt = 0; dt < DTILES; dt += AT_ONCE) {
          bf16x8v vf[AT_ONCE];
#pragma unroll
          for (int j = 0; j < AT_ONCE; ++j)
            vf[j] = column_frag<DH>(vt, r0 + u * 32 + ks * 16, dt + j, lane);
          if constexpr (TEXT)
            add_products(&acc_o[dt], vf, pf);
          else
            acc_o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                vf[0], pf, acc_o[dt], 0, 0, 0);
        }
      }
    }
  };

  // waits for tile t and sends for the next one
  auto arrive = [&](int t) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                    // nobody reads the other buffer any more
    if (t + 1 < n_tiles) {
      char *next = smem + (~t & 1) * 2 * TILE;
      load(kb, (t + 1) * ROWS, S, next, wid);
      load(vb, (t + 1) * ROWS, S, next + TILE, wid);
    }
  };
  // first all-visible tiles, then those on the diagonal, then those that only
  // other waves need
  const Walk mine = walk(wrow, S);
  int t = 0;
  for (; t < mine.full; ++t) {
    arrive(t);
    const char *kt = smem + (t & 1) * 2 * TILE;
#pragma unroll
    for (int i = 0; i < ROWS; i += SUB * 32 * SPLIT)
      keys(kt, kt + TILE, t * ROWS + i + part * 32, i + part * 32,
           std::false_type{});
  }
  // (TEXT: a branch around the sums would have them moved, so that a half that is
  // hidden from all rows of a wave is computed too)
  const int seen = TEXT ? min(n_tiles, (mine.last + ROWS) / ROWS) : n_tiles;
  for (; t < seen; ++t) {
    arrive(t);
    const char *kt = smem + (t & 1) * 2 * TILE;
#pragma unroll
    for (int i = 0; i < ROWS; i += SUB * 32 * SPLIT) {
      const int r0 = i + part * 32, kbase = t * ROWS + r0;
      if (TEXT || kbase <= mine.last)
        keys(kt, kt + TILE, kbase, r0, std::true_type{});
    }
  }
  for (; t < n_tiles; ++t) arrive(t);

  settle();
  if constexpr (SPLIT == 2) {
    // lane-major pieces of 16 bytes: the result, maximum and sum of part 1
    constexpr int PIECES = DTILES * 4;
    static_assert(PIECES == DH / 8, "merge buffer");
    float4 *ex = reinterpret_cast<float4 *>(smem) +
                 group * (PIECES + 1) * 64 + lane;
    __syncthreads();                        // the last tile has been read
    if (part == 1) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const f32x16v &a = acc_o[i / 4];
        ex[i * 64] = make_float4(a[i % 4 * 4], a[i % 4 * 4 + 1],
                                 a[i % 4 * 4 + 2], a[i % 4 * 4 + 3]);
      }
      ex[PIECES * 64] = make_float4(m_run, l_run, 0.0f, 0.0f);
    }
    __syncthreads();
    if (part == 1) return;
    const float4 ml = ex[PIECES * 64];
    const float mn = fmaxf(m_run, ml.x);
    const float ref = mn == -INFINITY ? 0.0f : mn;
    const float f0 = __builtin_amdgcn_exp2f(m_run - ref);
    const float f1 = __builtin_amdgcn_exp2f(ml.x - ref);
    l_run = l_run * f0 + ml.y * f1;
    m_run = mn;
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const float4 o = ex[i * 64];
      f32x16v &a = acc_o[i / 4];
      a[i % 4 * 4] = a[i % 4 * 4] * f0 + o.x * f1;
      a[i % 4 * 4 + 1] = a[i % 4 * 4 + 1] * f0 + o.y * f1;
      a[i % 4 * 4 + 2] = a[i % 4 * 4 + 2] * f0 + o.z * f1;
      a[i % 4 * 4 + 3] = a[i % 4 * 4 + 3] * f0 + o.w * f1;
    }
  }

  // ---- epilogue: O^T regs -> out[b, qrow, h, :] ---------------------------
  if (q_valid) {
    const float l_full = l_run + __shfl_xor(l_run, 32, 64);
    const float inv_l = (l_full > 0.0f) ? 1.0f / l_full : 0.0f;
    if (lsep != nullptr && hi == 0)
      lsep[((int64_t)b * Hq + h) * S + qrow] =
          (l_full > 0.0f)
              ? (ORDERED ? m_run : m_run / LOG2E) + __logf(l_full)
              : -INFINITY;
    uint16_t *orow = op + ((int64_t)(b * S + qrow) * Hq + h) * DH;
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt) {
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        uint2 w;
        w.x = pack2(acc_o[dt][rq * 4] * inv_l, acc_o[dt][rq * 4 + 1] * inv_l);
        w.y = pack2(acc_o[dt][rq * 4 + 2] * inv_l,
                    acc_o[dt][rq * 4 + 3] * inv_l);
        *reinterpret_cast<uint2 *>(orow + dt * 32 + 8 * rq + 4 * hi) = w;
      }
    }
  }
}

struct Problem {
  const uint16_t *q, *k, *v;
  uint16_t *out;
  float *lse;
  int64_t B, S, Hq, Hkv, q_stride, kv_stride;
  float scale;
};

template <int DH, int NW, int SPLIT, bool ORDERED = false>
void launch_prefill(const Problem &p) {
  constexpr size_t merge =
      SPLIT == 1 ? 0 : (size_t)NW / SPLIT * (DH / 8 + 1) * 1024;
  constexpr size_t shmem = std::max((size_t)4 * tile_bytes<DH>(), merge);
  static const bool once = hipFuncSetAttribute(
      reinterpret_cast<const void *>(
          &flash_prefill_kernel<DH, NW, SPLIT, ORDERED>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) == hipSuccess;
  TORCH_CHECK(once, "flash_prefill: LDS size");
  constexpr int QT = NW / SPLIT * 32;
  const int64_t grid = (p.S + QT - 1) / QT * p.Hq * p.B;
  TORCH_CHECK(grid < (int64_t)1 << 31, "flash_prefill: grid");
  hipLaunchKernelGGL((flash_prefill_kernel<DH, NW, SPLIT, ORDERED>),
                     dim3((unsigned)grid), dim3(NW * 64), shmem,
                     at::hip::getCurrentHIPStream(), p.q, p.k, p.v, p.out,
                     p.lse, (int)p.B, (int)p.S, (int)p.Hq, (int)p.Hkv,
                     p.q_stride, p.kv_stride, p.scale);
}

template <int DH> void launch_prefill(const Problem &p) {
  // Tiles of 32 query rows in all heads: one or two waves each, on 1024 SIMDs.
  // As long as there are fewer of them than SIMDs, the chain of a tile's keys
  // is what takes the time, and two waves halve it; small workgroups then use
  // more CUs. us at 128 columns for <2,2> <4,2> <4,1> <8,1>:
  //   256 tokens, 32 heads ( 256 tiles)   8.3   9.2  10.4  14.1
  //   1000 tokens         (1024 tiles)   29.6  21.6  25.6  31.6
  //   1500 tokens         (1504 tiles)   51.3  34.8  37.4  44.1
  //   2000 tokens         (2016 tiles)   84.1  56.1  51.9  60.1
  //   7931 tokens         (7936 tiles)   1098   614   502   484
  // 256 columns take a SIMD's registers for one wave, so four waves fill a CU
  // (3000 tokens, 16 heads, 1504 tiles: <4,2> 151, <4,1> 141; with eight, which
  // spill, 281).
  const int64_t tiles = (p.S + 31) / 32 * p.Hq * p.B;
  if constexpr (DH == 256) {
    if (tiles <= 1280) launch_prefill<DH, 4, 2>(p);
    else launch_prefill<DH, 4, 1>(p);
  } else {
    if (tiles <= 512) launch_prefill<DH, 2, 2>(p);
    else if (tiles <= 1536) launch_prefill<DH, 4, 2>(p);
    else if (tiles < 6144) launch_prefill<DH, 4, 1>(p);
    else launch_prefill<DH, 8, 1>(p);
  }
}

void launch_prefill(int64_t DH, const Problem &p, bool ordered) {
  TORCH_CHECK(!ordered || DH == 64, "flash_prefill: ordered heads of 64 only");
  if (ordered) launch_prefill<64, 4, 1, true>(p);
  else if (DH == 128) launch_prefill<128>(p);
  else if (DH == 64) launch_prefill<64>(p);
  else if (DH == 256) launch_prefill<256>(p);
  else TORCH_CHECK(false, "flash_prefill: DH must be 64, 128 or 256, got ", DH);
}

}  // namespace

static at::Tensor flash_fwd_impl(at::Tensor q, at::Tensor k, at::Tensor v,
                                 double scale, float *lsep,
                                 bool ordered = false) {
  TORCH_CHECK(q.is_cuda() && q.is_contiguous() && k.is_contiguous() &&
                  v.is_contiguous(), "flash_prefill: contiguous GPU tensors");
  TORCH_CHECK(q.scalar_type() == at::kBFloat16, "flash_prefill: bf16 only");
  TORCH_CHECK(q.dim() == 4, "flash_prefill: q must be [B, S, Hq, DH]");
  const int B = (int)q.size(0), S = (int)q.size(1), Hq = (int)q.size(2),
            DH = (int)q.size(3);
  const int Hkv = (int)k.size(2);
  TORCH_CHECK(Hq % Hkv == 0, "flash_prefill: Hq % Hkv");
  TORCH_CHECK(k.dim() == 4 && k.size(0) == B && k.size(1) == S &&
              k.size(3) == DH && v.sizes() == k.sizes() &&
              k.scalar_type() == at::kBFloat16 &&
              v.scalar_type() == at::kBFloat16, "flash_prefill: k, v");
  auto out = at::empty_like(q);
  if (out.numel() == 0) return out;
  q = flash::aligned16(q);
  k = flash::aligned16(k);
  v = flash::aligned16(v);
  launch_prefill(DH, {(const uint16_t *)q.data_ptr(),
                      (const uint16_t *)k.data_ptr(),
                      (const uint16_t *)v.data_ptr(),
                      (uint16_t *)out.data_ptr(), lsep, B, S, Hq, Hkv,
                      (int64_t)Hq * DH, (int64_t)Hkv * DH, (float)scale},
                 ordered);
  return out;
}

// q, k and v side by side in the rows of y [B * S, (Hq + 2 Hkv) * DH].
static at::Tensor flash_qkv_impl(const at::Tensor &y, int64_t B, int64_t S,
                                 int64_t Hq, int64_t Hkv, int64_t DH,
                                 double scale, float *lse) {
  const int64_t width = (Hq + 2 * Hkv) * DH;
  TORCH_CHECK(y.is_cuda() && y.is_contiguous() && y.dim() == 2 &&
              y.scalar_type() == at::kBFloat16 && y.size(0) == B * S &&
              y.size(1) == width && Hkv > 0 && Hq % Hkv == 0 &&
              reinterpret_cast<uintptr_t>(y.data_ptr()) % 16 == 0,
              "flash_prefill_qkv: y");
  auto out = at::empty({B, S, Hq, DH}, y.options());
  if (out.numel() == 0) return out;
  const uint16_t *p = (const uint16_t *)y.data_ptr();
  launch_prefill(DH, {p, p + Hq * DH, p + (Hq + Hkv) * DH,
                      (uint16_t *)out.data_ptr(), lse, B, S, Hq, Hkv, width,
                      width, (float)scale}, false);
  return out;
}

at::Tensor flash_prefill_qkv(at::Tensor y, int64_t B, int64_t S, int64_t Hq,
                             int64_t Hkv, int64_t DH, double scale) {
  return flash_qkv_impl(y, B, S, Hq, Hkv, DH, scale, nullptr);
}

std::vector<at::Tensor> flash_fwd_train_qkv(at::Tensor y, int64_t B, int64_t S,
                                            int64_t Hq, int64_t Hkv,
                                            int64_t DH, double scale) {
  auto lse = at::empty({B, Hq, S}, y.options().dtype(at::kFloat));
  auto out = flash_qkv_impl(y, B, S, Hq, Hkv, DH, scale,
                            lse.data_ptr<float>());
  return {out, lse};
}

at::Tensor flash_prefill(at::Tensor q, at::Tensor k, at::Tensor v,
                         double scale) {
  return flash_fwd_impl(q, k, v, scale, nullptr);
}

// The walks of the waves of every workgroup of `rows` query rows: {tiles of the
// workgroup, full, last} each.
std::vector<std::vector<int64_t>> flash_walks(int64_t S, int64_t rows) {
  std::vector<std::vector<int64_t>> out;
  for (int64_t q0 = 0; q0 < S; q0 += rows)
    for (int64_t w = q0; w < q0 + rows; w += 32) {
      const Walk k = walk((int)w, (int)S);
      out.push_back({(std::min(S, q0 + rows) + ROWS - 1) / ROWS, k.full,
                     k.last});
    }
  return out;
}

// Training forward: additionally returns the per-row log-sum-exp
// ([B, Hq, S] f32) consumed by fa_bwd (attention_bwd.hip).
std::vector<at::Tensor> flash_fwd_train(at::Tensor q, at::Tensor k,
                                        at::Tensor v, double scale,
                                        bool ordered) {
  const int B = (int)q.size(0), S = (int)q.size(1), Hq = (int)q.size(2);
  auto lse = at::empty({B, Hq, S}, q.options().dtype(at::kFloat));
  auto out = flash_fwd_impl(q, k, v, scale, lse.data_ptr<float>(), ordered);
  return {out, lse};
}

// ---------------------------------------------------------------------------
// Layout probe: one v_mfma_f32_32x32x16_bf16 computing C = A @ B with the
// fragment maps this file assumes. The GPU test compares it against torch
// matmul — if the assumed lane->element maps are wrong, THIS fails first
// and pinpoints the bug (instead of the whole flash kernel).
// a: [32, 16] bf16 (A[i][k]);  b: [16, 32] bf16 (B[k][j]) -> c: [32, 32] f32
// ---------------------------------------------------------------------------
namespace {
__global__ void mfma_probe_kernel(const uint16_t *__restrict__ a,
                                  const uint16_t *__restrict__ b,
                                  float *__restrict__ c) {
  const int lane = threadIdx.x & 63;
  const int hi = lane >> 5;
  const int i = lane & 31;
  union { unsigned short u[8]; bf16x8v v; } af, bf;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    af.u[e] = a[i * 16 + hi * 8 + e];         // A[i][k], k = hi*8+e
    bf.u[e] = b[(hi * 8 + e) * 32 + i];       // B[k][j], j = lane&31
  }
  f32x16v acc = (f32x16v)(0.0f);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af.v, bf.v, acc, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = (r & 3) + 8 * (r >> 2) + 4 * hi;
    c[row * 32 + i] = acc[r];                  // C[row][j = lane&31]
  }
}
}  // namespace

at::Tensor mfma_probe_32x32x16(at::Tensor a, at::Tensor b) {
  TORCH_CHECK(a.is_cuda() && a.scalar_type() == at::kBFloat16);
  TORCH_CHECK(a.sizes() == at::IntArrayRef({32, 16}) &&
              b.sizes() == at::IntArrayRef({16, 32}), "probe shapes");
  auto c = at::zeros({32, 32}, a.options().dtype(at::kFloat));
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, stream,
                     (const uint16_t *)a.contiguous().data_ptr(),
                     (const uint16_t *)b.contiguous().data_ptr(),
                     c.data_ptr<float>());
  return c;
}
