// Attention of a prompt's rows over the paged KV pool on the matrix cores: tiles of up to 32
// consecutive positions of one sequence share every K and V row they read.
// ref: kernels/attention_naive.cu:8-55 (causal GQA attention of a prompt). Values and precision
// are those of the decode kernels in attention.hip: softmax over positions <= the row's own of
// q.k / sqrt(64), scores, weights and sums in fp32, the result rounded once to fp16.
//
// What bounds it: run as decode rows (attention.hip), a prompt of L rows reads its K and V L / 2
// times over and does every product on the vector units: 1507 rows, 32 / 8 heads, 341 us a layer
// for 6 MB of K and V. Here a block holds one kv head of a tile: its waves are the 4 query heads,
// 2 or 4 times over, and a step is as many chunks of 64 positions, one for each set of 4 waves,
// which share it through LDS; the sets meet in LDS at the end. (One set: 59.7 us a layer there,
// bound by the longest block, 24 steps of the last rows; two 42.4, four 36.8.) The products run on
// v_mfma_f32_32x32x16_f16, transposed so that no operand changes lanes between the two:
//   S^T = K Q^T  (A: 32 positions of K from LDS, B: the wave's 32 query rows, held throughout):
//         lane l gets 16 scores of query row l % 32, positions 8 (i / 4) + 4 (l / 32) + i % 4, so
//         a row's maximum is 16 in-lane steps and one exchange with lane l ^ 32;
//   O^T += V^T P^T (A: V transposed into LDS as it arrives, B: the lane's own 16 weights, whose
//         position order the A reads follow).
// Weights stay 32-bit values: each enters the second product as hi + lo, two fp16 halves of
// 2^15 p, which doubles that product's 8 instructions to 16 a chunk; the vector work of the
// softmax (about 6 instructions and one exponential per score) is the larger part. Down to p =
// 2^-20 of the row's maximum the halves are as near as the decode kernels' fp32 weights, whose
// exponents are rounded; below, where lo runs out of exponents, what they leave goes through the
// product once more, 2^39 times as large, which serves to p = 2^-59. Only chunks that hold such a
// weight pay for it: 1507 rows 33.0 -> 34.1 us for finding none, 32.6 -> 59.7 where every chunk has
// some (scores of standard deviation 4). With the scores kept for it, or sums of its own, the
// registers run out: 50 us.
// The running maximum is rounded up to a whole number of log2 units: the offset 15 - m is then
// exact, so the scale 2^15 costs nothing, and rescaling is rarer. That holds for scores below
// kLargeScore; past it (finite, but far from a trained model's) the reference is m + f, f the row's
// largest exponent after m is taken off, and the exponents are made in two steps, so that a row's
// largest weight stays 2^15 however m rounds. The next step's K and V are in registers
// while this one is used. At 4000 rows staging alone (LDS writes, V transposed, two barriers) takes
// 32 of the 156 us, the loads 15.
#include <math.h>

#include <type_traits>

#include "attention.hpp"
#include "common.hpp"

namespace llmk {
namespace {

constexpr int kHeadDim = 64;
constexpr int kGroup = 4;  // query heads per kv head: the block's waves
constexpr int kPage = 16;
constexpr int kKeys = 64;  // positions per chunk
constexpr int kVStride = kKeys + 4;  // halves per row of the transposed V: 8-byte reads of 32 rows
                                     // fall on 64 distinct banks, the writes two to a bank
constexpr float kScoreScale = 0.125f * 1.44269504088896341f;  // 1 / sqrt(64), in log2 units
constexpr float kWeightLog2 = 15.0f;  // weights are held as 2^15 p
// Below it 15 - m is exact and a rounded maximum is at most 2^-4 short of the exact one.
constexpr float kLargeScore = 1048576.0f;
// The halves end at 2^-24, so a weight of 2^kLowLog2 (2^-20 of the row's maximum) is off by at most
// 2^-20 of itself, what rounding its exponent (-16 to -32 there) costs a weight of the decode
// kernels. Of weights below it at most 2^-25 is left: kRest times that fits.
constexpr float kLowLog2 = -5.0f, kLowWeight = 0.03125f, kRest = 549755813888.0f;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int PARTS>
struct Lds {
  union {
    struct {
      u32x4 k[PARTS * kKeys][8];  // 16-byte piece c of position j at [j][c ^ (j & 7)]
      f16 vt[PARTS][kHeadDim][kVStride];
    };
    struct {  // at the end: all sets of waves but the first
      f32x4 acc[kGroup][8][64];
      float m[kGroup][64], f[kGroup][64], l[kGroup][64];
    } merge[PARTS - 1];
  };
  int odd;  // whether some V element is infinite or NaN
};

// Bit 15 or 31 of the sum is set where the half below it is infinite or NaN (exponent all ones).
__device__ __forceinline__ uint32_t not_finite(uint32_t halves) {
  return (halves & 0x7C007C00u) + 0x04000400u;
}

// The halves with those that are not finite replaced by zero.
__device__ __forceinline__ uint32_t finite_only(uint32_t halves) {
  const uint32_t bad = not_finite(halves);
  return halves & ((bad & 0x8000u) ? 0xFFFF0000u : 0xFFFFFFFFu) &
         ((bad & 0x80000000u) ? 0xFFFFu : 0xFFFFFFFFu);
}

// Two weights as packed halves hi (rounded to nearest) and lo = w - hi. The difference reads the
// packed half in place (v_fma_mix_f32, exact): 4 instructions for two weights, 8 with conversions
// back, differences and packing apart.
__device__ __forceinline__ void split_weights(float a, float b, uint32_t& hi, uint32_t& lo) {
  const f16x2 h = {(f16)a, (f16)b};
  hi = __builtin_bit_cast(uint32_t, h);
  float ra, rb;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(ra) : "v"(hi), "v"(a));
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=v"(rb)
      : "v"(hi), "v"(b));
  const f16x2 r = {(f16)ra, (f16)rb};
  lo = __builtin_bit_cast(uint32_t, r);
}

// Grid (n_kv_heads, num_splits, n_tiles): with 8 kv heads, one XCD's L2 serves one head. The
// tiles run last to first, the longest causal ranges of a prompt before the short ones.
template <int PARTS>
__global__ void __launch_bounds__(64 * kGroup * PARTS, 4)
k_attn_prompt(const PromptTile* __restrict__ tiles, const int* __restrict__ positions,
              const int* __restrict__ tables, int max_pages, int pages_per_split, int n_heads,
              int n_kv_heads, int num_splits, const f16* __restrict__ q,
              const f16* __restrict__ k_pool, const f16* __restrict__ v_pool,
              f16* __restrict__ out, float* __restrict__ part_o, float2* __restrict__ part_ml) {
  constexpr int STEP = PARTS * kKeys;  // positions per step: a chunk for each set of kGroup waves
  __shared__ Lds<PARTS> lds;
  const int kvh = blockIdx.x, split = blockIdx.y;
  const PromptTile tile = tiles[gridDim.z - 1 - blockIdx.z];
  const int row0 = __builtin_amdgcn_readfirstlane(tile.row0);
  const int count = __builtin_amdgcn_readfirstlane(tile.count);
  const int pos0 = __builtin_amdgcn_readfirstlane(positions[row0]);
  const int key0 = split * pages_per_split * kPage;
  int key1 = pos0 + count;  // one past the last position that any row attends to
  if (key0 >= key1) return;
  if (key1 - key0 > pages_per_split * kPage) key1 = key0 + pages_per_split * kPage;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int part = wave / kGroup;
  const int tok = lane & 31, half = lane >> 5;
  const int h = kvh * kGroup + wave % kGroup;
  const int row = row0 + (tok < count ? tok : count - 1);
  const int pos = pos0 + (tok < count ? tok : count - 1);
  const int* __restrict__ pages = tables + (size_t)(row0 + count - 1) * max_pages;
  const size_t kv_row = (size_t)n_kv_heads * kHeadDim;  // halves per pool row

  // The thread's pieces of a step: K positions tid / 8 and tid / 8 + STEP / 2, V positions 2 (tid / 8)
  // and the next, all at dims 8 (tid % 8) .. + 7. Past the last cached position the last one is
  // read again: its scores are masked and its V is zeroed.
  const int piece = tid & 7, slot = tid >> 3;
  auto at = [&](int key) {
    const int k = key < key1 ? key : key1 - 1;
    return ((size_t)pages[k / kPage] * kPage + k % kPage) * kv_row + kvh * kHeadDim + piece * 8;
  };
  u32x4 kr[2], vr[2];
  auto load = [&](int base) {
#pragma unroll
    for (int i = 0; i < 2; ++i) kr[i] = ld16(k_pool + at(base + slot + STEP / 2 * i));
#pragma unroll
    for (int i = 0; i < 2; ++i) vr[i] = ld16(v_pool + at(base + 2 * slot + i));
  };

  f16x8 qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    qf[s] = as_h8(ld16(q + ((size_t)row * n_heads + h) * kHeadDim + 16 * s + 8 * half));

  // Weights are relative to 2^(m + f), f = 0 while |m| < kLargeScore; l: this half's positions only
  float m = -INFINITY, f = 0.0f, l = 0.0f;
  f32x16 acc[2];                  // dims 32 d + 8 (i / 4) + 4 half + i % 4
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = 0.0f;

  if (tid == 0) lds.odd = 0;
  load(key0);
  for (int step = key0; step < key1; step += STEP) {
    const bool masked = step + STEP - 1 > pos0;  // some row does not attend to all of it
    __syncthreads();  // the previous step is done with
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = slot + STEP / 2 * i;
      lds.k[key][piece ^ (key & 7)] = kr[i];
      if (step + 2 * slot + i >= key1) vr[i] = u32x4{0u, 0u, 0u, 0u};
    }
    // An infinite or NaN value would turn the zero weights of rows that do not attend to its
    // position, and the low halves of the others, into NaN: it is left out of the product and
    // added at the end.
    uint32_t bad = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      bad |= not_finite(elem(vr[0], e)) | not_finite(elem(vr[1], e));
    if (bad & 0x80008000u) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) vr[i][e] = finite_only(elem(vr[i], e));
      lds.odd = 1;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t a = elem(vr[0], e), b = elem(vr[1], e);
      f16* dst = &lds.vt[2 * slot / kKeys][piece * 8 + 2 * e][2 * slot % kKeys];
      *reinterpret_cast<uint32_t*>(dst) = (a & 0xFFFFu) | (b << 16);
      *reinterpret_cast<uint32_t*>(dst + kVStride) = (a >> 16) | (b & 0xFFFF0000u);
    }
    __syncthreads();
    if (step + STEP < key1) load(step + STEP);
    if (step + kKeys * part >= key1) continue;

    const int own = pos - step - kKeys * part - 4 * half;  // positions past it are masked
    auto scores = [&](int t) {
      f32x16 s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.0f;
      const int key = kKeys * part + 32 * t + tok;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            as_h8(lds.k[key][(2 * c + half) ^ (tok & 7)]), qf[c], s, 0, 0, 0);
      return s;
    };
    auto mask = [&](f32x16& s, int t) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (8 * (i / 4) + i % 4 > own - 32 * t) s[i] = -INFINITY;
    };
    f32x16 s[2] = {scores(0), scores(1)};
    // The lowest score, of positions that the row does not attend to as well.
    float mi[2] = {s[0][0], s[1][0]};
#pragma unroll
    for (int i = 1; i < 16; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) mi[t] = fminf(mi[t], s[t][i]);
    float lowest = fminf(mi[0], mi[1]);
    asm volatile("" : "+v"(lowest));  // now: the scores need not be kept for it
    if (masked) {
#pragma unroll
      for (int t = 0; t < 2; ++t) mask(s[t], t);
    }
    float mx[2] = {s[0][0], s[1][0]};
#pragma unroll
    for (int i = 1; i < 16; ++i)
#pragma unroll
      for (int t = 0; t < 2; ++t) mx[t] = fmaxf(mx[t], s[t][i]);
    float mc = fmaxf(mx[0], mx[1]);
    const auto halves = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, mc),
                                                         __builtin_bit_cast(uint32_t, mc), false,
                                                         false);
    const uint32_t h0 = halves[0], h1 = halves[1];
    mc = fmaxf(__builtin_bit_cast(float, h0), __builtin_bit_cast(float, h1));
    const float mn = fmaxf(m, __builtin_ceilf(mc * kScoreScale));
    const float base = mn == -INFINITY ? 0.0f : mn;  // nothing seen yet: every weight is 0
    float scale = kScoreScale, off = kWeightLog2 - base, fn = 0.0f;
    const bool large =
        __builtin_amdgcn_ballot_w64(__builtin_fabsf(base) >= kLargeScore || f != 0.0f) != 0;
    if (large) {
      const float top = __builtin_fmaf(mc, kScoreScale, -base);
      if (__builtin_fabsf(base) >= kLargeScore) fn = mn > m ? top : fmaxf(f, top);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[t][i] = __builtin_fmaf(s[t][i], kScoreScale, -base) - fn;
      lowest = __builtin_fmaf(lowest, kScoreScale, -base) - fn;
      scale = 1.0f;
      off = kWeightLog2;
    }
    if (__builtin_amdgcn_ballot_w64(mn != m || fn != f)) {
      const float corr = __builtin_amdgcn_exp2f((m - base) + (f - fn));
      l = l * corr;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = acc[d][i] * corr;
    }
    m = mn;
    f = fn;
    unsigned long long low =
        __builtin_amdgcn_ballot_w64(__builtin_fmaf(lowest, scale, off) < kLowLog2);
    asm volatile("" : "+s"(low));
    // 16 positions into the sums: their weights, or kRest times what the halves of the weights
    // below kLowWeight leave of them.
    auto weigh = [&](const f32x16& s, float scale, float off, int t, int c, auto rest) {
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float p[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          p[k] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * c + 2 * e + k], scale, off));
          if constexpr (!rest) l = l + p[k];
        }
        split_weights(p[0], p[1], hi[e], lo[e]);
        if constexpr (rest) {
          const f16x2 h = __builtin_bit_cast(f16x2, hi[e]), r = __builtin_bit_cast(f16x2, lo[e]);
#pragma unroll
          for (int k = 0; k < 2; ++k)
            p[k] = p[k] < kLowWeight ? ((p[k] - (float)h[k]) - (float)r[k]) * kRest : 0.0f;
          split_weights(p[0], p[1], hi[e], lo[e]);
        }
      }
      const f16x8 h8 = as_h8(u32x4{hi[0], hi[1], hi[2], hi[3]});
      const f16x8 l8 = as_h8(u32x4{lo[0], lo[1], lo[2], lo[3]});
      // element e of the lane's weights is position 16 c + 4 half + e, + 4 from e = 4 on
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const f16* v = &lds.vt[part][32 * d + tok][32 * t + 16 * c + 4 * half];
        const uint2 v0 = *reinterpret_cast<const uint2*>(v);
        const uint2 v1 = *reinterpret_cast<const uint2*>(v + 8);
        const f16x8 vf = as_h8(u32x4{v0.x, v0.y, v1.x, v1.y});
        acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, h8, acc[d], 0, 0, 0);
        acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, l8, acc[d], 0, 0, 0);
      }
    };
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < 2; ++c) weigh(s[t], scale, off, t, c, std::false_type{});
    asm volatile("" : "+v"(l));  // now: the weights need not be kept for it
    if (low) {
      // The scores are made again, 32 positions at a time, and the sums are scaled instead of the
      // rest (exactly): the registers of the loop are full.
      float ref = m;
      asm volatile("" : "+v"(ref));
      ref = ref == -INFINITY ? 0.0f : ref;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = acc[d][i] * kRest;
#pragma unroll 1
      for (int t = 0; t < 2; ++t) {
        f32x16 again = scores(t);
        if (masked) mask(again, t);
        if (large) {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            again[i] = __builtin_fmaf(again[i], kScoreScale, -ref) - f;
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
          weigh(again, large ? 1.0f : kScoreScale, kWeightLog2 - (large ? 0.0f : ref), t, c,
                std::true_type{});
      }
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = acc[d][i] * (1.0f / kRest);
    }
  }
  l = l + __shfl_xor(l, 32);

  // The sets of waves: all but the first leave their state in LDS, and the first merges them. A
  // set that saw nothing has m = -inf, l = 0 and weight 0.
  __syncthreads();
  const int w = wave % kGroup;
  if (part > 0) {
    auto& to = lds.merge[part - 1];
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        to.acc[w][4 * d + g][lane] = f32x4{acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2],
                                           acc[d][4 * g + 3]};
    to.m[w][lane] = m;
    to.f[w][lane] = f;
    to.l[w][lane] = l;
  }
  __syncthreads();
  if (part > 0 || tok >= count || key0 > pos) return;
  float M = m, F = f;  // finite unless a score is not: the first set saw position key0
#pragma unroll
  for (int p = 0; p < PARTS - 1; ++p) {
    const float mp = lds.merge[p].m[w][lane], fp = lds.merge[p].f[w][lane];
    if (mp > M || (mp == M && fp > F)) M = mp, F = fp;
  }
  const float own = __builtin_amdgcn_exp2f((m - M) + (f - F));
  l = l * own;
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[d][i] = acc[d][i] * own;
#pragma unroll 1
  for (int p = 0; p < PARTS - 1; ++p) {
    const auto& from = lds.merge[p];
    const float wt = __builtin_amdgcn_exp2f((from.m[w][lane] - M) + (from.f[w][lane] - F));
    l = __builtin_fmaf(from.l[w][lane], wt, l);
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 o = from.acc[w][4 * d + g][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[d][4 * g + e] = __builtin_fmaf(o[e], wt, acc[d][4 * g + e]);
      }
  }
  if (lds.odd) {  // a weight is positive: what it is does not change the sum with these
    for (int key = key0; key < key1 && key <= pos; ++key) {
      const f16* v = v_pool + ((size_t)pages[key / kPage] * kPage + key % kPage) * kv_row +
                     kvh * kHeadDim + 4 * half;
      for (int g = 0; g < 8; ++g)
        for (int e = 0; e < 4; ++e) {
          const float x = (float)v[8 * g + e];
          if (!(__builtin_fabsf(x) < INFINITY)) {
#pragma unroll
            for (int i = 0; i < 32; ++i)
              if (i == 4 * g + e) acc[i / 16][i % 16] = acc[i / 16][i % 16] + x;
          }
        }
    }
  }

  const int P = pos / kPage + 1;
  if ((P + pages_per_split - 1) / pages_per_split == 1) {
    f16* dst = out + ((size_t)row * n_heads + h) * kHeadDim + 4 * half;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f16x2 o[2];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e / 2][e % 2] = (f16)(acc[d][4 * g + e] / l);
        uint2 v;
        v.x = __builtin_bit_cast(uint32_t, o[0]);
        v.y = __builtin_bit_cast(uint32_t, o[1]);
        *reinterpret_cast<uint2*>(dst + 32 * d + 8 * g) = v;
      }
  } else {
    if (F != 0.0f) {  // pieces meet by M alone
      const float c = __builtin_amdgcn_exp2f(F);
      l = l * c;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] = acc[d][i] * c;
    }
    const size_t idx = ((size_t)row * num_splits + split) * n_heads + h;
    float* dst = part_o + idx * kHeadDim + 4 * half;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(dst + 32 * d + 8 * g) =
            make_float4(acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2], acc[d][4 * g + 3]);
    if (half == 0) part_ml[idx] = make_float2(M, l);
  }
}

// Launches of at most this many blocks (two on each CU) run 16 waves to a block, 4 chunks a step
// (unless two hold all of a split's positions):
// the longest block, which ends last, takes half the steps. Past it the CUs are full either way,
// and the wider block's LDS (104 KB, one block on a CU) costs more. One layer, 32 / 8 heads, from
// position 0, 8 / 16 waves, us: 1507 rows 42.4 / 36.8, 2048 rows 57.3 / 55.4, 4000 rows 156 / 170.
constexpr long long kWideBlocks = 512;

template <int PARTS>
int tiles_launch(const PromptAttention& a, float2* ml, hipStream_t stream) {
  return launch(k_attn_prompt<PARTS>,
                dim3((unsigned)a.n_kv_heads, (unsigned)a.splits.num_splits, (unsigned)a.n_tiles),
                dim3(64 * kGroup * PARTS), 0, stream, a.tiles, a.positions, a.tables, a.max_pages,
                a.splits.pages_per_split, a.n_heads, a.n_kv_heads, a.splits.num_splits,
                reinterpret_cast<const f16*>(a.q), reinterpret_cast<const f16*>(a.k_pool),
                reinterpret_cast<const f16*>(a.v_pool), reinterpret_cast<f16*>(a.out),
                a.workspace, ml);
}

}  // namespace

int prompt_attention(const PromptAttention& a, hipStream_t stream) {
  if (a.n_tiles == 0) return LLMK_OK;
  if (a.n_tiles > 65535 || a.splits.num_splits > 65535) return LLMK_ERR_UNSUPPORTED;
  float2* ml = reinterpret_cast<float2*>(a.workspace + (size_t)a.n_rows * a.splits.num_splits *
                                                            a.n_heads * kHeadDim);
  const long long blocks = (long long)a.n_tiles * a.splits.num_splits * a.n_kv_heads;
  const int st = blocks <= kWideBlocks && a.splits.pages_per_split * kPage > 2 * kKeys
                     ? tiles_launch<4>(a, ml, stream)
                     : tiles_launch<2>(a, ml, stream);
  if (st != LLMK_OK || a.splits.num_splits == 1) return st;
  return merge_split_pieces(a.workspace, a.lens, a.out, a.n_rows, a.max_pages, a.n_heads,
                            a.splits.num_splits, a.splits.pages_per_split, stream);
}

}  // namespace llmk
