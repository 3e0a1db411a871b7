// y[T, out] = x[T, in] W^T for 9 to 512 rows on the matrix cores: W stored [out, in] row-major (a
// PyTorch Linear without bias), fp16 in and out, fp32 accumulation. ref: kernels/linear.cu:5-25
// (cublasGemmEx with CUBLAS_COMPUTE_32F).
//
// What bounds it: with this few rows a projection is a stream over W (a few MB to a few hundred)
// between two fixed costs, about 2.3 us from a block's start to its first stage in LDS and 1 to 3
// from its last store to the next kernel's first instruction. hipBLASLt's plans spend 11 us and
// more on the small matrices. So every shape is cut into about one block per CU:
//   - a block computes BN features x BM rows. Stages of BK of the in dimension go from memory
//     straight to LDS (global_load_lds_dwordx4, no registers), ST of them in a ring with one
//     barrier per stage: wait for the stage's loads (counted, the later ones stay in flight),
//     barrier, issue the loads of the slot that the barrier has freed, read, multiply;
//   - 16-byte pieces of a row are XOR-ed by the row's low bits, on the way in by the lane's choice
//     of source and on the way out in the address, so that a fragment read is free of bank
//     conflicts;
//   - the KW sets of a block's waves take different slices of each stage and meet in LDS after the
//     last one, so a wave's accumulators cover a large tile (fewer LDS reads per product) however
//     small the block's tile is;
//   - blocks start at different stages of the in dimension. Rows are a power of two apart, so
//     blocks in step would all read from the same few memory channels: 16384 x 2048 at 40 rows
//     16.3 -> 14.5 us;
//   - a long in dimension over few features is also cut over blocks (splits): fp32 partial sums,
//     added in split order by the consumer or by k_tiles_reduce;
//   - the row tiles of one feature tile run on one XCD, next to each other: W crosses HBM once.
// The product is W x^T (v_mfma_f32_16x16x32_f16, A: 16 features, B: 16 rows of x), so a lane ends
// up with 4 consecutive features of one row. Same box, cold W, inside a graph, us, hipBLASLt's
// first choice -> here (tuned, hipBLASLt takes 8.7, 7.2, 18.2 and 14.3 us at 40 rows, 13.5, 10.4,
// 30.3 and 27.4 at 256):
//   in x out        40 rows        64 rows        128 rows       256 rows
//   2048 x 3072     8.9 -> 6.4     9.3 -> 6.5     12.2 -> 8.1    11.1 -> 11.0
//   2048 x 2048     8.8 -> 6.4     9.2 -> 6.4     8.8 -> 6.6     10.1 -> 8.1
//   2048 x 16384    18.0 -> 14.5   18.1 -> 15.4   22.1 -> 19.8   29.3 -> 26.8
//   8192 x 2048     14.4 -> 12.7   22.6 -> 14.1   21.8 -> 16.4   27.6 -> 21.7
#include "gemm_tiles.hpp"

#include "layer_ops.hpp"

namespace llmk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ void dma16(const void* g, void* wave_base) {
  __builtin_amdgcn_global_load_lds(g, (lds_void*)wave_base, 16, 0, 0);
}
// s_waitcnt vmcnt(VM) lgkmcnt(0) (gfx9 fields): at most VM loads still in flight, and every LDS read
// of the wave returned, so that after the barrier its last stage's slot may be written. The products
// have used those reads by then, so the second wait costs nothing.
template <int VM>
__device__ __forceinline__ void wait_vm() {
  static_assert(VM >= 0 && VM < 64, "waitcnt field range");
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));
}
// s_barrier alone: __syncthreads() would wait for every load in flight.
__device__ __forceinline__ void raw_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ void store4(f16* to, f16x4 v) {
  *reinterpret_cast<uint2*>(to) = __builtin_bit_cast(uint2, v);
}

// What a launch does with the product. The last two take pairs of features, whose sums the tile's
// feature order brings into one lane, and every row of W in one block (no splits).
enum Epi : int {
  kStore = 0,    // y[t][j] = r16(sum)
  kPartial = 1,  // partial[split][t][j] = sum
  kSwiglu = 2,   // features j (gate) and out / 2 + j (up) -> y[t][j] = r16(r16(silu(g)) * u)
  kRope = 3,     // q, k, v heads of 64: RoPE on q and k, k and v into the paged pools
};
constexpr bool paired(int epi) { return epi == kSwiglu || epi == kRope; }

struct TileArgs {
  const f16* x;  // [T, in]
  const f16* w;  // [out, in]
  f16* y;        // [T, out]
  float* partial;  // [splits, T, out]
  int T, in, out, splits;
  int row_tiles, col_tiles;
  RopeTarget rope;  // kRope
};

// The feature at LDS row `row` of the tile's BN features; tile number `tile`. Paired: 16
// features of a wave's 32 are the first halves of its pairs, the next 16 the second halves.
template <class C, int EPI>
__device__ __forceinline__ int feature_of(int tile, int row, int out) {
  if constexpr (paired(EPI)) {
    static_assert(C::TN == 2, "a pair's halves are the wave's two feature tiles");
    const int group = tile * C::WGN + row / 32, half = row / 16 % 2, c = row % 16;
    return EPI == kSwiglu ? half * (out / 2) + 16 * group + c
                          : 64 * (group / 2) + 32 * half + 16 * (group % 2) + c;
  } else {
    return tile * C::BN + row;
  }
}

// TM x TN 16 x 16 products per wave, WGM x WGN waves over the block's rows and features, KW sets
// of them over each stage; KI 32-wide products per wave and stage, ST stages.
template <int TM_, int TN_, int WGM_, int WGN_, int KW_, int KI_, int ST_, int WAVES_PER_SIMD_>
struct Tile {
  static constexpr int TM = TM_, TN = TN_, WGM = WGM_, WGN = WGN_, KW = KW_, KI = KI_, ST = ST_;
  static constexpr int WAVES_PER_SIMD = WAVES_PER_SIMD_;
  static constexpr int BM = 16 * TM * WGM, BN = 16 * TN * WGN, BK = 32 * KW * KI;
  static constexpr int NW = WGM * WGN * KW;          // waves
  static constexpr int PIECES = BK / 8;              // 16-byte pieces of a row in a stage
  static constexpr int ROWS_PER_LOAD = 64 / PIECES;  // rows that one wave's load covers
  static constexpr int LOADS = (BM + BN) / ROWS_PER_LOAD / NW;  // per wave and stage
  static constexpr int STAGE = (BM + BN) * BK;                  // halves
  static constexpr size_t RING = (size_t)ST * STAGE * sizeof(f16);
  static constexpr size_t MEET = KW == 1 ? 0 : (size_t)NW * TM * TN * 64 * sizeof(f32x4);
  static constexpr size_t LDS = RING > MEET ? RING : MEET;
  static_assert(PIECES >= 8, "the XOR moves a piece within 8");
  static_assert(LOADS * NW * ROWS_PER_LOAD == BM + BN && BN % ROWS_PER_LOAD == 0, "whole loads");
  static_assert((ST - 1) * LOADS < 64, "the wait counts every load in flight");
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

template <class C, int EPI>
__global__ void __launch_bounds__(64 * C::NW, C::WAVES_PER_SIMD) k_tiles(TileArgs a) {
  constexpr int TM = C::TM, TN = C::TN, KW = C::KW, BK = C::BK, ST = C::ST, LOADS = C::LOADS;
  extern __shared__ __align__(16) f16 lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kw = wave % KW, wn = wave / KW % C::WGN, wm = wave / KW / C::WGN;

  // Block b runs on XCD b % 8: consecutive tiles go to one XCD, a feature tile's row tiles first.
  const int per_split = a.row_tiles * a.col_tiles, total = per_split * a.splits;
  const int xcd = blockIdx.x % 8, q = total / 8, r = total % 8;
  const int id = xcd * q + (xcd < r ? xcd : r) + (int)blockIdx.x / 8;
  const int split = id / per_split, tile = id % per_split;
  const int tn = tile / a.row_tiles, tm = tile % a.row_tiles;
  const int stages = a.in / BK;
  const int s0 = (int)((long long)stages * split / a.splits);
  const int n = (int)((long long)stages * (split + 1) / a.splits) - s0;
  const int first = n > 0 ? tn % n : 0;  // the stage that this feature tile starts with

  // The wave's loads of a stage: LDS rows (BN features, then BM rows of x) in groups of
  // ROWS_PER_LOAD. Features and rows past the end repeat the last one and are not stored.
  const f16* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int group = wave * LOADS + i;
    const int row = group * C::ROWS_PER_LOAD + lane / C::PIECES;
    const f16* base;
    if (group * C::ROWS_PER_LOAD < C::BN) {
      const int j = feature_of<C, EPI>(tn, row, a.out);
      base = a.w + (size_t)(j < a.out ? j : a.out - 1) * a.in;
    } else {
      const int t = tm * C::BM + row - C::BN;
      base = a.x + (size_t)(t < a.T ? t : a.T - 1) * a.in;
    }
    src[i] = base + (size_t)s0 * BK + ((lane % C::PIECES) ^ (row & 7)) * 8;
  }
  auto issue = [&](int s) {
    f16* to = lds + (s % ST) * C::STAGE + wave * LOADS * 512;
    const int at = s + first < n ? s + first : s + first - n;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) dma16(src[i] + (size_t)at * BK, to + i * 512);
  };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < ST - 1; ++s)
    if (s < n) issue(s);
  const int l16 = lane & 15, lq = lane >> 4;
  for (int s = 0; s < n; ++s) {
    // Issued so far: min(n, s + ST - 1) stages; stage s has landed when those after it are all
    // that is left.
    if (s + ST - 1 <= n)
      wait_vm<(ST - 2) * LOADS>();
    else
      wait_vm<0>();
    raw_barrier();
    if (s + ST - 1 < n) issue(s + ST - 1);  // the slot of stage s - 1, read by every wave
    const f16* st = lds + (s % ST) * C::STAGE;
#pragma unroll
    for (int ki = 0; ki < C::KI; ++ki) {
      const int piece = (kw * C::KI + ki) * 4 + lq;
      f16x8 wf[TN], xf[TM];
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int row = (wn * TN + i) * 16 + l16;
        wf[i] = as_h8(ld16(st + row * BK + (piece ^ (row & 7)) * 8));
      }
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int row = C::BN + (wm * TM + j) * 16 + l16;
        xf[j] = as_h8(ld16(st + row * BK + (piece ^ (row & 7)) * 8));
      }
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[i], xf[j], acc[i][j], 0, 0, 0);
    }
  }

  // The KW sets meet in LDS: set kw adds up the vectors v with v % KW == kw.
  f32x4* meet = reinterpret_cast<f32x4*>(lds) + (size_t)(wave - kw) * TN * TM * 64 + lane;
  if constexpr (KW > 1) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) meet[((size_t)kw * TN * TM + i * TM + j) * 64] = acc[i][j];
    __syncthreads();
  }
  auto total_of = [&](int i, int j) {
    if constexpr (KW == 1) return acc[i][j];
    const int v = i * TM + j;
    f32x4 sum = meet[(size_t)v * 64];
#pragma unroll
    for (int k = 1; k < KW; ++k) sum = sum + meet[((size_t)k * TN * TM + v) * 64];
    return sum;
  };
  if constexpr (paired(EPI)) {
    const int group = tn * C::WGN + wn;
    // The set's pairs of vectors: j = kw, kw + KW, ...
    constexpr int NJ = (TM + KW - 1) / KW;
    f16x4 lo[NJ], hi[NJ];
#pragma unroll
    for (int m = 0; m < NJ; ++m) {
      const int j = kw + KW * m;
      f32x4 a0 = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, a1 = a0;
      if constexpr (KW == 1) {
        a0 = acc[0][m];
        a1 = acc[1][m];
      } else if (j < TM) {
        a0 = total_of(0, j);
        a1 = total_of(1, j);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lo[m][e] = (f16)a0[e];
        hi[m][e] = (f16)a1[e];
      }
    }
    if constexpr (EPI == kSwiglu) {
      constexpr int NV = (NJ + 1) / 2;  // vectors of 8 gates; a spare half holds 1.0
      u32x4 g[NV], sv[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        f16x8 gh;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          gh[e] = 2 * v + e / 4 < NJ ? lo[2 * v + e / 4 < NJ ? 2 * v + e / 4 : 0][e % 4] : (f16)1.0f;
        g[v] = as_u4(gh);
      }
      silu_vectors<NV>(g, sv);
#pragma unroll
      for (int m = 0; m < NJ; ++m) {
        const int j = kw + KW * m, t = tm * C::BM + (wm * TM + j) * 16 + l16;
        const int col = 16 * group + 4 * lq;
        if (j >= TM || t >= a.T || col >= a.out / 2) continue;
        const f16x8 sh = as_h8(sv[m / 2]);
        f16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = sh[4 * (m % 2) + e] * hi[m][e];
        store4(a.y + (size_t)t * (a.out / 2) + col, o);
      }
    } else {
      const RopeTarget& to = a.rope;
      const int h = group / 2, i0 = 16 * (group % 2) + 4 * lq;
      const int nq = to.n_heads, nkv = to.n_kv_heads;
      if (h >= nq + 2 * nkv) return;
#pragma unroll
      for (int m = 0; m < NJ; ++m) {
        const int j = kw + KW * m, t = tm * C::BM + (wm * TM + j) * 16 + l16;
        if (j >= TM || t >= a.T) continue;
        f16x4 x1 = lo[m], x2 = hi[m];
        if (h < nq + nkv) {
          const u32x4 cs = ld16(to.cos_sin + (size_t)t * 32 + i0);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const f16x2 p = __builtin_bit_cast(f16x2, elem(cs, e));
            x1[e] = lo[m][e] * p[0] - hi[m][e] * p[1];
            x2[e] = hi[m][e] * p[0] + lo[m][e] * p[1];
          }
        }
        f16* dst;
        if (h < nq) {
          dst = to.q_out + ((size_t)t * nq + h) * 64;
        } else {
          const int hk = h < nq + nkv ? h - nq : h - nq - nkv;
          dst = (h < nq + nkv ? to.k_pool : to.v_pool) +
                ((size_t)to.pool_rows[t] * nkv + hk) * 64;
        }
        store4(dst + i0, x1);
        store4(dst + i0 + 32, x2);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        if ((i * TM + j) % KW != kw) continue;
        const int t = tm * C::BM + (wm * TM + j) * 16 + l16;
        const int f = tn * C::BN + (wn * TN + i) * 16 + lq * 4;
        if (t >= a.T || f >= a.out) continue;
        const f32x4 sum = total_of(i, j);
        if constexpr (EPI == kPartial)
          *reinterpret_cast<f32x4*>(a.partial + ((size_t)split * a.T + t) * a.out + f) = sum;
        else
          store4(a.y + (size_t)t * a.out + f,
                 f16x4{(f16)sum[0], (f16)sum[1], (f16)sum[2], (f16)sum[3]});
      }
  }
}

// y = r16 of the partial sums, added in split order: 4 values per thread (out is a multiple of 4).
__global__ void __launch_bounds__(256)
k_tiles_reduce(const float* __restrict__ partial, f16* __restrict__ y, size_t n, int splits) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 sum = *reinterpret_cast<const f32x4*>(partial + i);
  for (int s = 1; s < splits; ++s)
    sum = sum + *reinterpret_cast<const f32x4*>(partial + (size_t)s * n + i);
  store4(y + i, f16x4{(f16)sum[0], (f16)sum[1], (f16)sum[2], (f16)sum[3]});
}

// The tile shapes, smallest first, features x rows. More waves to a tile issue its loads faster (a
// wave alone gets about 12 bytes a ns into LDS, 16 waves 110 together): 32x64 with 8 waves of 32x32
// instead of 4 of 64x32 10.2 -> 9.6 us (2048 x 3072, 128 rows), 64x128 with 16 waves in one block
// instead of 8 in each of two 20.3 -> 19.2 (2048 x 16384, 128 rows). 128x128 takes 26 us at 256
// rows of that matrix with 4, 8 or 16 waves, one block or two, and any ring depth.
using T32x32 = Tile<2, 2, 1, 1, 4, 1, 4, 2>;
using T32x64 = Tile<2, 2, 2, 1, 4, 1, 4, 4>;
using T64x64 = Tile<2, 2, 2, 2, 2, 2, 3, 2>;
using T64x128 = Tile<2, 2, 4, 2, 2, 2, 3, 4>;
using T128x128 = Tile<4, 2, 2, 4, 1, 2, 4, 2>;
constexpr int kTiles = 5;
// What a launch takes by shape, in us, with the blocks in rounds of one per CU and `n` stages of 128
// to a block: start + (stage + full * the share of CUs with a block) * n, and round + round_stage *
// n for each round after the first. Fitted to sweeps of every shape and split count over 9 to 512
// rows of 22 matrices (2048 x 2048, 3072, 16384 and 32000, 8192 and 6144 x 2048, 1024 x 1024, 1536
// and 8192, 4096 x 1024, 4096, 6144 and 24576, 12288 x 4096, 3072 x 3072, 4608 and 8192, 9216 x
// 3072, 512 x 512, 640 x 4100, 256 x 16384, 16384 x 1024; cold W, in a graph) and tried on 18 more:
// the choice it leads to takes 0.6% more than the fastest on average, 13% at most.
struct Shape {
  int bm, bn;
  float start, stage, full, round, round_stage;
  float piece;  // partial sums, per MB
};
constexpr Shape kShapes[kTiles] = {{32, 32, 2.72f, 0.24f, 0.04f, 0.90f, 0.18f, 0.18f},
                                   {64, 32, 3.28f, 0.25f, 0.10f, 1.77f, 0.31f, 0.20f},
                                   {64, 64, 3.55f, 0.40f, 0.16f, 2.17f, 0.46f, 0.12f},
                                   {128, 64, 4.57f, 0.57f, 0.24f, 2.95f, 0.72f, 0.14f},
                                   {128, 128, 3.88f, 0.89f, 0.49f, 2.94f, 1.10f, 0.17f}};

long long tile_blocks(const Shape& s, int T, int out) {
  return (long long)((T + s.bm - 1) / s.bm) * ((out + (long long)s.bn - 1) / s.bn);
}

template <class C, int EPI>
int tile_launch(TileArgs a, hipStream_t stream) {
  a.row_tiles = (a.T + C::BM - 1) / C::BM;
  a.col_tiles = (a.out + C::BN - 1) / C::BN;
  // More than 64 KiB of LDS has to be asked for, once per kernel and device.
  static int granted[64];
  int dev = 0;
  int st = (int)hipGetDevice(&dev);
  if (st != LLMK_OK) return st;
  if (dev < 0 || dev >= 64) return LLMK_ERR_UNSUPPORTED;
  if (!__atomic_load_n(&granted[dev], __ATOMIC_RELAXED)) {
    st = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(k_tiles<C, EPI>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS);
    if (st != LLMK_OK) return st;
    __atomic_store_n(&granted[dev], 1, __ATOMIC_RELAXED);
  }
  const long long blocks = (long long)a.row_tiles * a.col_tiles * a.splits;
  if (blocks > 0x7FFFFFFFLL) return LLMK_ERR_UNSUPPORTED;
  return launch(k_tiles<C, EPI>, dim3((unsigned)blocks), dim3(64 * C::NW), C::LDS, stream, a);
}

template <int EPI>
int tiles_launch(int tile, const TileArgs& a, hipStream_t stream) {
  switch (tile) {
    case 0: return tile_launch<T32x32, EPI>(a, stream);
    case 1: return tile_launch<T32x64, EPI>(a, stream);
    case 2: return tile_launch<T64x64, EPI>(a, stream);
    case 3: return tile_launch<T64x128, EPI>(a, stream);
    default: return tile_launch<T128x128, EPI>(a, stream);
  }
}

}  // namespace

// Where this library's tiles beat hipBLASLt's first choice; us, hipBLASLt / here. Up to 128 rows they
// do, except past 24 rows of more than a round of 128 x 128 tiles if the product is short or, past
// 32, its last round mostly empty: 1024 x 128256 at 16 rows 52.8 / 51.9, at 64 rows 59.1 / 64.7, 2048
// x 40000 (1.2 rounds) at 32 rows 40.8 / 33.6, at 64 rows 43.0 / 46.2, 2048 x 128256 (3.9 rounds) 126
// / 113. Past 128 rows hipBLASLt's larger tiles win:
//   - more than a round of 128 x 128 tiles: 4096 x 24576 at 160 rows 54.6 / 83, 2048 x 32000 at 256
//     43 / 53 (at most a round: 2048 x 16384 at 256 rows 30 / 27, 4096 x 8192 41 / 31);
//   - 129 to 224 rows with more than a round of 64 x 64 tiles but no more than half a round of 128 x
//     128 (less than half where in < 2048), unless a launch after them goes too: 4096 x 8192 at 129
//     rows 25.7 / 27.9, 3072 x 8192 21.2 / 23.3, 4096 x 6144 at 200 rows 26.5 / 28.5 (at 160 rows
//     28.1 / 26.6, at 256 40 / 28; 1024 x 8192 at 129 rows 12.8 / 10.9; past half a round: 2048 x
//     12288 at 129 to 256 0.88 to 0.95 of it);
//   - past 256 rows more than a round of 64 x 64 tiles, unless a launch goes too or the product is
//     3 times as long as wide: 4096 x 6144 at 300 rows 30.7 / 38.7, 4096 x 4096 26.0 / 26.6, 2048 x
//     6144 1.24 of it (6144 x 2048 0.75, 8192 x 2048 0.73, 9216 x 3072 0.90, 16384 x 4096 0.90; in one
//     round 1024 x 1536 0.65, 2048 x 3072 0.99, 3072 x 3072 0.90).
bool tiles_apply(const void* x, const void* w, const void* y, int T, int in, int out, bool fused) {
  if (T <= LLMK_LINEAR_ROWS_MAX || T > kTilesMaxRows || in % 128 != 0 || out % 4 != 0 ||
      !aligned16(x) || !aligned16(w) || (reinterpret_cast<uintptr_t>(y) & 7u) != 0)
    return false;
  const int cus = device_cus();
  const long long large = tile_blocks(kShapes[kTiles - 1], T, out);
  if (T <= 128) {
    const long long rounds = (large + cus - 1) / (cus > 0 ? cus : 1);
    return large <= cus || T <= 24 ||
           (in >= 2048 && (T <= 32 || 20 * large >= 17 * rounds * cus));
  }
  const bool one_round = tile_blocks(kShapes[2], T, out) <= cus;
  if (large > cus) return false;
  if (fused || one_round) return true;
  if (T > 256) return in >= 3LL * out;
  return T > 224 || 2 * large > cus || (in < 2048 && 2 * large == cus);
}

// The cheapest shape and split count by the model at kShapes; pieces are read again, by
// k_tiles_reduce, with reduce_launch, or by the consumer: the residual add and norm of 256 rows of
// 2048 take 5.1 us over 1, 4 or 8 pieces, so what counts there is the launch before it (8192 x 2048 at
// 256 rows: 128 x 128 in 8 pieces 17.8 us, 128 x 64 in 4 19.3). The model does not know that wide
// matrices past kWideW weights come from HBM alone. Their fastest shape stages the fewest bytes (128
// x 128), or, if W takes more than a round of it, to 32 rows, multiplies the least (32 x 32): 2048 x
// 128256 with 32 x 32 / 64 x 64 / 128 x 128 tiles at 16 rows 92 / 102 / 100 us, at 64 rows 150 / 117 /
// 113; 4096 x 24576, one round, at 16 rows 37.0 / 43 / 40.8, at 64 rows 50 / 48 / 42.7.
constexpr long long kWideW = 64 << 20;
constexpr int kWideOut = 16384;

TilePlan tiles_plan(int T, int in, int out, size_t max_floats, bool reduce_launch) {
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const bool rounds = tile_blocks(kShapes[kTiles - 1], T, out) > cus;
  if ((long long)in * out >= kWideW && out >= kWideOut && (T > 24 || rounds))
    return {T <= 32 && rounds ? 0 : kTiles - 1, 1};
  TilePlan best = {0, 1};
  float best_us = 0.0f;
  const float per_cu = 1.0f / (float)cus;
#pragma unroll
  for (int tile = 0; tile < kTiles; ++tile) {
    const Shape& s = kShapes[tile];
    const float one = (float)tile_blocks(s, T, out) * per_cu;  // rounds of one split
    for (int splits = 1; splits <= 8 && splits <= in / 128; splits *= 2) {
      const size_t floats = (size_t)splits * T * out;
      if (splits > 1 && floats > max_floats) break;
      const float mb = (float)floats * 4e-6f;
      const float n = (float)in / 128.0f / (float)splits, rounds = one * (float)splits;
      const float more = rounds > 1.0f ? __builtin_ceilf(rounds - 1e-3f) - 1.0f : 0.0f;
      const float share = rounds < 1.0f ? rounds : 1.0f;
      float us = s.start + (s.stage + s.full * share) * n + more * (s.round + s.round_stage * n);
      if (splits > 1)
        us += s.piece * mb + (reduce_launch ? 1.4f + 0.18f * mb + 0.30f * (float)splits
                                            : 0.5f + 0.20f * (float)splits);
      if ((tile == 0 && splits == 1) || us < best_us) {
        best = {tile, splits};
        best_us = us;
      }
    }
  }
  return best;
}

namespace {

TileArgs tile_args(const uint16_t* x, const uint16_t* w, int T, int in, int out, int splits) {
  TileArgs a = {};
  a.x = reinterpret_cast<const f16*>(x);
  a.w = reinterpret_cast<const f16*>(w);
  a.T = T;
  a.in = in;
  a.out = out;
  a.splits = splits;
  return a;
}

}  // namespace

int tiles_linear(const TilePlan& p, const uint16_t* x, const uint16_t* w, uint16_t* y,
                 float* partial, int T, int in, int out, hipStream_t stream) {
  TileArgs a = tile_args(x, w, T, in, out, p.splits);
  a.y = reinterpret_cast<f16*>(y);
  a.partial = partial;
  if (p.splits == 1) return tiles_launch<kStore>(p.tile, a, stream);
  const int st = tiles_launch<kPartial>(p.tile, a, stream);
  if (st != LLMK_OK) return st;
  const size_t n = (size_t)T * out;
  return launch(k_tiles_reduce, dim3(ceil_div(n, 1024)), dim3(256), 0, stream,
                (const float*)partial, a.y, n, p.splits);
}

int tiles_partial(const TilePlan& p, const uint16_t* x, const uint16_t* w, float* partial, int T,
                  int in, int out, hipStream_t stream) {
  TileArgs a = tile_args(x, w, T, in, out, p.splits);
  a.partial = partial;
  return tiles_launch<kPartial>(p.tile, a, stream);
}

int tiles_swiglu(const uint16_t* x, const uint16_t* w_gate_up, uint16_t* act, int T, int in,
                 int inter, hipStream_t stream) {
  TileArgs a = tile_args(x, w_gate_up, T, in, 2 * inter, 1);
  a.y = reinterpret_cast<f16*>(act);
  return tiles_launch<kSwiglu>(tiles_plan(T, in, 2 * inter, 0, false).tile, a, stream);
}

int tiles_qkv_rope_scatter(const uint16_t* x, const uint16_t* w_qkv, const RopeTarget& to, int T,
                           int in, hipStream_t stream) {
  const int out = (to.n_heads + 2 * to.n_kv_heads) * 64;
  TileArgs a = tile_args(x, w_qkv, T, in, out, 1);
  a.rope = to;
  return tiles_launch<kRope>(tiles_plan(T, in, out, 0, false).tile, a, stream);
}

// Two rows per block, a thread per rotation pair: a pass's (cos, sin) pairs and pool rows, once
// for all layers.
namespace {
__global__ void __launch_bounds__(64)
k_rope_rows(const int* __restrict__ positions, const int* __restrict__ tables,
            const float* __restrict__ inv_freq, int max_pages, int n, f16x2* cos_sin,
            long long* pool_rows) {
  const int t = blockIdx.x * 2 + (threadIdx.x >> 5), i = threadIdx.x & 31;
  if (t >= n) return;
  const int pos = positions[t];
  f16 c, s;
  cos_sin_f16((float)pos * inv_freq[i], &c, &s);
  cos_sin[(size_t)t * 32 + i] = f16x2{c, s};
  if (i == 0)
    pool_rows[t] = (long long)tables[(size_t)t * max_pages + pos / 16] * 16 + pos % 16;
}
}  // namespace

int rope_rows(const int32_t* positions, const int32_t* tables, const float* inv_freq,
              int max_pages, int n, void* cos_sin, long long* pool_rows, hipStream_t stream) {
  return launch(k_rope_rows, dim3(ceil_div((size_t)n, 2)), dim3(64), 0, stream, positions, tables,
                inv_freq, max_pages, n, static_cast<f16x2*>(cos_sin), pool_rows);
}

}  // namespace llmk
