// Grouped FP32 GEMM on the BF16 matrix cores (v_mfma_f32_32x32x16_bf16).
//
// The FP32 matrix instructions run at 157 TFLOP/s, the BF16 ones at 2.5 PFLOP/s
// with FP32 accumulation. Every operand is split into three BF16 numbers,
//     x0 = bf16(x),   x1 = bf16(x - x0),   x2 = bf16(x - x0 - x1),
// rounded to nearest; the differences are exact in FP32, and x0 + x1 + x2 = x: all 24
// bits over FP32's own exponent range, without scales. A product is
//     x y = x0 y0 + (x0 y1 + x1 y0) + (x1 y1 + x0 y2 + x2 y0) + ...;
// the first six terms are computed (six MFMAs), the others are at most 2^-25 of the
// product and left out. x0 y0 is summed in one FP32 accumulator and the five small
// terms in another, which is added once at the end: the large sum is rounded once
// per 16 k instead of once per 4 k as on the FP32 instructions. Against 64-bit sums
// the result is closer than the FP32 instructions' (2-norm error, this / FP32 MFMA,
// 1e-7: N(0,1) operands K = 128 0.65 / 2.03, K = 1024 1.86 / 5.73, K = 4096 3.96 / 11.4;
// non-negative K = 128 0.62 / 1.59; both half zero K = 128 0.43 / 1.04; K = 1024 with 16
// nonzero values a row 0.34 / 0.74, with one 0.26 / 0.25), whatever the scales of
// features and weights, and a row of one 1 returns its weight row exactly.
// (Two FP16 numbers, scaled per row and column, and three products took two thirds
// of the time - T = 8192, E = 8, K = 4096, N = 14336 call 6.8 ms against 9.8, chain T =
// 16384, E = 128, K = 2048, N = 768 600 us against 800 - but hold 23 bits over 2^30 of
// range: values 2^-20 and less of the one that set the scale lost bits without a
// sign. Marking rows that have such values for the FP32 instructions cost 3 to 7 %
// and left single ones wrong; correcting those spilled the loop's registers.)
//
// Outputs that are not finite (an infinity or NaN in an operand, |x| that rounds past
// BF16's range, an overflowing sum) or not zero and below 2^-80 (operands under 2^-109
// have parts below BF16's least value, 2^-133; met by values up to 2^20 they make
// nothing larger: x of 2^-114 times w of 2^40, 2^-74, is off by 5.6e-7, of 2^-110 by
// 1.05e-7) are computed again on the FP32 instructions, with the bits of the
// FP32 kernels, in a second pass of the tile over its slices that multiplies only
// 16-row blocks with such an output (E = 8, 16384 rows, K = 4096, N = 14336, one infinite
// row in a thousand 9.0 -> 12.5 ms; all on the FP32 kernel 13.8). Which outputs those
// are is a matter of each one's own value, so that no row's bits depend on the
// rows it shares a tile with, or on the tile's height.
//
// Work split: output tiles of 128 columns and 128 or 256 rows on four or eight
// waves (split_grouped picks), tiles dealt as in gemm.hip. A slice of 16 k of
// both operands is loaded into registers one slice ahead, or two where registers
// are left (16-byte A quads, 8-byte B pairs; rows may start at any 4-byte boundary;
// two ahead: chain T = 16384, E = 128, K = 2048, N = 768 842 -> 798 us), split there (5.5
// instructions an element), and written to LDS as three BF16 planes in MFMA
// operand order (k contiguous per row of A and per column of B), two stages. Four
// waves: two workgroups share a CU and one's MFMAs run under the other's staging.
// Eight waves: the two halves of the workgroup run a phase apart, so that one has
// the matrix pipe while the other stages. Tiles with few rows take layouts of fewer
// 32-row blocks. (Slices of 32 k: 96 KiB of planes for four waves, one workgroup a
// CU, and no registers for both halves' operands.)
// Loads are buffer loads (scalar base, 32-bit lane offset), which need no address
// registers or arithmetic of the lanes.
//
// Large problems: matrix pipes busy 65 % of the cycles at 1.70 of 2.4 GHz (the power
// limit holds the clock down): E = 8, K = 4096, N = 14336, 16384 rows (1.92 TFLOP) FP32
// instructions 13.8 ms, four waves 10.8, eight waves on 256 rows 9.0 (213 TFLOP/s of
// FP32 products, 1.28 PFLOP/s of BF16 ones), 6.7 ms with operands of ones, which
// draw less power. Elsewhere by each tile's serial parts and the combine: pipes busy
// 44 % in the chain T = 16384, E = 128, K = 2048, N = 768 at 1.9 GHz, 24 % in T = 2048, E =
// 64, K = 1024, N = 512. (B staged as columns instead of column pairs in the eight-wave
// shapes: a fifth of the LDS conflicts, 42 % of its index cycles, but twice the loads:
// no faster anywhere, chain T = 2048 79 -> 82 us.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "split_gemm.h"
#include "tiles.h"
#include "wave.h"

namespace rr::kern {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kParts = 3;                   // BF16 parts of a value
constexpr int kBN = 128, kBK = 16;
constexpr int kPlaneB = kBN * kBK;          // values of one plane (part) of B (4 KiB)
constexpr int kBufferFlags = 0x00027000;    // raw 32-bit buffer

// BM x 128 output tiles on W waves (four: two workgroups per CU; eight: one).
template <int W, int BM>
struct Shape {
  static constexpr int kWaves = W;
  static constexpr int kThreads = 64 * W;
  static constexpr int kBM = BM;
  static constexpr int kPassRows = 16 * W;                       // rows of A staged per pass
  static constexpr int kKPer = kBK / W;                          // k rows of B a thread stages
  static constexpr int kPlaneA = kBM * kBK;                      // values
  static constexpr int kStage = kParts * (kPlaneA + kPlaneB);    // A's planes, B's planes
  static constexpr int kStage32 = (kBM + kBN) * kBK;             // floats
  static constexpr int kMaskAt = 2 * kStage32;                   // masks of the outputs to recompute: words from here
  static_assert((kMaskAt + kBM * (kBN / 32)) * sizeof(float) <= 2 * kStage * sizeof(__bf16),
                "two FP32 slices and the masks fit the stages");
};

// Wave tiles of TM x TN blocks of 32 x 32. GRID: W / 2 x 2 waves of TN = 2 column
// blocks; else W / 4 x 4 waves of one.
template <int W, int TM_, bool GRID>
struct Layout {
  static constexpr int TM = TM_;
  static constexpr int TN = GRID ? 2 : 1;
  static constexpr int kRows = TM_ * 32 * (GRID ? W / 2 : W / 4);
  static constexpr int kPasses = (kRows + 16 * W - 1) / (16 * W);  // staging passes that hold the tile's rows
  __device__ static int row(int wave) { return (GRID ? wave >> 1 : wave >> 2) * 32 * TM_; }
  // first tile column
  __device__ static int col(int wave) { return GRID ? 64 * (wave & 1) : 32 * (wave & 3); }
};

// A plane row holds 16 k, two 16-byte chunks; chunk c of row r sits at chunk
// c ^ swizzle(r), so that the 16 rows read together, and 16 rows written together,
// land in distinct bank groups. Column c of B has plane row c / 2 (odd columns 64
// further): a thread stages columns 2 l and 2 l + 1, its wave adjacent rows.
__device__ __forceinline__ int swizzle(int r) { return ((r >> 3) ^ (r >> 6)) & 1; }
__device__ __forceinline__ int plane_row(int c) { return (c >> 1) | ((c & 1) << 6); }

// The BF16 parts of two values (see the file comment): eleven instructions.
__device__ __forceinline__ void split2(float x0, float x1, uint32_t (&part)[kParts]) {
  typedef float f2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int i = 0; i < kParts; ++i) {
    part[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x0, x1}, b2));
    if (i + 1 < kParts) {
      x0 -= __uint_as_float(part[i] << 16);
      x1 -= __uint_as_float(part[i] & 0xFFFF0000U);
    }
  }
}

// Sums that the parts cannot be trusted with: not finite, or nonzero and below 2^-80.
__device__ __forceinline__ bool untrusted(float v) {
  constexpr uint32_t kLeast = (127U - 80U) << 23;
  const uint32_t bits = __float_as_uint(v) & 0x7FFFFFFFU;
  return bits - kLeast >= 0x7F800000U - kLeast && bits != 0;
}

// What a tile needs from the kernel (all workgroup-uniform).
struct Tile {
  const float* B;  // the expert's weights
  int row0, rows;  // first segment row, rows in the tile (1..kBM)
  int n0, ct;      // first column, column tile
};
struct Lds {
  __bf16* stages;    // [2][kStage]
  int32_t* src;      // [kBM] chain: token row of X per tile row (-1: none)
  float* w;          // [kBM] chain: route weight per tile row
};

// One output tile for one wave layout (L::kPasses passes hold its rows).
template <class S, class L, bool CHAIN>
__device__ __forceinline__ void run_tile(const GemmParams& prm, const Tile& tl, const Lds& sh, int col_tiles, int wave) {
  constexpr int W = S::kWaves;
  constexpr int P = L::kPasses;
  constexpr int PR = S::kPassRows;
  constexpr int KP = S::kKPer;
  constexpr int TM = L::TM, TN = L::TN;
  // (the thread id passes an empty asm so that nothing of this is built before
  // the tile loop, for all four layouts, and kept live across it)
  int tid = static_cast<int>(threadIdx.x);
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int K = prm.K;
  const int N = prm.N;
  const int rows = tl.rows;
  const int nk = (K + kBK - 1) / kBK;
  // the last slice is loaded float by float where a quad or pair could cross
  // the end of a row
  const int guarded = (K % kBK != 0 || (N & 1) != 0) ? nk - 1 : nk;
  const int li = lane & 31;
  const int hi = lane >> 5;
  // staging: A quad ac of row PR p + ar; B columns 2 pair, 2 pair + 1 at k
  // KP wave .. + KP - 1
  const int ar = tid >> 2;
  const int ac = tid & 3;
  const int pair = lane;
  const int a_put = ar * kBK + (((ac >> 1) ^ swizzle(ar & 63)) << 3) + ((ac & 1) << 2);
  const int b_k = KP * wave;
  const int b_put = pair * kBK + (((b_k >> 3) ^ swizzle(pair)) << 3) + (b_k & 7);
  const int b_put1 = (64 + pair) * kBK + (((b_k >> 3) ^ swizzle(64 + pair)) << 3) + (b_k & 7);
  // passes that hold rows of the layout for this wave
  auto staged = [&](int p) { return L::kRows % PR == 0 || PR * p + 16 * wave < L::kRows; };

  // Rows past the tile's last read a row that exists (their products land in
  // output rows that are never stored); columns past N the last pair.
  // Loads take a workgroup-uniform base, a 32-bit byte offset per lane and one
  // per instruction in a scalar register (split_gemm_fits bounds the sizes), so
  // that the slices need no address registers or arithmetic of the lanes.
  const auto a_base = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(CHAIN ? prm.X : prm.X + static_cast<std::size_t>(tl.row0) * K), 0, -1, kBufferFlags);
  const auto b_base = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(tl.B), 0, -1, kBufferFlags);
  uint32_t a_lane[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int r = PR * p + ar;
    int src = r < rows ? r : 0;
    if constexpr (CHAIN) {
      src = sh.src[r];
      if (src < 0) src = 0;
    }
    a_lane[p] = 4u * (static_cast<uint32_t>(src) * static_cast<uint32_t>(K) + 4u * static_cast<uint32_t>(ac));
  }
  const int n = tl.n0 + 2 * pair;
  const int nl = n < N ? n : N - 2;
  const uint32_t b_lane = 4u * (static_cast<uint32_t>(b_k) * static_cast<uint32_t>(N) + static_cast<uint32_t>(nl));
  auto b_row = [&](int kt, int j) {  // bytes from tl.B to its k row kBK kt + j
    return 4u * (static_cast<uint32_t>(kt) * kBK + static_cast<uint32_t>(j)) * static_cast<uint32_t>(N);
  };

  struct Slice {  // as loaded
    f4u a[P];
    f2u b[KP];
  };
  auto load = [&](int kt, Slice& s) {  // whole slices
#pragma unroll
    for (int p = 0; p < P; ++p) {
      if (staged(p)) s.a[p] = __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(a_base, a_lane[p], 4 * kBK * kt, 0));
    }
    // (a pair that crosses N reads the next k row's first float)
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      s.b[j] = __builtin_bit_cast(f2u, __builtin_amdgcn_raw_buffer_load_b64(b_base, b_lane, b_row(kt, j), 0));
    }
  };
  auto load_any = [&](int kt, Slice& s) {
    if (kt != guarded) {
      load(kt, s);
      return;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v = 0.0F;
        if (kt * kBK + 4 * ac + q < K) {
          v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(a_base, a_lane[p] + 4 * q, 4 * kBK * kt, 0));
        }
        s.a[p][q] = v;
      }
    }
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      float v0 = 0.0F, v1 = 0.0F;
      if (kt * kBK + b_k + j < K) {
        v0 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b_base, b_lane, b_row(kt, j), 0));
        if (nl + 1 < N) v1 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b_base, b_lane + 4, b_row(kt, j), 0));
      }
      s.b[j] = f2u{v0, v1};
    }
  };

  // Gathered rows go to x_permuted spread over the column tiles: tile ct
  // writes the pairs of k slices 2 i, 2 i + 1 (128 bytes a row) with i % col_tiles == ct.
  // Plain stores: rows of odd lengths share 64-byte blocks between slices, which only the
  // cache puts together. Against stores past the caches, the chain at T = 9723, E = 68,
  // K = 1345: N = 128 151 -> 90 us, N = 164 181 -> 140, N = 256 190 -> 150; where a slice
  // is a whole block (K = 1344 or 2048) the two are within 1 %, at T = 12000, E = 24,
  // K = 2000, N = 400 322 -> 340, and choosing by K keeps both in one loop and gains neither.
  int next_xp = CHAIN && prm.x_permuted != nullptr ? tl.ct : -1;
  auto store_xp = [&](int kt, const Slice& s) {
    if constexpr (CHAIN) {
      if (kt >> 1 != next_xp) return;
      if ((kt & 1) != 0) next_xp += col_tiles;
      const int k = kt * kBK + 4 * ac;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int r = PR * p + ar;
        if (r < rows) {
          float* out = prm.x_permuted + static_cast<std::size_t>(tl.row0 + r) * K + k;
          if (k + 4 <= K) {
            *reinterpret_cast<f4u*>(out) = s.a[p];
          } else {
            for (int q = 0; k + q < K; ++q) out[q] = s.a[p][q];
          }
        }
      }
    } else {
      (void)kt, (void)s;
    }
  };
  // a slice, split, into an LDS stage
  auto put = [&](__bf16* __restrict__ st, const Slice& s) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      if (!staged(p)) continue;
      uint32_t lo[kParts], up[kParts];
      split2(s.a[p][0], s.a[p][1], lo);
      split2(s.a[p][2], s.a[p][3], up);
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        *reinterpret_cast<uint2*>(st + i * S::kPlaneA + p * PR * kBK + a_put) = make_uint2(lo[i], up[i]);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      __bf16* out = st + kParts * S::kPlaneA + (j == 0 ? b_put : b_put1);
      uint32_t part[KP / 2][kParts];
#pragma unroll
      for (int q = 0; q < KP / 2; ++q) split2(s.b[2 * q][j], s.b[2 * q + 1][j], part[q]);
#pragma unroll
      for (int i = 0; i < kParts; ++i) {
        if constexpr (KP == 4) {
          *reinterpret_cast<uint2*>(out + i * kPlaneB) = make_uint2(part[0][i], part[1][i]);
        } else {
          *reinterpret_cast<uint32_t*>(out + i * kPlaneB) = part[0][i];
        }
      }
    }
  };

  const int wrow = L::row(wave);
  v16f acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.0F;
    }
  }
  {
    // operand chunk: k = 8 hi .. + 7 of a plane row
    const int aget = (wrow + li) * kBK + ((hi ^ swizzle(li)) << 3);
    const int brow = plane_row(L::col(wave) + li);  // (block j: 16 j rows further, whose swizzle is the same)
    const int bget = brow * kBK + ((hi ^ swizzle(brow)) << 3);
    struct Operands {
      b8 a[kParts][TM], b[kParts][TN];
    };
    auto fetch_a = [&](const __bf16* __restrict__ st, int part, b8 (&a)[TM]) {
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const b8*>(st + part * S::kPlaneA + aget + i * 32 * kBK);
    };
    auto fetch_b = [&](const __bf16* __restrict__ st, int part, b8 (&b)[TN]) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        b[j] = *reinterpret_cast<const b8*>(st + kParts * S::kPlaneA + part * kPlaneB + bget + j * 16 * kBK);
      }
    };
    auto fetch = [&](const __bf16* __restrict__ st, Operands& o) {
#pragma unroll
      for (int t = 0; t < kParts; ++t) {
        fetch_a(st, t, o.a[t]);
        fetch_b(st, t, o.b[t]);
      }
    };
    auto product = [&](const b8 (&a)[TM], const b8 (&b)[TN], v16f (&sum)[TM][TN]) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], sum[i][j], 0, 0, 0);
      }
    };
    // (one order of the sums in every shape)
    auto multiply = [&](const Operands& o) {
      product(o.a[0], o.b[0], acc);
      product(o.a[0], o.b[1], low);
      product(o.a[0], o.b[2], low);
      product(o.a[1], o.b[0], low);
      product(o.a[1], o.b[1], low);
      product(o.a[2], o.b[0], low);
    };
    // Slice kt is multiplied while slices kt + 2 .. kt + D are on their way; slice
    // kt + 1 has landed and goes to the other stage, and its registers take the
    // loads of slice kt + 1 + D. D = 2 where registers are left (slice i in set i & 1).
    constexpr int D = S::kBM == 128 ? 2 : 1;
    Slice even, odd;  // (D = 1: the first only)
    load_any(0, even);
    put(sh.stages, even);
    store_xp(0, even);
    if (nk > 1) load_any(1, D == 2 ? odd : even);
    if (D == 2 && nk > 2) load_any(2, even);
    __syncthreads();
    auto next = [&](int kt, Slice& s) {
      if (kt + 1 < nk) {
        put(sh.stages + (~kt & 1) * S::kStage, s);
        store_xp(kt + 1, s);
      }
      if (kt + 1 + D < nk) load_any(kt + 1 + D, s);
    };
    auto next_whole = [&](int kt, Slice& s) {
      put(sh.stages + (~kt & 1) * S::kStage, s);
      store_xp(kt + 1, s);
      load(kt + 1 + D, s);
    };
    if constexpr (W == 8) {
      // Two waves share a SIMD, one of each half of the workgroup. The halves
      // run a phase apart: while one fetches its operands of slice kt and stages
      // its part of slice kt + 1, the other has the matrix pipe to itself.
      // Slice kt + 1 is complete after the second half's phase, one barrier
      // before the first half reads it, and the stage it takes was last read
      // one barrier before the first half writes it.
      if (wave >= W / 2) __syncthreads();
      auto phases = [&](int kt, Slice& s, auto more) {
        Operands o;
        fetch(sh.stages + (kt & 1) * S::kStage, o);
        more(kt, s);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_s_setprio(1);
        multiply(o);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
      };
      int kt = 0;
      if constexpr (D == 2) {
#pragma unroll 1
        for (; kt + 5 < nk; kt += 2) {
          phases(kt, odd, next_whole);
          phases(kt + 1, even, next_whole);
        }
#pragma unroll 1
        for (; kt < nk; kt += 2) {
          phases(kt, odd, next);
          if (kt + 1 < nk) phases(kt + 1, even, next);
        }
      } else {
#pragma unroll 1
        for (; kt + 3 < nk; ++kt) phases(kt, even, next_whole);
#pragma unroll 1
        for (; kt < nk; ++kt) phases(kt, even, next);
      }
      if (wave < W / 2) __syncthreads();
    } else {
      static_assert(D == 2, "two sets of slice registers");
      auto slice = [&](int kt) {
        const __bf16* st = sh.stages + (kt & 1) * S::kStage;
        // (parts read as they are needed: all at once leave no registers for the
        // second slice on its way)
        b8 a[TM], b[kParts][TN];
        fetch_a(st, 0, a);
#pragma unroll
        for (int t = 0; t < kParts; ++t) fetch_b(st, t, b[t]);
        product(a, b[0], acc);
        product(a, b[1], low);
        product(a, b[2], low);
        fetch_a(st, 1, a);
        product(a, b[0], low);
        product(a, b[1], low);
        fetch_a(st, 2, a);
        product(a, b[0], low);
        __syncthreads();
      };
      int kt = 0;
#pragma unroll 1
      for (; kt + 5 < nk; kt += 2) {
        next_whole(kt, odd);
        __builtin_amdgcn_sched_barrier(0);  // (the scheduler would sink the loads to the slice's end)
        slice(kt);
        next_whole(kt + 1, even);
        __builtin_amdgcn_sched_barrier(0);
        slice(kt + 1);
      }
#pragma unroll 1
      for (; kt < nk; kt += 2) {
        next(kt, odd);
        slice(kt);
        if (kt + 1 < nk) {
          next(kt + 1, even);
          slice(kt + 1);
        }
      }
    }
  }

  // (the lane id passes an empty asm so that none of the epilogue's addresses
  // is built before the loop and kept live across it)
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const int eli = ln & 31;
  const int ehi = ln >> 5;
  // output rows of accumulator register r: 32 i + 8 (r / 4) + 4 hi + r % 4 of the wave's
  const int ec = L::col(wave) + eli;  // tile column; block j: 32 j further
  bool any = false;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rl = wrow + 32 * i + 8 * (r >> 2) + 4 * ehi + (r & 3);
        acc[i][j][r] += low[i][j][r];
        any = any || (rl < rows && tl.n0 + ec + 32 * j < N && untrusted(acc[i][j][r]));
      }
    }
  }
  const bool redo = __syncthreads_or(any ? 1 : 0) != 0;
  // the combined row of tile row rl (chain) and an output's way to memory
  auto combined_row = [&](int rl) -> float* {
    if constexpr (CHAIN) {
      if (prm.y_out != nullptr) return prm.y_out + static_cast<std::size_t>(sh.src[rl]) * N + tl.n0;
    }
    return nullptr;
  };
  auto emit = [&](float v, float* y, float* comb, float w) {
    if (comb != nullptr) {
      __builtin_nontemporal_store(v, y);  // y_permuted is not read again by the chain
      // Both routes of a token add into the zeroed output: fl(0 + a) + b
      // is the same in either order, so the combine is deterministic
      // and equals the rank-order unpermute.
      unsafeAtomicAdd(comb, __fmul_rn(w, v));
    } else {
      *y = v;
    }
  };
  float* const ytile = prm.Y + static_cast<std::size_t>(tl.row0) * N + tl.n0;
  uint32_t* mask = reinterpret_cast<uint32_t*>(sh.stages) + S::kMaskAt;  // [row][column / 32]
  uint32_t again[TM] = {};  // bit 16 j + r: output (i, j, r) is one of those
  if (redo) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rl = wrow + 32 * i + 8 * (r >> 2) + 4 * ehi + (r & 3);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const bool a = rl < rows && tl.n0 + ec + 32 * j < N && untrusted(acc[i][j][r]);
          const uint64_t m = __ballot(a);
          if (eli == 0) mask[4 * rl + (L::col(wave) >> 5) + j] = static_cast<uint32_t>(ehi == 0 ? m : m >> 32);
          again[i] |= a ? 1U << (16 * j + r) : 0U;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rl = wrow + 32 * i + 8 * (r >> 2) + 4 * ehi + (r & 3);
      if (rl >= rows) continue;
      float* yrow = ytile + static_cast<std::size_t>(rl) * N + ec;
      float* comb = combined_row(rl);
      const float w = comb != nullptr ? sh.w[rl] : 0.0F;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (tl.n0 + ec + 32 * j >= N || (again[i] >> (16 * j + r) & 1) != 0) continue;
        emit(acc[i][j][r], yrow + 32 * j, comb != nullptr ? comb + ec + 32 * j : nullptr, w);
      }
    }
  }
  if (!redo) return;

  // ---- the masked outputs on the FP32 instructions (v_mfma_f32_16x16x4_f32) ----
  // Slices of both operands as they are, k order as in every FP32 GEMM here
  // (chunks of 16 k ascending, MFMA step s sums k = 16 c + 4 g + s over g): the bits
  // of the FP32 kernels. Wave w takes kBN / W columns and those of the tile's
  // 16-row blocks that have a masked output there.
  constexpr int CW = kBN / W;
  constexpr int NJ = CW / 16;
  constexpr int NB = L::kRows / 16;
  const int g = ln >> 4 & 3;
  const int fl = ln & 15;
  __syncthreads();  // masks
  uint32_t blocks = 0;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const uint32_t m = mask[4 * (16 * i + fl) + (CW * wave >> 5)] >> (CW * wave & 31);
    if (__ballot((CW == 32 ? m : m & 0xFFFFU) != 0) != 0) blocks |= 1U << i;
  }
  v4f sum[NB][NJ];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) sum[i][j] = v4f{0.0F, 0.0F, 0.0F, 0.0F};
  }
  // quad q of row r sits at quad q ^ (r & 3) (B: q ^ (r / 2 & 3))
  Slice s;
  load_any(0, s);
#pragma unroll 1
  for (int kt = 0; kt < nk; ++kt) {
    float* As = reinterpret_cast<float*>(sh.stages) + (kt & 1) * S::kStage32;
    float* Bs = As + S::kBM * kBK;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int r = PR * p + ar;
      if (staged(p)) *reinterpret_cast<v4f*>(As + r * kBK + 4 * (ac ^ (r & 3))) = v4f{s.a[p][0], s.a[p][1], s.a[p][2], s.a[p][3]};
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float* out = Bs + (2 * pair + j) * kBK + 4 * ((b_k >> 2) ^ (pair & 3)) + (b_k & 3);
#pragma unroll
      for (int q = 0; q < KP; ++q) out[q] = s.b[q][j];
    }
    if (kt + 1 < nk) load_any(kt + 1, s);
    __syncthreads();  // (the other stage was last read before the previous slice's barrier)
    v4f b[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = CW * wave + 16 * j + fl;
      b[j] = *reinterpret_cast<const v4f*>(Bs + col * kBK + 4 * (g ^ (col >> 1 & 3)));
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if ((blocks >> i & 1) == 0) continue;
      const v4f a = *reinterpret_cast<const v4f*>(As + (16 * i + fl) * kBK + 4 * (g ^ (fl & 3)));
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[j][q], sum[i][j], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if ((blocks >> i & 1) == 0) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rl = 16 * i + 4 * g + r;
      float* comb = rl < rows ? combined_row(rl) : nullptr;
      const float w = comb != nullptr ? sh.w[rl] : 0.0F;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int c = CW * wave + 16 * j + fl;
        if ((mask[4 * rl + (c >> 5)] >> (c & 31) & 1) == 0) continue;
        emit(sum[i][j][r], ytile + static_cast<std::size_t>(rl) * N + c, comb != nullptr ? comb + c : nullptr, w);
      }
    }
  }
}

template <int W, int BM, bool CHAIN>
__global__ __launch_bounds__(64 * W, 2) void rr_split_gemm_kernel(GemmParams prm) {
  using S = Shape<W, BM>;
  constexpr int kBM = BM;
  extern __shared__ __align__(16) __bf16 smem[];
  Lds sh;
  sh.stages = smem;
  sh.src = reinterpret_cast<int32_t*>(smem + 2 * S::kStage);
  sh.w = reinterpret_cast<float*>(sh.src + kBM);
  int32_t* s_off = reinterpret_cast<int32_t*>(sh.w + kBM);  // [E + 1]
  int32_t* s_pre = s_off + prm.experts + 1;                 // [E + 1] full row tiles before expert e
  int32_t* s_pre2 = s_pre + prm.experts + 1;                // [E + 1] short row tiles before expert e
  const int tid = static_cast<int>(threadIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int experts = prm.experts;

  for (int e = tid; e <= experts; e += S::kThreads) s_off[e] = prm.offsets[e];
  __syncthreads();
  if (wave == 0) build_tile_prefix<kBM, true>(s_off, s_pre, s_pre2, experts, rr::dev::lane_id());
  __syncthreads();
  const int full_rows = s_pre[experts];
  const int short_rows = s_pre2[experts];
  const int col_tiles = (prm.N + kBN - 1) / kBN;
  const long total_full = static_cast<long>(full_rows) * col_tiles;
  const long total = total_full + static_cast<long>(short_rows) * col_tiles;
  const int grid = static_cast<int>(gridDim.x);
  const int worker = tile_worker(static_cast<int>(blockIdx.x), grid);

#pragma unroll 1
  for (long dealt = 0; dealt < total; dealt += grid) {
    // The last, partial round goes to the workgroups in dispatch order, over all
    // XCDs and one a CU first, instead of filling the first XCDs (staged T = 3001,
    // E = 9, K = 1023, N = 1535 153.6 -> 145.4 us; chain T = 16384, E = 64, K = N = 512
    // 170 -> 161).
    const int mine = total - dealt >= grid ? worker : static_cast<int>(blockIdx.x);
    const long t = dealt + mine;
    if (t >= total) break;
    const bool is_short = t >= total_full;
    int rt, ct;
    decode_tile(static_cast<int>(is_short ? t - total_full : t), is_short ? short_rows : full_rows,
                col_tiles, &rt, &ct);
    const int e = __builtin_amdgcn_readfirstlane(tile_expert(is_short ? s_pre2 : s_pre, experts, rt));
    const int first = __builtin_amdgcn_readfirstlane(s_off[e]);
    const int end = __builtin_amdgcn_readfirstlane(s_off[e + 1]);
    Tile tl;
    tl.B = prm.W + static_cast<std::size_t>(e) * prm.K * prm.N;
    tl.row0 = first + (is_short ? (end - first) / kBM : rt - __builtin_amdgcn_readfirstlane(s_pre[e])) * kBM;
    tl.rows = end - tl.row0 < kBM ? end - tl.row0 : kBM;
    tl.n0 = ct * kBN;
    tl.ct = ct;

    __syncthreads();  // the previous tile's epilogue is done with the LDS tables
    if constexpr (CHAIN) {
      if (tid < kBM) {
        int32_t token = -1;
        float w = 0.0F;
        if (tid < tl.rows) {
          const int32_t route = prm.sorted_route[tl.row0 + tid];
          token = route / prm.top_k;  // route = top_k * token + rank
          if (prm.y_out != nullptr) w = prm.route_weights[route];
        }
        sh.src[tid] = token;
        sh.w[tid] = w;
      }
      __syncthreads();
    }
    if constexpr (BM == 32 * W) {
      if (tl.rows > BM / 4 * 3) {
        run_tile<S, Layout<W, 2, true>, CHAIN>(prm, tl, sh, col_tiles, wave);
        continue;
      }
      if (tl.rows > BM / 2) {
        run_tile<S, Layout<W, 3, false>, CHAIN>(prm, tl, sh, col_tiles, wave);
        continue;
      }
    }
    if (tl.rows > 8 * W) {
      run_tile<S, Layout<W, 2, false>, CHAIN>(prm, tl, sh, col_tiles, wave);
    } else {
      run_tile<S, Layout<W, 1, false>, CHAIN>(prm, tl, sh, col_tiles, wave);
    }
  }
}

template <int W, int BM, bool CHAIN>
hipError_t launch(const GemmParams& prm, long rows_per_expert, int cus, hipStream_t stream) {
  using S = Shape<W, BM>;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(rr_split_gemm_kernel<W, BM, CHAIN>), hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
  if (attr != hipSuccess) return attr;
  const long bound = static_cast<long>(prm.experts) * ((rows_per_expert + BM - 1) / BM) *
                     ((static_cast<long>(prm.N) + kBN - 1) / kBN);
  const long cap = static_cast<long>(8 / W) * cus;
  long grid = bound < cap ? bound : cap;
  if (grid >= kXcds) grid = grid / kXcds * kXcds;
  if (grid < 1) grid = 1;
  const std::size_t lds = 2 * S::kStage * sizeof(__bf16) + 2 * S::kBM * sizeof(int32_t) +
                          3 * static_cast<std::size_t>(prm.experts + 1) * sizeof(int32_t);
  rr_split_gemm_kernel<W, BM, CHAIN><<<dim3(static_cast<unsigned>(grid)), S::kThreads, lds, stream>>>(prm);
  return hipGetLastError();
}

long ceil_div(long a, long b) { return (a + b - 1) / b; }

// Tiles of the rows of the whole problem plus a part tile per expert.
long tiles(long rows, int experts, int bm, int n, int bn) { return (ceil_div(rows, bm) + experts) * ceil_div(n, bn); }

}  // namespace

// Where the FP32 kernels stay (grouped GEMM alone, experts' rows drawn at random,
// FP32 kernels / this one):
//  - K < 128 or N <= 64, where neither side is bound by the matrix instructions, and
//    K and N both below 256;
//  - problems of so few tiles that their smaller tiles spread over more CUs: with
//    K >= 512 below 1.1 64 x 64 tiles a CU (E = 32, K = 1024, N = 256, 2048 rows, 256 tiles
//    47 / 49 us; E = 8, K = 2048, N = 1536, 192 rows, 264 tiles 82 / 66), or 1.25 where the
//    experts have less than eight rows each (E = 8, K = 512, N = 2048, 32 rows 16.4 /
//    21.8); with shorter K, where a tile's first loads and last stores weigh more,
//    below 2.5 (E = 16, K = 256, N = 1024, 1600 rows, 656 tiles 17.5 / 19.4; E = 16,
//    K = 320, N = 768, 768 rows, 336 tiles 20.0 / 16.4, but E = 8, K = 256, N = 1536, 1200
//    rows, 648 tiles 28 / 20), and 3.25 with K < 192 (E = 64, K = 128, N = 768, 640 rows, 888
//    tiles 17.0 / 19.0);
//  - few rows an expert where the FP32 side has its 128 x 128 tiles (two a CU): both
//    are bound by the weights, which those load straight into LDS. E = 128, K = 128,
//    N = 2048: 24 rows each 43 / 54 us, 48 rows 52 / 57; E = 128, K = 1024, N = 2048: 16 rows
//    each 192 / 225; E = 128, K = 512, N = 1536: 16 rows 82 / 96, 24 rows 98 / 103, and E = 64,
//    K = 4096, N = 2048 24 rows 442 / 458, but most shapes of 24 rows 1.0 to 1.4 times
//    faster here.
// The lines are those of the whole range. Where N leaves a fifth or more of its 128-column
// tiles empty, problems just past them are up to 15 % slower here (E = 24, K = 512, N = 400,
// 3600 rows 26.5 / 30.3; E = 128, K = 512, N = 72, 8192 rows 25.5 / 29.4; 78 of 1344
// combinations by more than 4 %), but of the same tile counts others are up to 1.9 times
// faster (E = 8, K = 2048, N = 130, 12000 rows), and over 1344 combinations no line by
// the padded columns came nearer to the faster side of each (2.0 % off on average).
bool split_gemm_ok(int k, int n, int experts, long rows, int cus) {
  if (k < 128 || n <= 64 || (k < 256 && n < 256)) return false;
  const long few = k < 192 ? 40 : 20;  // rows an expert
  if (rows < few * experts && tiles(rows, experts, 128, n, 128) >= 2L * cus) return false;
  const long t = tiles(rows, experts, 64, n, 64);
  if (k >= 512) return 20 * t >= (rows < 8L * experts ? 25L : 22L) * cus;
  return k < 192 ? 4 * t > 13L * cus : 2 * t >= 5L * cus;
}

// 32-bit byte offsets: a tile's A rows (chain: all of X) and an expert's weights.
bool split_gemm_fits(const GemmParams& prm) {
  const long limit = 1L << 30;
  const long a_rows = prm.sorted_route != nullptr ? prm.dense_rows : 256;
  return prm.K > 0 && prm.N >= 2 && a_rows * prm.K < limit && static_cast<long>(prm.K + kBK) * prm.N < limit;
}

// Workgroup shape:
//  - eight waves on 128-row tiles where there are no more tiles than CUs: more waves
//    for the one a CU gets (E = 16, K = 2048, N = 300 with 8192 rows: 95 us against 132 with
//    four waves; chain T = 2048, E = 64, K = 1024, N = 512 75 / 83, but T = 4096, E = 16,
//    K = 2048, N = 512, just past one tile a CU, 200 / 159). Tiles: full ones, and half
//    of the experts with a part tile, but every expert that can have rows has one;
//  - eight waves on 256-row tiles where there are many of them and the experts
//    have the rows (E = 8, K = 4096, N = 8192 with 16384 rows 5.09 ms against
//    6.11; E = 64, K = 1024, N = 512, 256 rows an expert: 90 / 100 us, but E = 64,
//    K = 512, N = 768, 256 rows an expert: 90 / 87). Not for the chain: nothing runs
//    under a tile's combine with one workgroup a CU (T = 8192, E = 64, K = 1024, N = 768
//    275 / 237 us, T = 16384, E = 128, K = 2048, N = 768 836 / 835);
//  - else four waves on 128-row tiles, two workgroups a CU.
hipError_t split_grouped(const GemmParams& prm, long rows_per_expert, long rows, int cus, SplitShape shape,
                         hipStream_t stream) {
  const bool chain = prm.sorted_route != nullptr;
  if (shape == SplitShape::kBySize) {
    const long halves = std::max(2 * ceil_div(rows, 128) + prm.experts, 2 * std::min<long>(rows, prm.experts));
    if (halves * ceil_div(prm.N, kBN) <= 2L * cus) {
      shape = SplitShape::kEightWaves;
    } else if (prm.K >= 512 && tiles(rows, prm.experts, 256, prm.N, kBN) >= 2L * cus &&
               rows * prm.K >= (1L << 18) * prm.experts) {
      shape = SplitShape::kRows256;
    }
  }
  if (shape == SplitShape::kEightWaves) {
    return chain ? launch<8, 128, true>(prm, rows_per_expert, cus, stream)
                 : launch<8, 128, false>(prm, rows_per_expert, cus, stream);
  }
  if (chain) return launch<4, 128, true>(prm, rows_per_expert, cus, stream);
  if (shape == SplitShape::kRows256) return launch<8, 256, false>(prm, rows_per_expert, cus, stream);
  return launch<4, 128, false>(prm, rows_per_expert, cus, stream);
}

}  // namespace rr::kern
