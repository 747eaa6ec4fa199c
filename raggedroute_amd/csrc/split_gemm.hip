// Grouped FP32 GEMM on the FP16 matrix cores (v_mfma_f32_32x32x16_f16).
//
// The FP32 matrix instructions run at 157 TFLOP/s, the FP16 ones at 2.5 PFLOP/s
// with FP32 accumulation. Every operand x is scaled by a power of two of its
// own row (A) or column (B), xs = x * s, and split into two FP16 numbers
//     h = fp16(xs),   l = fp16(xs - h),   l stored times 2^11,
// both rounded to nearest; xs - h is exact in FP32 and at most 2^-11 of xs, so
// h + l carries x to within 2^-23 of itself (half of all values exactly). A
// product is
//     xs * ys = hx hy + (lx hy + hx ly) + lx ly;
// the first three terms are computed (three MFMAs), the last is at most 2^-22 of
// the product (2^-25 in the mean) and left out. hx hy is summed in one FP32
// accumulator and the two small terms in another, which is added once, times
// 2^-11, at the end: the large sum is rounded once per 16 k instead of once per
// 4 k as on the FP32 instructions. Against 64-bit sums dense operands' results
// are closer than the FP32 instructions' at every K (2-norm error over N(0,1) operands, this / FP32 MFMA:
// K = 64 0.98 / 1.43e-7, K = 128 1.10 / 2.03e-7, K = 256 1.31 / 2.87e-7, K = 1024
// 2.2 / 5.8e-7, K = 4096 4.1 / 11.4e-7; non-negative operands K = 128 0.64 / 1.59e-7;
// both operands half zero K = 128 1.06 / 1.04e-7, K = 192 1.16 / 1.26e-7). Sums of few
// products have the split's own error instead: K = 1024, rows of 64 nonzero values
// 1.46 / 1.44e-7, of 16 1.03 / 0.74e-7, of one 0.77 / 0.25e-7.
//
// Range. The scale puts the largest of a row's (column's) first slice of 32 k
// near 2^6, so later values may be 2^9 times larger before fp16(xs)
// overflows. (Where that slice is all zero, 1 is taken for the largest; reading on
// to the first value made a tile with one all-zero row, a padding token, scan all
// of K first: E = 8, 16384 rows, K = 4096, N = 14336 11.7 ms, now 6.3 as without such
// rows; E = 64, 4096 rows, K = 1024, N = 512 72 -> 36 us.) l, stored times 2^11,
// keeps its 11 bits down to |xs| = 2^-14 (2^-20 of the sampled maximum); below, the
// split's error stays at 2^-36, so that values much smaller than the sample lose
// their bits: with one feature 2^p times the rest and its weights zero, K = 320, the
// 2-norm error was 1.8e-6 at p = 24, 1.1e-4 at p = 30, 0.1 at p = 40 (FP32
// instructions 3.2e-7). Nothing of that kind is computed this way. A row or column is marked when
//  - its sample is below 2^-100, or 2^41 and more (or not finite);
//  - four of its values in slice 0 are nonzero and scale to less than 2^-14;
//  - of four consecutive k (4 i .. 4 i + 3) past slice 0 the largest does.
// So of any four k of an unmarked row past slice 0 the split's error is at most
// 2^-22 of the largest, and values whose xs is below 2^-14 are few among larger
// ones. (A scaled value under 2^-149 counts as zero: |x| < 2^-115 in a row whose
// sample is 2^40.) An operand past the FP16 range makes every output it meets
// non-finite. Outputs of marked rows and columns and non-finite ones are computed
// on the FP32 instructions instead, with the bits of the FP32 kernels. Which those
// are is a matter of each output's own row and column, so that no row's bits
// depend on the rows it shares a tile with, or on the tile's height. A tile
// with such outputs goes through its slices once more, with FP32 products only
// for the 16-row blocks that hold one: E = 8, 16384 rows, K = 4096, N = 14336, one
// infinite row in a thousand 10.4 ms (17.4 when whole tiles were computed again, as
// 32 x 32 products without a slice on its way; FP32 kernel 13.8); E = 128, 32768
// rows, K = 2048, N = 768 569 us (979; 760). Where every row has such a value (a
// feature 2^14 times the others) the second pass is a whole FP32 product and comes
// on top: 23.0 ms and 1.36 ms. N(0,1) rows are as good as
// never marked (four neighbours below 2^-19); of rows with every other value zero at
// random, four in 10^4 at K = 4096. The marks take 24 of 132 vector instructions of a slice of
// the 256-row loop: T = 8192, E = 8, K = 4096, N = 14336 call 6.80 -> 7.21 ms, T = 3001,
// E = 9, K = 1023, N = 1535 150 -> 156 us, chain T = 16384, E = 128, K = 2048, N = 768
// 607 -> 626 us, T = 2048, E = 64, K = 1024, N = 512 70.2 -> 72.1 us. (Pairs of k, and
// groups over two slices or two lanes, were slower: 7.1 - 8.0 ms in the first.)
//
// Work split: output tiles of 128 columns and 128 or 256 rows on four or eight
// waves (split_grouped picks), tiles dealt as in gemm.hip. A slice of 32 k of
// both operands is loaded into registers one slice ahead (16-byte A quads, 8-byte
// B pairs; rows may start at any 4-byte boundary), split there, and written to
// LDS as FP16 planes in MFMA operand order (k contiguous per row of A and per
// column of B), two stages; the split costs four full-rate instructions per
// element. Four waves: two workgroups share a CU and
// one's MFMAs run under the other's staging. Eight waves: the two halves of the
// workgroup run a phase apart, so that one has the matrix pipe while the other
// stages. Tiles with few rows take layouts of fewer 32-row blocks.
// Loads are buffer loads (scalar base, 32-bit lane offset): with 64-bit lane
// addresses the eight-wave loop spilled (256 registers).
//
// Large problems are bound by the staging phase (operand reads, split, marks and
// plane writes of one half, longer than the other half's matrix instructions) at a
// clock that the power limit holds down: E = 8, K = 4096, N = 14336, 16384 rows (1.92
// TFLOP), matrix pipes busy 42 % of the cycles at 1.77 of 2.4 GHz. FP32
// instructions 13.8 ms, four waves 7.1, eight waves 6.3 ms (304 TFLOP/s of FP32
// products, 912 of FP16 ones; a library FP16 product of random 8192 x 8192 matrices
// reaches 1300 on this card), 5.3 ms with operands of ones, which draw less
// power. Elsewhere by each tile's serial parts and the combine: T = 16384, E = 128,
// K = 2048, N = 768 chain, expert GEMM 927 / 557 us, matrix pipes 28 % busy at 2.0 GHz;
// T = 2048, E = 64, K = 1024, N = 512 13 %.
#include <hip/hip_runtime.h>

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
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int kBN = 128, kBK = 32;
constexpr int kPlaneB = kBN * kBK;          // halfs of one plane of B (8 KiB)
constexpr float kLowScale = 2048.0F;        // l is stored times 2^11
constexpr float kLeast = 0x1p-14F;          // scaled values from here on keep all bits of l
constexpr int kFewSmall = 4;                // too small values of slice 0 that send a row or column to FP32
constexpr int kMarked = 1 << 16;            // scale exponent of a row or column that is not computed in FP16
constexpr int kBufferFlags = 0x00027000;    // raw 32-bit buffer

// BM x 128 output tiles on W waves (four: two workgroups per CU; eight: one).
template <int W, int BM>
struct Shape {
  static constexpr int kWaves = W;
  static constexpr int kThreads = 64 * W;
  static constexpr int kBM = BM;
  static constexpr int kPassRows = 8 * W;                        // rows of A staged per pass
  static constexpr int kKPer = kBK / W;                          // k rows of B a thread stages
  static constexpr int kPlaneA = kBM * kBK;                      // halfs
  static constexpr int kStage = 2 * (kPlaneA + kPlaneB);         // A high, A low, B high, B low
  static constexpr int kStage32 = (kBM + kBN) * kBK;             // floats
  static_assert(2 * kStage32 * sizeof(float) <= 2 * kStage * sizeof(_Float16), "two FP32 slices fit the stages");
  static_assert(kBM * (kBN / 32) * sizeof(uint32_t) <= W * 64 * sizeof(uint2), "the masks fit the column samples");
};

// Wave tiles of TM x TN blocks of 32 x 32. GRID: W / 2 x 2 waves of TN = 2 column
// blocks; else W / 4 x 4 waves of one.
template <int W, int TM_, bool GRID>
struct Layout {
  static constexpr int TM = TM_;
  static constexpr int TN = GRID ? 2 : 1;
  static constexpr int kRows = TM_ * 32 * (GRID ? W / 2 : W / 4);
  static constexpr int kPasses = kRows / (8 * W);  // staging passes that hold the tile's rows
  static_assert(kPasses * (8 * W) == kRows, "whole passes");
  __device__ static int row(int wave) { return (GRID ? wave >> 1 : wave >> 2) * 32 * TM_; }
  // first tile column (plane row of B)
  __device__ static int col(int wave) { return GRID ? 64 * (wave & 1) : 32 * (wave & 3); }
};

// 16-byte chunk c (8 halfs) of plane row r sits at chunk c ^ ((r >> 2) & 3): the
// 16 rows read together land in 16 distinct 16-byte bank groups. (B's writes do
// not: 16 lanes write every second row, half of the groups; 30 % of the LDS's index
// cycles at E = 8, K = 4096, N = 14336 are conflicts.)
__device__ __forceinline__ int plane_swizzle(int r) { return (r >> 2) & 3; }

// x * s = h + l (see the file comment): eight full-rate instructions for two
// values. (Four v_fma_mixlo / mixhi_f16 would do, but they issue at half rate:
// 9.7 against 4.7 cycles.)
// x0 and x1 are left scaled.
__device__ __forceinline__ void split2(float& x0, float& x1, float s, h2& h, h2& l) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  const float s0 = x0 * s, s1 = x1 * s;
  h = __builtin_convertvector(f2{s0, s1}, h2);
  asm("" : "+v"(h));  // both halves in their register: the next two read them there
  l = __builtin_convertvector(f2{__builtin_fmaf(x0, s, -static_cast<float>(h[0])) * kLowScale,
                                 __builtin_fmaf(x1, s, -static_cast<float>(h[1])) * kLowScale}, h2);
  x0 = s0;
  x1 = s1;
}

// The largest of four magnitudes (without the canonicalizing copies of fmaxf).
__device__ __forceinline__ float most_of(float a, float b, float c, float d) {
  float m;
  asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(m) : "v"(a), "v"(b), "v"(c));
  asm("v_max_f32 %0, %1, |%2|" : "=v"(m) : "v"(m), "v"(d));
  return m;
}

__device__ __forceinline__ uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7FFFFFFFU; }
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }

// The scale of a row or column whose sampled maximum has these bits: s = 2^t
// with t = 6 - floor(log2(max)). An all-zero sample is taken for one of largest
// value 1: an all-zero row or column is exact under any scale, and later values
// between 2^-20 and 2^9 are carried.
struct Scale {
  float s;
  int t;
  bool bad;  // not computed in FP16: below 2^-100, or 2^41 and more (or not finite)
};
__device__ __forceinline__ Scale scale_of(uint32_t bits) {
  Scale sc;
  int e = static_cast<int>(bits >> 23);
  sc.bad = bits != 0 && (e > 167 || e < 27);
  e = bits == 0 ? 127 : (e < 27 ? 27 : e);
  sc.t = 133 - e;
  sc.s = __uint_as_float(static_cast<uint32_t>(260 - e) << 23);
  return sc;
}

// Whether a scaled magnitude (its bits) is too small for the split: nonzero and below kLeast.
__device__ __forceinline__ bool too_small(uint32_t m) { return m - 1U < __float_as_uint(kLeast) - 1U; }

// What a tile needs from the kernel (all workgroup-uniform).
struct Tile {
  const float* B;  // the expert's weights
  int row0, rows;  // first segment row, rows in the tile (1..128)
  int n0, ct;      // first column, column tile
};
struct Lds {
  _Float16* stages;  // [2][kStage]
  int32_t* ta;       // [kBM] scale exponents of the rows (kMarked: FP32)
  int32_t* tb;       // [128] ... of the plane rows of B
  uint2* cmax;       // [W][64] column samples; after the slices [kBM][4] masks of the outputs to recompute
  int32_t* few;      // [128] values of slice 0 too small for their column's scale
  int32_t* src;      // [kBM] chain: token row of X per tile row (-1: none)
  float* w;          // [kBM] chain: route weight per tile row
};

// One output tile for one wave layout (L::kPasses 32-row passes hold its rows).
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
  const int ar = tid >> 3;
  const int ac = tid & 7;
  const int pair = lane;
  const int a_put = ar * kBK + (((ac >> 1) ^ plane_swizzle(ar)) << 3) + ((ac & 1) << 2);
  const int b_k = KP * wave;
  const int b_put = 2 * pair * kBK + (((b_k >> 3) ^ plane_swizzle(2 * pair)) << 3) + (b_k & 7);

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

  f4u ra[P];
  f2u rb[KP];
  auto load = [&](int kt) {  // whole slices
#pragma unroll
    for (int p = 0; p < P; ++p) {
      ra[p] = __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(a_base, a_lane[p], 4 * kBK * kt, 0));
    }
    // (a pair that crosses N reads the next k row's first float)
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      rb[j] = __builtin_bit_cast(f2u, __builtin_amdgcn_raw_buffer_load_b64(b_base, b_lane, b_row(kt, j), 0));
    }
  };
  auto load_any = [&](int kt) {
    if (kt != guarded) {
      load(kt);
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
        ra[p][q] = v;
      }
    }
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      float v0 = 0.0F, v1 = 0.0F;
      if (kt * kBK + b_k + j < K) {
        v0 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b_base, b_lane, b_row(kt, j), 0));
        if (nl + 1 < N) v1 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b_base, b_lane + 4, b_row(kt, j), 0));
      }
      rb[j] = f2u{v0, v1};
    }
  };

  // ---- scales, from the first slice ----
  load_any(0);
  if (tid < kBN) sh.few[tid] = 0;
  uint32_t ma[P];
  uint32_t mb0 = 0, mb1 = 0;
#pragma unroll
  for (int p = 0; p < P; ++p) {
    uint32_t m = umax(umax(abs_bits(ra[p][0]), abs_bits(ra[p][1])), umax(abs_bits(ra[p][2]), abs_bits(ra[p][3])));
    // over the row's eight lanes: quad neighbours, then the half row's mirror
    m = umax(m, rr::dev::dpp_move<0xB1>(m));
    m = umax(m, rr::dev::dpp_move<0x4E>(m));
    ma[p] = umax(m, rr::dev::dpp_move<0x141>(m));
  }
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    mb0 = umax(mb0, abs_bits(rb[j][0]));
    mb1 = umax(mb1, abs_bits(rb[j][1]));
  }
  sh.cmax[64 * wave + pair] = make_uint2(mb0, mb1);
  __syncthreads();
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const uint2 m = sh.cmax[64 * w + pair];
    mb0 = umax(mb0, m.x);
    mb1 = umax(mb1, m.y);
  }
  float sa[P], sb[2];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const Scale sc = scale_of(ma[p]);
    sa[p] = sc.s;
    uint32_t few = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) few += too_small(abs_bits(ra[p][q] * sc.s)) ? 1U : 0U;
    few += rr::dev::dpp_move<0xB1>(few);
    few += rr::dev::dpp_move<0x4E>(few);
    few += rr::dev::dpp_move<0x141>(few);
    if (ac == 0) sh.ta[PR * p + ar] = sc.bad || few >= kFewSmall ? kMarked : sc.t;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const Scale sc = scale_of(j == 0 ? mb0 : mb1);
    sb[j] = sc.s;
    if (wave == 0) sh.tb[2 * pair + j] = sc.bad ? kMarked : sc.t;
    int32_t few = 0;
#pragma unroll
    for (int q = 0; q < KP; ++q) few += too_small(abs_bits(rb[q][j] * sc.s)) ? 1 : 0;
    if (few != 0) atomicAdd(sh.few + 2 * pair + j, few);
  }

  // Gathered rows go to x_permuted spread over the column tiles: tile ct
  // writes the k slices kt with kt % col_tiles == ct.
  int next_xp = CHAIN && prm.x_permuted != nullptr ? tl.ct : -1;
  auto store_xp = [&](int kt) {
    if constexpr (CHAIN) {
      if (kt != next_xp) return;
      next_xp += col_tiles;
      const int k = kt * kBK + 4 * ac;
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int r = PR * p + ar;
        if (r < rows) {
          float* out = prm.x_permuted + static_cast<std::size_t>(tl.row0 + r) * K + k;
          if (k + 4 <= K) {
            __builtin_nontemporal_store(ra[p], reinterpret_cast<f4u*>(out));
          } else {
            for (int q = 0; k + q < K; ++q) out[q] = ra[p][q];
          }
        }
      }
    } else {
      (void)kt;
    }
  };
  // The slice in registers, split, into an LDS stage; slices past the first also
  // note the rows and columns with four k too small for the scale.
  uint64_t small_a[P] = {}, small_b[2] = {};  // lane masks
  auto put = [&](_Float16* __restrict__ st, int kt) {
    float most_a[P], most_b[2][KP / 4];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      h2 h0, l0, h1, l1;
      float x0 = ra[p][0], x1 = ra[p][1], x2 = ra[p][2], x3 = ra[p][3];
      split2(x0, x1, sa[p], h0, l0);
      split2(x2, x3, sa[p], h1, l1);
      most_a[p] = most_of(x0, x1, x2, x3);
      *reinterpret_cast<h4*>(st + p * PR * kBK + a_put) = h4{h0[0], h0[1], h1[0], h1[1]};
      *reinterpret_cast<h4*>(st + S::kPlaneA + p * PR * kBK + a_put) = h4{l0[0], l0[1], l1[0], l1[1]};
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      typedef _Float16 hk __attribute__((ext_vector_type(KP)));
      hk h, l;
#pragma unroll
      for (int q = 0; q < KP / 4; ++q) {
        h2 h0, l0, h1, l1;
        float x0 = rb[4 * q][j], x1 = rb[4 * q + 1][j], x2 = rb[4 * q + 2][j], x3 = rb[4 * q + 3][j];
        split2(x0, x1, sb[j], h0, l0);
        split2(x2, x3, sb[j], h1, l1);
        most_b[j][q] = most_of(x0, x1, x2, x3);
        h[4 * q] = h0[0], h[4 * q + 1] = h0[1], h[4 * q + 2] = h1[0], h[4 * q + 3] = h1[1];
        l[4 * q] = l0[0], l[4 * q + 1] = l0[1], l[4 * q + 2] = l1[0], l[4 * q + 3] = l1[1];
      }
      *reinterpret_cast<hk*>(st + 2 * S::kPlaneA + b_put + j * kBK) = h;
      *reinterpret_cast<hk*>(st + 2 * S::kPlaneA + kPlaneB + b_put + j * kBK) = l;
    }
    if (kt > 0) {
#pragma unroll
      for (int p = 0; p < P; ++p) {
        small_a[p] |= __ballot(too_small(__float_as_uint(most_a[p])));
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int q = 0; q < KP / 4; ++q) small_b[j] |= __ballot(too_small(__float_as_uint(most_b[j][q])));
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
    const int prow = L::col(wave) + li;
    // operand chunk of k step ks: k = 16 ks + 8 hi .. + 7
    const int aget = (wrow + li) * kBK, bget = prow * kBK;
    const int achunk[2] = {(hi ^ plane_swizzle(li)) << 3, ((2 + hi) ^ plane_swizzle(li)) << 3};
    const int bchunk[2] = {(hi ^ plane_swizzle(prow)) << 3, ((2 + hi) ^ plane_swizzle(prow)) << 3};
    struct Operands {
      h8 ah[TM], al[TM], bh[TN], bl[TN];
    };
    auto fetch = [&](const _Float16* __restrict__ st, int ks, Operands& o) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        o.ah[i] = *reinterpret_cast<const h8*>(st + aget + achunk[ks] + i * 32 * kBK);
        o.al[i] = *reinterpret_cast<const h8*>(st + S::kPlaneA + aget + achunk[ks] + i * 32 * kBK);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        o.bh[j] = *reinterpret_cast<const h8*>(st + 2 * S::kPlaneA + bget + bchunk[ks] + j * 32 * kBK);
        o.bl[j] = *reinterpret_cast<const h8*>(st + 2 * S::kPlaneA + kPlaneB + bget + bchunk[ks] + j * 32 * kBK);
      }
    };
    auto multiply = [&](const Operands& o) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ah[i], o.bh[j], acc[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.al[i], o.bh[j], low[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ah[i], o.bl[j], low[i][j], 0, 0, 0);
      }
    };
    put(sh.stages, 0);
    store_xp(0);
    if (nk > 1) load_any(1);
    __syncthreads();
    // Slice kt is multiplied while slice kt + 2 is on its way; slice kt + 1 has
    // landed and goes to the other stage, and its registers take the loads.
    if constexpr (W == 8) {
      // Two waves share a SIMD, one of each half of the workgroup. The halves
      // run a phase apart: while one fetches its operands of slice kt and stages
      // its part of slice kt + 1, the other has the matrix pipe to itself.
      // Slice kt + 1 is complete after the second half's phase, one barrier
      // before the first half reads it, and the stage it takes was last read
      // one barrier before the first half writes it.
      if (wave >= W / 2) __syncthreads();
      auto phases = [&](int kt, auto more) {
        const _Float16* cur = sh.stages + (kt & 1) * S::kStage;
        Operands o0, o1;
        fetch(cur, 0, o0);
        fetch(cur, 1, o1);
        more();
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_s_setprio(1);
        multiply(o0);
        multiply(o1);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
      };
      int kt = 0;
#pragma unroll 1
      for (; kt + 3 < nk; ++kt) {
        phases(kt, [&]() {
          put(sh.stages + (~kt & 1) * S::kStage, kt + 1);
          store_xp(kt + 1);
          load(kt + 2);
        });
      }
#pragma unroll 1
      for (; kt < nk; ++kt) {
        phases(kt, [&]() {
          if (kt + 1 < nk) {
            put(sh.stages + (~kt & 1) * S::kStage, kt + 1);
            store_xp(kt + 1);
          }
          if (kt + 2 < nk) load_any(kt + 2);
        });
      }
      if (wave < W / 2) __syncthreads();
    } else {
      auto both = [&](const _Float16* cur) {
        Operands o;
        fetch(cur, 0, o);
        multiply(o);
        fetch(cur, 1, o);
        multiply(o);
        __syncthreads();
      };
      int kt = 0;
#pragma unroll 1
      for (; kt + 3 < nk; ++kt) {
        put(sh.stages + (~kt & 1) * S::kStage, kt + 1);
        store_xp(kt + 1);
        load(kt + 2);
        __builtin_amdgcn_sched_barrier(0);  // (the scheduler would sink the loads to the slice's end)
        both(sh.stages + (kt & 1) * S::kStage);
      }
#pragma unroll 1
      for (; kt < nk; ++kt) {
        if (kt + 1 < nk) {
          put(sh.stages + (~kt & 1) * S::kStage, kt + 1);
          store_xp(kt + 1);
        }
        if (kt + 2 < nk) load_any(kt + 2);
        both(sh.stages + (kt & 1) * S::kStage);
      }
    }
  }

  // What the scales could not carry: marked rows and columns, and sums that are
  // not finite. (Each a matter of the output's own row and column, whatever else
  // is in the tile.)
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if ((small_a[p] >> lane & 1) != 0) sh.ta[PR * p + ar] = kMarked;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if ((small_b[j] >> lane & 1) != 0) sh.tb[2 * pair + j] = kMarked;
  }
  if (tid < kBN && sh.few[tid] >= kFewSmall) sh.tb[tid] = kMarked;
  __syncthreads();

  // (the lane id passes an empty asm so that none of the epilogue's addresses
  // is built before the loop and kept live across it)
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const int eli = ln & 31;
  const int ehi = ln >> 5;
  // output rows of accumulator register r: 32 i + 8 (r / 4) + 4 hi + r % 4 of the wave's
  const int ec = L::col(wave) + eli;  // tile column; block j: 32 j further
  bool odd = tid < rows && sh.ta[tid] == kMarked;
  if (tid < kBN && tl.n0 + tid < N) odd = odd || sh.tb[tid] == kMarked;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rl = wrow + 32 * i + 8 * (r >> 2) + 4 * ehi + (r & 3);
        acc[i][j][r] = __builtin_fmaf(low[i][j][r], 1.0F / kLowScale, acc[i][j][r]);
        odd = odd || (rl < rows && tl.n0 + ec + 32 * j < N && abs_bits(acc[i][j][r]) >= 0x7F800000U);
      }
    }
  }
  const bool redo = __syncthreads_or(odd ? 1 : 0) != 0;
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
  uint32_t* mask = reinterpret_cast<uint32_t*>(sh.cmax);  // [row][column / 32]
  int tb[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) tb[j] = sh.tb[ec + 32 * j];
  uint32_t again[TM] = {};  // bit 16 j + r: output (i, j, r) is one of those
  if (redo) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rl = wrow + 32 * i + 8 * (r >> 2) + 4 * ehi + (r & 3);
        const int ta = sh.ta[rl];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const bool a = rl < rows && tl.n0 + ec + 32 * j < N &&
                         (ta == kMarked || tb[j] == kMarked || abs_bits(acc[i][j][r]) >= 0x7F800000U);
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
      const int ta = sh.ta[rl];
      float* yrow = ytile + static_cast<std::size_t>(rl) * N + ec;
      float* comb = combined_row(rl);
      const float w = comb != nullptr ? sh.w[rl] : 0.0F;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (tl.n0 + ec + 32 * j >= N || (again[i] >> (16 * j + r) & 1) != 0) continue;
        emit(ldexpf(acc[i][j][r], -(ta + tb[j])), yrow + 32 * j, comb != nullptr ? comb + ec + 32 * j : nullptr, w);
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
  // quad q of plane row r sits at quad q ^ (r & 7) (B: q ^ (r / 2 & 7))
  load_any(0);
#pragma unroll 1
  for (int kt = 0; kt < nk; ++kt) {
    float* As = reinterpret_cast<float*>(sh.stages) + (kt & 1) * S::kStage32;
    float* Bs = As + S::kBM * kBK;
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int r = PR * p + ar;
      *reinterpret_cast<v4f*>(As + r * kBK + 4 * (ac ^ (r & 7))) = v4f{ra[p][0], ra[p][1], ra[p][2], ra[p][3]};
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int q = 0; q < KP / 4; ++q) {
        *reinterpret_cast<v4f*>(Bs + (2 * pair + j) * kBK + 4 * ((b_k / 4 + q) ^ (pair & 7))) =
            v4f{rb[4 * q][j], rb[4 * q + 1][j], rb[4 * q + 2][j], rb[4 * q + 3][j]};
      }
    }
    if (kt + 1 < nk) load_any(kt + 1);
    __syncthreads();  // (the other stage was last read before the previous slice's barrier)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      v4f b[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int col = CW * wave + 16 * j + fl;
        b[j] = *reinterpret_cast<const v4f*>(Bs + col * kBK + 4 * ((4 * c + g) ^ (col >> 1 & 7)));
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        if ((blocks >> i & 1) == 0) continue;
        const v4f a = *reinterpret_cast<const v4f*>(As + (16 * i + fl) * kBK + 4 * ((4 * c + g) ^ (fl & 7)));
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
          for (int j = 0; j < NJ; ++j) sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[j][s], sum[i][j], 0, 0, 0);
        }
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
  extern __shared__ __align__(16) _Float16 smem[];
  Lds sh;
  sh.stages = smem;
  sh.ta = reinterpret_cast<int32_t*>(smem + 2 * S::kStage);
  sh.tb = sh.ta + kBM;
  sh.cmax = reinterpret_cast<uint2*>(sh.tb + kBN);
  sh.few = reinterpret_cast<int32_t*>(sh.cmax + W * 64);
  sh.src = sh.few + kBN;
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
  const std::size_t lds = 2 * S::kStage * sizeof(_Float16) + (S::kBM + kBN) * sizeof(int32_t) +
                          W * 64 * sizeof(uint2) + kBN * sizeof(int32_t) + 2 * S::kBM * sizeof(int32_t) +
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
//    K and N both below 256 (chain T = 10296, E = 12, K = 100, N = 153 53 / 59 us, T =
//    2523, E = 10, K = 106, N = 667 49 / 53);
//  - problems of so few tiles that their smaller tiles spread over more CUs: with
//    K >= 512 below one 64 x 64 tile a CU (E = 8, K = 1024, N = 512, 1024 rows, 192 tiles
//    22 / 40 us; 4096 rows, 576 tiles 48 / 42), or 1.25 where the experts have less than
//    eight rows each (E = 8, K = 512, N = 2048, 32 rows 16.3 / 20.0); with shorter K,
//    where a tile's scales and first loads weigh more, below 2.5 (E = 16, K = 256,
//    N = 1024, 1600 rows 17.8 / 18.9; E = 8, K = 256, N = 1536, 1200 rows, 648 tiles
//    28.1 / 19.4), and up to 3 with K < 192 (E = 16, K = 128, N = 1024, 1600 rows, 656
//    tiles 11.3 / 15.0; E = 64, K = 128, N = 768, 1536 rows, 1056 tiles 18.2 / 12.8);
//  - few rows an expert where the FP32 side has its 128 x 128 tiles (two a CU): both
//    are bound by the weights, which those load straight into LDS. E = 64, K = 128,
//    N = 1024: 256 rows 8.6 / 11.7, 2048 rows 15.7 / 16.7, 3072 rows 19.6 / 18.0; E = 128,
//    K = 320, N = 1024: 16 rows each 34.0 / 36.1, 24 rows 49.0 / 41.0; K = 1024: 4 rows each
//    89 / 99, 16 rows 99 / 105, 24 rows 141 / 111; K = 4096: 4 rows each 314 / 349, 10 rows
//    342 / 358, 16 rows 365 / 359 (chain K = 2048, N = 768, 10 rows each 222 / 215).
bool split_gemm_ok(int k, int n, int experts, long rows, int cus) {
  if (k < 128 || n <= 64 || (k < 256 && n < 256)) return false;
  const long few = k < 192 ? 36 : (k < 512 ? 20 : (k < 2048 ? 16 : 8));  // rows an expert
  if (rows < few * experts && tiles(rows, experts, 128, n, 128) >= 2L * cus) return false;
  const long t = tiles(rows, experts, 64, n, 64);
  if (k >= 512) return 4 * t >= (rows < 8L * experts ? 5L : 4L) * cus;
  return k < 192 ? t > 3L * cus : 2 * t >= 5L * cus;
}

// 32-bit byte offsets: a tile's A rows (chain: all of X) and an expert's weights.
bool split_gemm_fits(const GemmParams& prm) {
  const long limit = 1L << 30;
  const long a_rows = prm.sorted_route != nullptr ? prm.dense_rows : 256;
  return prm.K > 0 && prm.N >= 2 && a_rows * prm.K < limit && static_cast<long>(prm.K + kBK) * prm.N < limit;
}

// Workgroup shape:
//  - eight waves on 128-row tiles where a CU gets hardly more than one tile:
//    more waves for it (E = 16, K = 2048, N = 300 with 8192 rows, 240 tiles: 72 us
//    against 89 with four waves; E = 64, K = 1024, N = 512, 4096 rows, 384
//    tiles: 34 / 39; E = 64, K = 512, N = 768, 512 rows, 408 tiles: 36 / 22);
//  - eight waves on 256-row tiles where there are many of them and the experts
//    have the rows (E = 8, K = 4096, N = 8192 with 16384 rows 3.58 ms against
//    3.90; E = 64, K = 1024, N = 512, 256 rows an expert: 68 / 71 us, but E = 64,
//    K = 512, N = 768, 256 rows an expert: 76 / 67).
//    Not for the chain: nothing runs under a tile's combine with one workgroup
//    a CU (T = 16384, E = 128, K = 2048, N = 768 chain 724 against 641 us);
//  - else four waves on 128-row tiles, two workgroups a CU.
hipError_t split_grouped(const GemmParams& prm, long rows_per_expert, long rows, int cus, SplitShape shape,
                         hipStream_t stream) {
  const bool chain = prm.sorted_route != nullptr;
  if (shape == SplitShape::kBySize) {
    if (2 * tiles(rows, prm.experts, 128, prm.N, kBN) <= 3L * cus) {
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
