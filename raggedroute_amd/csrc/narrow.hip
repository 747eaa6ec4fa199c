// Dense FP32 GEMM with at most 128 output columns and any K (the router GEMM
// of shapes the strip kernel does not cover: K > 256, or rows off 16 bytes),
// with the top-2 gate in its epilogue when the chain asks for it.
//
// A workgroup owns RB strips of 16 rows and all columns, wave w the columns
// [16 w, 16 w + 16). Slices of 64 k of both operands go through registers (two
// slices on their way) into one of two LDS stages, as they lie in memory, with
// the 16-byte quads of a row XOR-ed so that operand reads spread over the banks:
// a lane (li, g) of k chunk c reads the quad A[row li][16 c + 4 g .. + 3] and the
// floats B[16 c + 4 g + s][16 w + li], s = 0..3. (Both operands straight from
// global memory in operand order, twelve chunks ahead and without barriers, was
// bound by the loads: one takes 16 cycles a wave whatever its width, 80 a
// chunk and wave against 128 of MFMAs: T = 2048, E = 64, K = 1024 11.4 us; T = 16384,
// E = 128, K = 2048 125 us.)
// k order as in every FP32 GEMM here (chunks ascending, MFMA step s sums
// k = 16 c + 4 g + s over g): the results are those of the tiled kernel, bit
// for bit.
// Bound: few rows (one strip a workgroup), each wave's chain of K / 4 dependent
// MFMAs, 44 cycles each; many rows, the FP32 matrix pipe. Measured, tiled kernel
// / this: T = 2048, E = 64, K = 1024 15.2 / 9.6 us; T = 4096, E = 64, K = 333 8.3 /
// 5.8; T = 8192, E = 128, K = 2048 51 / 39; T = 16384, E = 128, K = 2048 82.8 / 67.1 us
// (128 TFLOP/s, 0.81 of the FP32 matrix peak; a loop of this launch alone: the bench,
// after minutes of other load, reads 77 - 79, before 85 - 95), and with the gate,
// whose own launch is gone, 17.7 / 10.7, 10.9 / 6.9, 55.3 / 41.1 and 88.1 / 71.4 us.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "gate.h"
#include "launchers.h"
#include "tiles.h"
#include "wave.h"

namespace rr::kern {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;                 // rows per strip
constexpr int kBK = 64;                   // k per slice
constexpr int kBufferFlags = 0x00027000;  // raw 32-bit buffer

struct NarrowParams {
  const float* A;  // [M, K]
  const float* W;  // [K, N]
  float* C;        // [M, N]
  int M;
  int K;
  int N;
  // gate
  int32_t* ids;
  float* weights;
  float* y_zero;  // optional: [M, y_cols] zeroed
  int y_cols;
};

template <int W, int RB, bool GATE>
__global__ __launch_bounds__(W * 64, 2) void rr_narrow_gemm_kernel(NarrowParams p) {
  constexpr int kThreads = W * 64;
  constexpr int kCols = 16 * W;
  constexpr int kLd = kCols + 4;  // padded row of the logit tile
  constexpr int kTileRows = kRows * RB;
  constexpr int kAFloats = kTileRows * kBK;
  constexpr int kStage = kAFloats + kBK * kCols;
  constexpr int kAQuads = kAFloats / 4;
  constexpr int NA = (kAQuads + kThreads - 1) / kThreads;  // quads a thread stages (W = 8, RB = 1: half the threads)
  constexpr int NB = kBK * kCols / 4 / kThreads;
  static_assert(kTileRows * kLd <= 2 * kStage, "the logit tile fits the stages");
  extern __shared__ __align__(16) float lds[];  // [2][kStage]; the logit tile after the loop
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4;
  const int li = lane & 15;
  const int K = p.K;
  const int N = p.N;
  const int row0 = static_cast<int>(blockIdx.x) * kTileRows;
  const int rows = p.M - row0 < kTileRows ? p.M - row0 : kTileRows;
  const int col = 16 * wave + li;
  const int nk = (K + kBK - 1) / kBK;
  // the last slice is loaded float by float where a quad could cross the end of a row
  const int guarded = (K % kBK != 0 || (N & 3) != 0) ? nk - 1 : nk;

  const auto a_base = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.A + static_cast<std::size_t>(row0) * K), 0, -1, kBufferFlags);
  const auto b_base = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.W), 0, -1, kBufferFlags);
  // A quad f: row f / 16, k quad f % 16; B quad f: k row f / (kCols / 4)
  uint32_t a_lane[NA], b_lane[NB];
  int a_put[NA], b_put[NB];
  const bool loads_a = NA * kThreads == kAQuads || tid < kAQuads;  // (wave-uniform)
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int f = tid + i * kThreads;
    const int r = f >> 4, q = f & 15;
    // (rows past the last repeat it)
    a_lane[i] = 4u * (static_cast<uint32_t>(r < rows ? r : rows - 1) * static_cast<uint32_t>(K) + 4u * static_cast<uint32_t>(q));
    a_put[i] = r * kBK + 4 * (q ^ (r & 15));
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int f = tid + i * kThreads;
    const int k = f / (kCols / 4), q = f % (kCols / 4);
    // (columns past N repeat the last quad: their products are not stored)
    b_lane[i] = 4u * (static_cast<uint32_t>(k) * static_cast<uint32_t>(N) + static_cast<uint32_t>(4 * q < N ? 4 * q : N - 4));
    b_put[i] = kAFloats + k * kCols + 4 * (q ^ (4 * ((k >> 2) & 3)));
  }
  struct Slice {
    v4f a[NA];
    v4f b[NB];
  };
  auto b_row = [&](int kt) { return 4u * static_cast<uint32_t>(kt) * kBK * static_cast<uint32_t>(N); };
  auto load = [&](int kt, Slice& s) {
    if (loads_a) {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        s.a[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(a_base, a_lane[i], 4 * kBK * kt, 0));
      }
    }
    // (a quad that crosses N reads the next k row's first floats)
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      s.b[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(b_base, b_lane[i], b_row(kt), 0));
    }
  };
  auto load_any = [&](int kt, Slice& s) {
    if (kt != guarded) {
      load(kt, s);
      return;
    }
    if (loads_a) {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const int k = kt * kBK + 4 * ((tid + i * kThreads) & 15);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float v = 0.0F;
          if (k + j < K) v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(a_base, a_lane[i] + 4 * j, 4 * kBK * kt, 0));
          s.a[i][j] = v;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int f = tid + i * kThreads;
      const int k = kt * kBK + f / (kCols / 4), n = 4 * (f % (kCols / 4));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = 0.0F;
        if (k < K && (n >= N || n + j < N)) {
          v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b_base, b_lane[i] + 4 * j, b_row(kt), 0));
        }
        s.b[i][j] = v;
      }
    }
  };
  auto put = [&](float* __restrict__ st, const Slice& s) {
    if (loads_a) {
#pragma unroll
      for (int i = 0; i < NA; ++i) *reinterpret_cast<v4f*>(st + a_put[i]) = s.a[i];
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) *reinterpret_cast<v4f*>(st + b_put[i]) = s.b[i];
  };
  v4f acc[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) acc[i] = v4f{0.0F, 0.0F, 0.0F, 0.0F};
  // column quad of the lane in k rows whose (k >> 2) & 3 is g
  const int b_get = kAFloats + 4 * g * kCols + 4 * ((4 * wave + (li >> 2)) ^ (4 * g)) + (li & 3);
  auto multiply = [&](const float* __restrict__ st) {
#pragma unroll
    for (int c = 0; c < kBK / 16; ++c) {
      v4f a[RB], b;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        a[i] = *reinterpret_cast<const v4f*>(st + (kRows * i + li) * kBK + 4 * ((4 * c + g) ^ li));
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) b[s] = st[b_get + (16 * c + s) * kCols];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int i = 0; i < RB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], b[s], acc[i], 0, 0, 0);
      }
    }
  };

  // slice i is held in register set (i - 1) & 1 until it goes to stage i & 1
  Slice s0, s1;
  load_any(0, s0);
  if (nk > 2) load_any(2, s1);  // (set of even slices; slice 1 follows slice 0 into s0)
  put(lds, s0);
  if (nk > 1) load_any(1, s0);
  __syncthreads();
  int kt = 0;
#pragma unroll 1
  for (; kt + 5 < nk; kt += 2) {
    put(lds + kStage, s0);
    load(kt + 3, s0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(lds);
    __syncthreads();
    put(lds, s1);
    load(kt + 4, s1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(lds + kStage);
    __syncthreads();
  }
#pragma unroll 1
  for (; kt < nk; kt += 2) {
    if (kt + 1 < nk) put(lds + kStage, s0);
    if (kt + 3 < nk) load_any(kt + 3, s0);
    multiply(lds);
    __syncthreads();
    if (kt + 1 < nk) {
      if (kt + 2 < nk) put(lds, s1);
      if (kt + 4 < nk) load_any(kt + 4, s1);
      multiply(lds + kStage);
      __syncthreads();
    }
  }

  float* s_lg = lds;  // (every wave is past the last slice)
#pragma unroll
  for (int i = 0; i < RB; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rl = kRows * i + 4 * g + r;
      if constexpr (GATE) s_lg[rl * kLd + col] = acc[i][r];
      if (rl < rows && col < N) {
        float* out = p.C + static_cast<std::size_t>(row0 + rl) * N + col;
        if constexpr (GATE) {
          __builtin_nontemporal_store(acc[i][r], out);  // (the gate reads LDS)
        } else {
          *out = acc[i][r];
        }
      }
    }
  }
  if constexpr (GATE) {
    // the combined output rows of this workgroup's tokens
    if (p.y_zero != nullptr) {
      float* y = p.y_zero + static_cast<std::size_t>(row0) * p.y_cols;
      const long n = static_cast<long>(rows) * p.y_cols;
      if ((p.y_cols & 3) == 0 && (reinterpret_cast<std::uintptr_t>(p.y_zero) & 15u) == 0) {
        for (long i = tid; i < n / 4; i += kThreads) reinterpret_cast<v4f*>(y)[i] = v4f{0.0F, 0.0F, 0.0F, 0.0F};
      } else {
        for (long i = tid; i < n; i += kThreads) y[i] = 0.0F;
      }
    }
    // Top-2 of each row: a row's lanes take four adjacent columns each and merge
    // with register moves; keys carry the expert, so the order does not matter.
    constexpr int kRowLanes = kCols / 4;  // 16 or 32
    constexpr int kPerPass = kThreads / kRowLanes;  // 16 rows
    static_assert(kPerPass == kRows, "one strip per pass");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const int rl = kRows * i + tid / kRowLanes;
      const int c0 = 4 * (tid % kRowLanes);
      const v4f lg = *reinterpret_cast<const v4f*>(s_lg + rl * kLd + c0);
      uint64_t k1 = 0, k2 = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (c0 + j < N) rr::dev::insert_key(rr::dev::gate_key(lg[j], c0 + j), k1, k2);
      }
      rr::dev::merge_top2_row16(k1, k2);
      if constexpr (kRowLanes == 32) {  // the row's other 16 lanes
        rr::dev::merge_pair(k1, k2, rr::dev::shfl_xor_u64(k1, 16), rr::dev::shfl_xor_u64(k2, 16));
      }
      if (tid % kRowLanes == 0 && rl < rows) {
        float w1, w2;
        rr::dev::gate_weights(k1, k2, &w1, &w2);
        const std::size_t row = static_cast<std::size_t>(row0 + rl);
        p.ids[2 * row] = rr::dev::key_expert(k1);
        p.ids[2 * row + 1] = rr::dev::key_expert(k2);
        p.weights[2 * row] = w1;
        p.weights[2 * row + 1] = w2;
      }
    }
  }
}

template <int W, int RB, bool GATE>
hipError_t launch_one(const NarrowParams& p, hipStream_t stream) {
  constexpr std::size_t kLds = 2 * (kRows * RB + 16 * W) * kBK * sizeof(float);
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(rr_narrow_gemm_kernel<W, RB, GATE>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kLds));
  if (attr != hipSuccess) return attr;
  const unsigned grid = static_cast<unsigned>((p.M + kRows * RB - 1) / (kRows * RB));
  rr_narrow_gemm_kernel<W, RB, GATE><<<grid, W * 64, kLds, stream>>>(p);
  return hipGetLastError();
}

template <int W, int RB>
hipError_t launch(const NarrowParams& p, bool gate, hipStream_t stream) {
  return gate ? launch_one<W, RB, true>(p, stream) : launch_one<W, RB, false>(p, stream);
}

template <int W>
hipError_t launch_rows(const NarrowParams& p, bool gate, int cus, hipStream_t stream) {
  // the most strips a workgroup that still give every CU a workgroup
  const long strips = (static_cast<long>(p.M) + kRows - 1) / kRows;
  if (strips >= 4L * cus) return launch<W, 4>(p, gate, stream);
  if (strips >= 2L * cus) return launch<W, 2>(p, gate, stream);
  return launch<W, 1>(p, gate, stream);
}

}  // namespace

bool narrow_gemm_ok(int m, int n, int k) {
  // 32-bit byte offsets: 64 rows of A, all of W
  return m > 0 && n >= 4 && n <= 128 && k > 0 && k < (1 << 22);
}

hipError_t narrow_gemm(const float* a, const float* b, float* c, int m, int n, int k, int32_t* gate_ids,
                       float* gate_weights, float* y_zero, int y_cols, int cus, hipStream_t stream) {
  NarrowParams p{};
  p.A = a;
  p.W = b;
  p.C = c;
  p.M = m;
  p.K = k;
  p.N = n;
  p.ids = gate_ids;
  p.weights = gate_weights;
  p.y_zero = y_zero;
  p.y_cols = y_cols;
  const bool gate = gate_ids != nullptr;
  return n <= 64 ? launch_rows<4>(p, gate, cus, stream) : launch_rows<8>(p, gate, cus, stream);
}

}  // namespace rr::kern
