// Matrix products of some hundred rows for MI355X (gfx950): Y = X W^T, bf16
// operands, float32 sums, with the gate of a gated MLP in the epilogue and
// several weight matrices of one input in a launch.
//
// Bound: the weights' way in.  At 512 rows each weight is used 512 times, so
// the product is short and a workgroup streams its rows of W from HBM, about 2
// us away: the next kRing stages (32 KB each, 128 KB of a CU's register file)
// are always in flight to registers.  From there a stage goes to LDS, one of
// two buffers, and as 32x32x16 MFMA operands to registers a stage ahead:
//   write the next stage to LDS and load the stage kRing ahead (the writes
//   land under) the first half of this stage's products; barrier; read the
//   next stage's operands under the second half.
// One workgroup of four wavefronts a CU, each a quarter of the 128 x 128 tile.
// Tiles that share rows of W are on one XCD and share its L2.  A stage takes
// 0.85 us however few rows there are, so a product is worth it while its tiles
// are one round of the CUs.
//
// Measured on MI355X, inputs of 2048, this form and library products with the
// gate's launch: 8192 features in two matrices 28 and 38 us of kernels at 512
// rows; gate and up of 6144 29 and 50 us at 256, 52 and 55 at 512 (two
// rounds); three matrices of 5120 in all 27 and 40 us at 512 (53 us of host
// time).  Products of 2048 features, 64 such tiles at 512 rows, were no faster
// than the library's with 64 x 64 tiles (13.5 and 13.4 us; 31 and 29 us with
// inputs of 6144) and are left to it.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "pd_device.h"
#include "pd_internal.h"

namespace {

using namespace pdk;

typedef float floatx16_t __attribute__((ext_vector_type(16)));

constexpr int kMaxSegments = 4;
constexpr int kRing = 4;

constexpr int BM = 128, BN = 128;

enum { kStore, kSiluMul };

struct LinearArgs {
  const uint16_t* x;
  const uint16_t* w[kMaxSegments];
  uint16_t* out[kMaxSegments];
  int m[kMaxSegments];
  int segments, rows, K, row_tiles, feature_tiles;
};

__device__ __forceinline__ floatx16_t mfma32(u32x4_t a, u32x4_t b, floatx16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// BM operand rows of W (kSiluMul: 32 features of the gate and the same 32 of
// up in turn) by BN rows of X; a stage is 64 elements of K.
template <int kEpi>
__global__ void __launch_bounds__(256, 1) linear_kernel(const LinearArgs a) {
  constexpr int FM = BM / 64, FN = BN / 64, kSteps = 4;
  constexpr int kW = BM * 8 / 256, kX = BN * 8 / 256;       // pieces per thread
  constexpr int kPerTile = kEpi == kSiluMul ? BM / 2 : BM;  // features
  static_assert(kEpi != kSiluMul || FM == 2, "a wavefront's two blocks are gate and up");
  __shared__ __attribute__((aligned(16))) char lds[2][(BM + BN) * 128];
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;

  // Eight feature tiles in turn, one an XCD, each for every row tile.
  const int group = blockIdx.x / (8 * a.row_tiles), in = blockIdx.x % (8 * a.row_tiles);
  int tile = 8 * group + in % 8;
  const int n0 = in / 8 * BN;
  if (tile >= a.feature_tiles) return;
  int seg = 0;
  if constexpr (kEpi == kStore) {
    for (; seg < a.segments - 1; ++seg) {
      const int tiles = (a.m[seg] + kPerTile - 1) / kPerTile;
      if (tile < tiles) break;
      tile -= tiles;
    }
  }
  const int m0 = tile * kPerTile, M = a.m[seg];

  // Piece i of this thread: its source row (clamped to the last one, whose
  // copies are not stored) and its place in a stage.
  const uint16_t *wp[kW], *xp[kX];
  int wd[kW], xd[kX];
  const auto place_of = [&](int i, int& row, int& at, int& k) {
    const int idx = 256 * i + tid, piece = idx & 7;
    row = idx / 8;
    k = 8 * piece;
    at = row * 128 + 16 * (piece ^ kswz<64>(row));
  };
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    int row, k;
    place_of(i, row, wd[i], k);
    if constexpr (kEpi == kSiluMul) {
      const int f = min(m0 + 32 * (row >> 6) + (row & 31), M - 1);
      wp[i] = ((row >> 5) & 1 ? a.w[1] : a.w[0]) + int64_t(f) * a.K + k;
    } else {
      wp[i] = a.w[seg] + int64_t(min(m0 + row, M - 1)) * a.K + k;
    }
  }
#pragma unroll
  for (int i = 0; i < kX; ++i) {
    int row, k;
    place_of(i, row, xd[i], k);
    xp[i] = a.x + int64_t(min(n0 + row, a.rows - 1)) * a.K + k;
    xd[i] += BM * 128;
  }

  struct Stage {
    u32x4_t w[kW], x[kX];
  };
  struct Operands {
    u32x4_t w[kSteps][FM], x[kSteps][FN];
  };
  Stage ring[kRing];
  Operands ops[2];
  floatx16_t acc[FM][FN];
#pragma unroll
  for (int m = 0; m < FM; ++m)
#pragma unroll
    for (int n = 0; n < FN; ++n) acc[m][n] = floatx16_t{};

  const int stages = a.K / 64;
  const auto fetch = [&](int stage, Stage& s) {
    // Past the last stage it is loaded again, so that the loads in flight are
    // the same number everywhere.
    const int64_t k = int64_t(min(stage, stages - 1)) * 64;
#pragma unroll
    for (int i = 0; i < kW; ++i) s.w[i] = load16(wp[i] + k);
#pragma unroll
    for (int i = 0; i < kX; ++i) s.x[i] = load16(xp[i] + k);
  };
  const auto put = [&](int buf, const Stage& s) {
#pragma unroll
    for (int i = 0; i < kW; ++i) *reinterpret_cast<u32x4_t*>(lds[buf] + wd[i]) = s.w[i];
#pragma unroll
    for (int i = 0; i < kX; ++i) *reinterpret_cast<u32x4_t*>(lds[buf] + xd[i]) = s.x[i];
  };
  const auto read = [&](int buf, Operands& o) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int at = col * 128 + 16 * ((2 * s + half) ^ kswz<64>(col));
#pragma unroll
      for (int m = 0; m < FM; ++m)
        o.w[s][m] = *reinterpret_cast<const u32x4_t*>(
            lds[buf] + (wm * (BM / 2) + 32 * m) * 128 + at);
#pragma unroll
      for (int n = 0; n < FN; ++n)
        o.x[s][n] = *reinterpret_cast<const u32x4_t*>(
            lds[buf] + (BM + wn * (BN / 2) + 32 * n) * 128 + at);
    }
  };
  const auto multiply = [&](const Operands& o, int from, int to) {
#pragma unroll
    for (int s = from; s < to; ++s)
#pragma unroll
      for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n) acc[m][n] = mfma32(o.w[s][m], o.x[s][n], acc[m][n]);
  };

  // Scheduling barriers keep the loads in this order, which the waits count on.
#pragma unroll
  for (int i = 0; i < kRing; ++i) {
    fetch(i, ring[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  put(0, ring[0]);
  __builtin_amdgcn_sched_barrier(0);
  fetch(kRing, ring[0]);
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();
  read(0, ops[0]);
  // Every exit leaves the loop for good: a way back to its head would put the
  // shortest path's waits there.
  for (int k = 0;;) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
      const int next = (u + 1) % kRing;
      put((u + 1) & 1, ring[next]);
      __builtin_amdgcn_sched_barrier(0);
      fetch(k + 1 + kRing, ring[next]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(ops[u & 1], 0, kSteps / 2);
      __builtin_amdgcn_sched_barrier(0);
      lds_barrier();
      read((u + 1) & 1, ops[(u + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(ops[u & 1], kSteps / 2, kSteps);
      __builtin_amdgcn_sched_barrier(0);
      if (++k == stages) goto done;
    }
  }
done:
  // The last MFMAs and the reads below are in different blocks.
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int m = 0; m < FM; ++m)
#pragma unroll
    for (int n = 0; n < FN; ++n) asm volatile("" : "+v"(acc[m][n]));

  // Element i of a block: feature 8 (i / 4) + 4 half + i % 4, row `col`.
#pragma unroll
  for (int n = 0; n < FN; ++n) {
    const int row = n0 + wn * (BN / 2) + 32 * n + col;
    if (row >= a.rows) continue;
#pragma unroll
    for (int m = 0; m < (kEpi == kSiluMul ? 1 : FM); ++m)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int f = m0 + wm * (kPerTile / 2) + 32 * m + 8 * g + 4 * half;
        if (f >= M) continue;
        u32x2_t* out = reinterpret_cast<u32x2_t*>(a.out[seg] + int64_t(row) * M + f);
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y[e] = acc[m][n][4 * g + e];
          if constexpr (kEpi == kSiluMul)
            y[e] = y[e] / (1.f + exp_fast(-y[e])) * acc[1][n][4 * g + e];
        }
        *out = u32x2_t{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])};
      }
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int kEpi>
int launch(LinearArgs& a, pd_stream_t stream) {
  constexpr int per = kEpi == kSiluMul ? BM / 2 : BM;
  int64_t tiles = 0;
  for (int i = 0; i < a.segments; ++i) tiles += (int64_t(a.m[i]) + per - 1) / per;
  a.row_tiles = (a.rows + BN - 1) / BN;
  const int64_t grid = (tiles + 7) / 8 * 8 * a.row_tiles;
  if (grid > 0x7fffffff) return pd::fail(PD_EINVAL, "grid dimension exceeds device limits");
  a.feature_tiles = int(tiles);
  hipLaunchKernelGGL(linear_kernel<kEpi>, dim3(unsigned(grid)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), a);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    return pd::fail(PD_ELAUNCH, "pd_linears launch failed: %s", hipGetErrorString(err));
  return PD_OK;
}

}  // namespace

extern "C" int pd_linears(const void* x, int32_t rows, int32_t dim, int32_t count,
                          const void* const* weights, const int32_t* features, void* const* outs,
                          int32_t form, pd_stream_t stream) {
  pd::clear_error();
  if (rows < 0) return pd::fail(PD_EINVAL, "rows must be non-negative");
  if (rows == 0) return PD_OK;
  if (dim < 64 || dim % 64) return pd::fail(PD_EINVAL, "input features must be a multiple of 64");
  if (count < 1 || count > kMaxSegments || form < kStore || form > kSiluMul ||
      (form == kSiluMul && count != 2))
    return pd::fail(PD_EINVAL, "1 to %d matrices, 2 for gate and up", kMaxSegments);
  if (!x || !weights || !features || !outs || !aligned16(x))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  LinearArgs a{};
  for (int i = 0; i < count; ++i) {
    const void* out = outs[form == kSiluMul ? 0 : i];
    if (!weights[i] || !out || !aligned16(weights[i]) || !aligned16(out) || features[i] < 4 ||
        features[i] % 4 || features[i] != features[form == kSiluMul ? 0 : i])
      return pd::fail(PD_EINVAL, "weights and outputs must be aligned, features multiples of 4");
    a.w[i] = static_cast<const uint16_t*>(weights[i]);
    a.out[i] = static_cast<uint16_t*>(outs[form == kSiluMul ? 0 : i]);
    a.m[i] = features[i];
  }
  a.x = static_cast<const uint16_t*>(x);
  a.segments = form == kSiluMul ? 1 : count, a.rows = rows, a.K = dim;
  return form == kSiluMul ? launch<kSiluMul>(a, stream) : launch<kStore>(a, stream);
}
