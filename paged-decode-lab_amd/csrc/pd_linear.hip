// Matrix products of some hundred rows for MI355X (gfx950): Y = X W^T, bf16
// operands, float32 sums, with the gate of a gated MLP in the epilogue and
// several weight matrices of one input in a launch.
//
// A workgroup of four wavefronts a CU has a tile of BM features by 128 rows;
// a stage is 64 elements of K.  Copies from memory go straight to LDS (no
// registers, no LDS write instructions), kRing stages of them: 128 or
// 144 KB a CU for the 2 us to HBM.  Per stage and wavefront, one wait for its own
// copies of the next stage and one barrier; then it reads the next stage's
// operands, sends for the stage kRing ahead (its place is free: the operands
// of this stage are in registers) and multiplies this one.  Tiles that share
// rows of W are on one XCD and share its L2.
//
// Bound: LDS.  A stage of 128 x 128 is 64 KB of operand reads and 32 KB of
// copies, 0.37 us at the LDS rate, takes 0.44 us (0.21 of MFMAs) and took 0.85
// with the ring in registers and stores to LDS.  256 x 128 reads a quarter
// less for each product: 0.82 us.
//
// A product is worth it while its tiles are one round of the CUs: the start
// and end of a tile, 5 us, meet nobody else's work.  Of two tiles that are, 128
// is the shorter, and 256 is one round for twice the features.  Measured on
// MI355X, inputs of 2048, this form, with the ring in registers and library
// products with the gate's launch (host-bound below 768 rows: 18 us a product):
// 8192 features in two matrices at 512 rows 24, 28 and 36 us, at 1024 (256)
// 41, - and 44; gate and up of 6144 at 256 rows 24, 29 and 50, at 512 38 (256;
// 43 in two rounds of 128), 52 and 54, at 1024, two rounds of either, 66, - and
// 71, at 2049 145, - and 108; three matrices of 5120 in all at 512 rows 21, 27
// and 54.  Products of 2048 features, 64 tiles at 512 rows, take 20 us and with
// inputs of 6144 48; the library's take 13 and 22 to 29, and are used.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "pd_device.h"
#include "pd_internal.h"
#include "pd_launch.h"

namespace {

using namespace pdk;
using pd::aligned16;
using pd::as_stream;
using pd::launch_status;

constexpr int kMaxSegments = 4;
constexpr int BN = 128;

enum { kStore, kSiluMul };

struct LinearArgs {
  const uint16_t* x;
  const uint16_t* w[kMaxSegments];
  uint16_t* out[kMaxSegments];
  int m[kMaxSegments];
  int segments, rows, K, row_tiles, feature_tiles;
};

// Waits until at most `n` of this wavefront's copies are under way.
template <int n>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory");
}

// BM operand rows of W (kSiluMul: 32 features of the gate and the same 32 of
// up in turn) by BN rows of X; a stage is 64 elements of K.
template <int kEpi, int BM>
__global__ void __launch_bounds__(256, 1) linear_kernel(const LinearArgs a) {
  constexpr int FM = BM / 64, FN = BN / 64, kSteps = 4;
  constexpr int kPerTile = kEpi == kSiluMul ? BM / 2 : BM;  // features
  constexpr int kStage = (BM + BN) * 128, kRing = BM == 128 ? 4 : 3;
  // One array a stage: the compiler then tells a stage's reads from the copies
  // on their way into the others.
  __shared__ __attribute__((aligned(16))) char lds0[kStage], lds1[kStage], lds2[kStage],
      lds3[kRing == 4 ? kStage : 16];
  char* const ring[4] = {lds0, lds1, lds2, lds3};
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

  // Copy i of a wavefront fills rows 32 i + 8 wave .. + 7 of the stage, 16
  // bytes a lane in lane order, so the lanes' sources carry the swizzle.  Rows
  // past the matrix read as zeros and their products are not stored.
  const auto rsrc_of = [&](const uint16_t* base, int first, int count, int rows) {
    const int held = __builtin_amdgcn_readfirstlane(max(min(count, rows - first), 0));
    return buffer_rsrc(base + int64_t(first) * a.K, held * a.K * 2);
  };
  __amdgpu_buffer_rsrc_t wr[kEpi == kSiluMul ? 2 : 1];
  if constexpr (kEpi == kSiluMul) {
    wr[0] = rsrc_of(a.w[0], m0, kPerTile, M);
    wr[1] = rsrc_of(a.w[1], m0, kPerTile, M);
  } else {
    wr[0] = rsrc_of(a.w[seg], m0, BM, M);
  }
  const __amdgpu_buffer_rsrc_t xr = rsrc_of(a.x, n0, BN, a.rows);
  int at[BM / 32];
#pragma unroll
  for (int i = 0; i < BM / 32; ++i) {
    const int row = 32 * i + 8 * wave + lane / 8;
    at[i] = row * a.K * 2 + 16 * ((lane & 7) ^ kswz<64>(row));
  }

  struct Operands {
    u32x4_t w[kSteps][FM], x[kSteps][FN];
  };
  Operands ops[2];
  floatx16_t acc[FM][FN];
#pragma unroll
  for (int m = 0; m < FM; ++m)
#pragma unroll
    for (int n = 0; n < FN; ++n) acc[m][n] = floatx16_t{};

  const int stages = a.K / 64;
  const auto fetch = [&](int stage, char* to) {
    // Past the last stage it is copied again, so that the copies in flight are
    // the same number everywhere.
    const int k = min(stage, stages - 1) * 128;
    char* mine = to + wave * 1024;
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
      if constexpr (kEpi == kSiluMul)
        lds_copy16(wr[i & 1], mine + 4096 * i, at[i] - (i + 1) / 2 * 64 * a.K + k);
      else
        lds_copy16(wr[0], mine + 4096 * i, at[i] + k);
    }
#pragma unroll
    for (int i = 0; i < BN / 32; ++i) lds_copy16(xr, mine + BM * 128 + 4096 * i, at[i] + k);
  };
  const auto read = [&](const char* lds, Operands& o) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      const int at = col * 128 + 16 * ((2 * s + half) ^ kswz<64>(col));
#pragma unroll
      for (int m = 0; m < FM; ++m)
        o.w[s][m] = *reinterpret_cast<const u32x4_t*>(
            lds + (wm * (BM / 2) + 32 * m) * 128 + at);
#pragma unroll
      for (int n = 0; n < FN; ++n)
        o.x[s][n] = *reinterpret_cast<const u32x4_t*>(
            lds + (BM + wn * (BN / 2) + 32 * n) * 128 + at);
    }
  };
  const auto multiply = [&](const Operands& o) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
#pragma unroll
      for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n) acc[m][n] = mfma32(o.w[s][m], o.x[s][n], acc[m][n]);
  };

  constexpr int kCopies = (BM + BN) / 32, kUnroll = kRing == 4 ? 4 : 6;
#pragma unroll
  for (int i = 0; i < kRing; ++i) fetch(i, ring[i]);
  wait_copies<kCopies * (kRing - 1)>();
  lds_barrier();
  read(ring[0], ops[0]);
  // Stage k: its operands are in registers, so its place in LDS is free, and
  // stage k + 1 is there once every wavefront's copies of it are.
  const auto step = [&](int k, int u) {
    wait_copies<kCopies * (kRing - 2)>();
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(ring[(u + 1) % kRing], ops[(u + 1) & 1]);
    __builtin_amdgcn_sched_barrier(0);
    fetch(k + kRing, ring[u % kRing]);
    multiply(ops[u & 1]);
    __builtin_amdgcn_sched_barrier(0);
  };
  int k = 0;
  for (; k + kUnroll <= stages; k += kUnroll) {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) step(k + u, u);
  }
#pragma unroll
  for (int u = 0; u < kUnroll - 1; ++u) {
    if (k + u >= stages) break;
    step(k + u, u);
  }
  wait_copies<0>();  // none may land in LDS that has a new owner
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
    for (int m = 0; m < FM; m += kEpi == kSiluMul ? 2 : 1)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int f = m0 + wm * (kPerTile / 2) + 32 * (kEpi == kSiluMul ? m / 2 : m) + 8 * g +
                      4 * half;
        if (f >= M) continue;
        u32x2_t* out = reinterpret_cast<u32x2_t*>(a.out[seg] + int64_t(row) * M + f);
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          y[e] = acc[m][n][4 * g + e];
          if constexpr (kEpi == kSiluMul)
            y[e] = y[e] / (1.f + exp_fast(-y[e])) * acc[m + 1][n][4 * g + e];
        }
        *out = u32x2_t{pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])};
      }
  }
}

template <int kEpi, int BM>
int launch(LinearArgs& a, pd_stream_t stream) {
  constexpr int per = kEpi == kSiluMul ? BM / 2 : BM;
  int64_t tiles = 0;
  for (int i = 0; i < a.segments; ++i) tiles += (int64_t(a.m[i]) + per - 1) / per;
  a.row_tiles = (a.rows + BN - 1) / BN;
  const int64_t grid = (tiles + 7) / 8 * 8 * a.row_tiles;
  if (grid > 0x7fffffff) return pd::fail(PD_EINVAL, "grid dimension exceeds device limits");
  a.feature_tiles = int(tiles);
  hipLaunchKernelGGL((linear_kernel<kEpi, BM>), dim3(unsigned(grid)), dim3(256), 0,
                     as_stream(stream), a);
  return launch_status("pd_linears");
}

}  // namespace

extern "C" int pd_linears(const void* x, int32_t rows, int32_t dim, int32_t count,
                          const void* const* weights, const int32_t* features, void* const* outs,
                          int32_t form, int32_t tile, pd_stream_t stream) {
  pd::clear_error();
  if (rows < 0) return pd::fail(PD_EINVAL, "rows must be non-negative");
  if (rows == 0) return PD_OK;
  if (dim < 64 || dim % 64 || dim > 1 << 22)  // a tile's rows are one buffer under 2 GiB
    return pd::fail(PD_EINVAL, "input features must be a multiple of 64, at most 2^22");
  if (count < 1 || count > kMaxSegments || form < kStore || form > kSiluMul ||
      (form == kSiluMul && count != 2))
    return pd::fail(PD_EINVAL, "1 to %d matrices, 2 for gate and up", kMaxSegments);
  if (tile != 128 && tile != 256) return pd::fail(PD_EINVAL, "tiles of 128 or 256 features");
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
  if (tile == 128)
    return form == kSiluMul ? launch<kSiluMul, 128>(a, stream) : launch<kStore, 128>(a, stream);
  return form == kSiluMul ? launch<kSiluMul, 256>(a, stream) : launch<kStore, 256>(a, stream);
}
