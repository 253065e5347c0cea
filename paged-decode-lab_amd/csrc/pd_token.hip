// One token per sequence through a decoder layer, for MI355X (gfx950): the
// matrix products of up to 16 rows and the gated delta rule's single step.
//
// Bound: HBM.  Every weight is read once, 2 bytes for 2 flops a row, so the
// products keep the whole chip's loads in flight and fold everything between
// them (norms, gates, convolution, residual) into their prologues and
// epilogues: a linear-attention layer is five launches, none of which moves
// more than its weights and the state.
//
// Products.  A workgroup computes 16 operand rows of weights for all
// activation rows: its wavefronts split K in units of 64 elements (whole
// 128-byte lines of each weight row) and run 16x16x32 MFMAs, weights as the
// row operand and the activations as the column operand, so the cost is the
// same for 1 to 16 rows.  The operand rows are (kForm)
//   kWide   16 features;
//   kHalves 8 features, twice: rows 8-15 take the second half of K, as do
//           the activations' columns 8-15, and the two diagonal blocks of the
//           result are the halves' sums.  Up to 8 activation rows; twice the
//           workgroups where 16 features each would not fill the CUs;
//   kPairs  8 features of two matrices (gate and up).
//
// Loads return in order, so what is needed first is issued first: the input
// rows, then a wavefront's whole share of the weights, then the epilogue's
// operands; the norm runs while the weights arrive.  Barriers are lds_barrier,
// which leaves the weight loads in flight.  With more tiles than resident
// workgroups (the vocabulary), a workgroup walks tiles and each unit's
// registers take the next tile's weights as soon as its MFMAs have read them.
//
// Measured on MI355X, one row of 2048 (6144 for down), in a captured sequence:
// qkv z b a with the convolution (8224 features) 9.7 us, gate and up (2 x
// 6144) 11.6, down 7.0, out 4.0, vocabulary (151936) 113 (5.5 TB/s), delta
// step 4.5; of each about 2.5 us is the launch's ramp and tail.  A 24-layer
// decode step: 2817 us with library products, 1092 with these.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "pd_device.h"
#include "pd_internal.h"
#include "pd_launch.h"

namespace {

using namespace pdk;
using pd::all_aligned16;
using pd::as_stream;
using pd::launch_status;
using pd::u16;

constexpr int kMaxRows = 16;     // activation rows of a product
constexpr int kMaxSegments = 4;  // weight matrices sharing one input
constexpr int kFlight = 8;       // units of 64 elements a wavefront has in flight
constexpr int kNormWaves = 4;    // of a normed product's workgroup
constexpr int kPlainWaves = 8;

struct TokenArgs {
  const uint16_t* x;       // input rows [rows, K]
  const uint16_t* norm;    // kNorm: RMS weight (1 + w)
  const uint16_t* gate;    // kGated: x[n, k] times sigmoid(gate[n, k / D, k % D]), heads 2 D
                           // apart, D = 2^head_shift
  const uint16_t* w[kMaxSegments];
  void* out[kMaxSegments];
  int m[kMaxSegments];     // output features of each matrix
  const uint16_t* taps;    // kConv: first matrix's channels
  uint16_t* conv_state;
  int segments, rows, K, head_shift, has_prev, tiles;
  float eps;
};

enum { kPlain, kNorm, kGated };               // prologues
enum { kStore, kConv, kResidual, kSiluMul };  // epilogues
enum { kWide, kHalves, kPairs };              // forms

// Input rows normed to bf16 in LDS, rows K + 8 elements apart.  kItems rows of
// up to 8 elements a thread (K <= 2048) are held in registers between the sum
// of squares and the scaling; kItems = 0 reads any rows twice, a wavefront a
// row.  `between` issues the weight loads once the row loads are out.
template <int kItems, typename Between>
__device__ __forceinline__ void norm_rows(const TokenArgs& a, uint16_t* h, float* sums, int w,
                                          int lane, Between between) {
  if constexpr (kItems == 0) {
    for (int n = w; n < a.rows; n += kNormWaves) {
      const uint16_t* x = a.x + int64_t(n) * a.K;
      float ss = 0.f;
      for (int k = 8 * lane; k < a.K; k += 512) {
        float v[8];
        unpack8(load16(x + k), v);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
      }
      const float r = rsqrtf(wave_sum(ss) / a.K + a.eps);
      for (int k = 8 * lane; k < a.K; k += 512) {
        float v[8], g[8];
        unpack8(load16(x + k), v);
        unpack8(load16(a.norm + k), g);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = v[e] * r * (1.f + g[e]);
        *reinterpret_cast<u32x4_t*>(h + n * (a.K + 8) + k) = pack8(v);
      }
    }
    between();
  } else {
    const int k = 8 * (64 * w + lane);
    const bool live = k < a.K;
    u32x4_t x[kItems], g = {};
#pragma unroll
    for (int n = 0; n < kItems; ++n) {
      x[n] = u32x4_t{};
      if (live && n < a.rows) x[n] = load16(a.x + int64_t(n) * a.K + k);
    }
    if (live) g = load16(a.norm + k);
    between();
#pragma unroll
    for (int n = 0; n < kItems; ++n) {
      float v[8], ss = 0.f;
      unpack8(x[n], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
      ss = wave_sum(ss);
      if (lane == 0) sums[n * kNormWaves + w] = ss;
    }
    lds_barrier();
    float gain[8];
    unpack8(g, gain);
#pragma unroll
    for (int n = 0; n < kItems; ++n) {
      const floatx4_t s = *reinterpret_cast<const floatx4_t*>(sums + n * kNormWaves);
      const float r = rsqrtf((s[0] + s[1] + s[2] + s[3]) / a.K + a.eps);
      float v[8];
      unpack8(x[n], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = v[e] * r * (1.f + gain[e]);
      if (live && n < a.rows) *reinterpret_cast<u32x4_t*>(h + n * (a.K + 8) + k) = pack8(v);
    }
  }
  lds_barrier();
}

template <int kPro, int kEpi, int kForm, int kItems, bool kWalk>
__global__ void __launch_bounds__(64 * (kPro == kNorm ? kNormWaves : kPlainWaves), kPro == kNorm ? 3 : 2)
token_kernel(const TokenArgs a) {
  constexpr int kWaves = kPro == kNorm ? kNormWaves : kPlainWaves;
  constexpr int kFeatures = kForm == kWide ? 16 : 8;
  // [2][kWaves][16][16] partial results of two tiles in turn, [8][4] sums of
  // squares, then the normed rows.
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* red = reinterpret_cast<float*>(smem);
  float* sums = red + 2 * kWaves * 256;
  uint16_t* h = reinterpret_cast<uint16_t*>(sums + 32);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Operand lanes: weight row (and half of K), activation row, 8-element piece.
  const int quad = lane >> 4, op = lane & 15;
  const int second = kForm == kWide ? 0 : op >> 3;
  const int n = min(kForm == kHalves ? op & 7 : op, a.rows - 1);
  const int k_part = kForm == kHalves ? a.K / 2 : a.K, units = k_part / 64;
  const int k_lane = (kForm == kHalves ? second * k_part : 0) + 8 * quad;

  // The segment and first feature of a tile.
  const auto locate = [&](int tile, int& seg) {
    seg = 0;
    if constexpr (kEpi == kStore || kEpi == kConv) {
      for (; seg < a.segments - 1; ++seg) {
        const int tiles = (a.m[seg] + kFeatures - 1) / kFeatures;
        if (tile < tiles) break;
        tile -= tiles;
      }
    }
    return tile * kFeatures;
  };
  const auto weight_row = [&](int tile) {
    int seg;
    const int m0 = locate(tile, seg);
    const int feature = min(m0 + (op & (kFeatures - 1)), a.m[seg] - 1);
    const uint16_t* base = kForm == kPairs && second ? a.w[1] : a.w[seg];
    return base + int64_t(feature) * a.K + k_lane;
  };

  u32x4_t wr[kFlight][2], xr[kFlight][2];
  const auto load_unit = [&](const uint16_t* wp, int i, int u) {
    wr[i][0] = load16(wp + 64 * u);
    wr[i][1] = load16(wp + 64 * u + 32);
  };
  const auto load_inputs = [&](int u0) {
#pragma unroll
    for (int i = 0; i < kFlight; ++i) {
      const int u = u0 + i * kWaves;
      if (u < units) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int k = k_lane + 64 * u + 32 * s;
          xr[i][s] = load16(a.x + int64_t(n) * a.K + k);
        }
      }
    }
  };
  const auto gate_inputs = [&](int u0) {
#pragma unroll
    for (int i = 0; i < kFlight; ++i) {
      const int u = u0 + i * kWaves;
      if (u < units) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int k = k_lane + 64 * u + 32 * s;
          const int d = (1 << a.head_shift) - 1;
          float v[8], g[8];
          unpack8(load16(a.gate + 2 * (int64_t(n) * a.K + (k & ~d)) + (k & d)), g);
          unpack8(xr[i][s], v);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= sigmoid(g[e]);
          xr[i][s] = pack8(v);
        }
      }
    }
  };

  int tile = blockIdx.x;
  const uint16_t* wp = weight_row(tile);
  const auto load_weights = [&](const uint16_t* from, int u0) {
#pragma unroll
    for (int i = 0; i < kFlight; ++i)
      if (u0 + i * kWaves < units) load_unit(from, i, u0 + i * kWaves);
  };
  if constexpr (kPro == kNorm) {
    norm_rows<kItems>(a, h, sums, w, lane, [&] { load_weights(wp, w); });
  } else {
    load_inputs(w);
    if constexpr (kPro == kGated) gate_inputs(w);
    load_weights(wp, w);
  }

  for (int turn = 0;; ++turn) {
    int seg;
    const int m0 = locate(tile, seg), M = a.m[seg];
    // The epilogue's element of this thread, and its operands.
    const int r = tid & 15, row = tid >> 4, m = m0 + r;
    const bool mine = tid < 256 && r < kFeatures && row < a.rows && m < M;
    const int64_t at = int64_t(row) * M + m;
    uint16_t before = 0;
    u32x2_t held = {0, 0}, taps = {0, 0};
    if constexpr (kEpi == kResidual) {
      if (mine) before = static_cast<const uint16_t*>(a.out[0])[at];
    } else if constexpr (kEpi == kConv) {
      if (mine && seg == 0) {
        taps = *reinterpret_cast<const u32x2_t*>(a.taps + 4 * m);
        if (a.has_prev) held = *reinterpret_cast<const u32x2_t*>(a.conv_state + 4 * at);
      }
    }

    const int next = tile + gridDim.x;
    const bool more_tiles = kWalk && next < a.tiles;
    const uint16_t* np = more_tiles ? weight_row(next) : wp;
    const bool one = units <= kFlight * kWaves;  // a wavefront's whole share is in flight
    floatx4_t acc[2] = {};
    for (int u0 = w; u0 < units; u0 += kFlight * kWaves) {
      if (kPro != kNorm && u0 != w) {
        load_inputs(u0);
        if constexpr (kPro == kGated) gate_inputs(u0);
      }
#pragma unroll
      for (int i = 0; i < kFlight; ++i) {
        const int u = u0 + i * kWaves;
        if (u < units) {
          if constexpr (kPro == kNorm) {
            const uint16_t* hp = h + n * (a.K + 8) + k_lane + 64 * u;
            xr[i][0] = *reinterpret_cast<const u32x4_t*>(hp);
            xr[i][1] = *reinterpret_cast<const u32x4_t*>(hp + 32);
          }
          acc[0] = mfma16(wr[i][0], xr[i][0], acc[0]);
          acc[1] = mfma16(wr[i][1], xr[i][1], acc[1]);
          if (one && more_tiles) load_unit(np, i, u);
        }
      }
      if (!one) {
        const int more = u0 + kFlight * kWaves;
        if (more < units)
          load_weights(wp, more);
        else if (more_tiles)
          load_weights(np, w);
      }
    }
    wp = np;
    // The loop's last MFMAs and these reads are in different blocks.
    mfma_result_barrier(acc);
    // Element i: operand row 4 quad + i, activation column lane % 16.
    float* part = red + (turn & 1) * kWaves * 256;
    *reinterpret_cast<floatx4_t*>(part + (w * 16 + op) * 16 + 4 * quad) = acc[0] + acc[1];
    lds_barrier();
    if (mine) {
      float y = 0.f, up = 0.f;
  #pragma unroll
      for (int v = 0; v < kWaves; ++v) {
        y += part[(v * 16 + row) * 16 + r];
        if constexpr (kForm == kHalves) y += part[(v * 16 + row + 8) * 16 + r + 8];
        if constexpr (kForm == kPairs) up += part[(v * 16 + row) * 16 + r + 8];
      }
      if constexpr (kEpi == kSiluMul) {
        static_cast<uint16_t*>(a.out[0])[at] = uint16_t(bf16_bits(silu(y) * up));
      } else if constexpr (kEpi == kResidual) {
        static_cast<uint16_t*>(a.out[0])[at] = uint16_t(bf16_bits(bf16_lo(before) + y));
      } else if (kEpi == kConv && seg == 0) {
        // This thread owns the channel's state: the oldest input leaves it.
        const uint32_t now = bf16_bits(y);
        const u32x2_t state = {held.x >> 16 | held.y << 16, held.y >> 16 | now << 16};
        *reinterpret_cast<u32x2_t*>(a.conv_state + 4 * at) = state;
        float s = bf16_lo(state.x) * bf16_lo(taps.x);
        s = fmaf(bf16_hi(state.x), bf16_hi(taps.x), s);
        s = fmaf(bf16_lo(state.y), bf16_lo(taps.y), s);
        s = fmaf(bf16_hi(state.y), bf16_hi(taps.y), s);
        static_cast<float*>(a.out[0])[at] = silu(s);
      } else {
        static_cast<uint16_t*>(a.out[seg])[at] = uint16_t(bf16_bits(y));
      }
    }
    if (!more_tiles) break;
    tile = next;
  }
}

// ---------------------------------------------------------- delta rule step
// One token of a value head: its state [DK, DV] is read once (16 bytes of a
// row a lane), k . S and q . S summed together, and written back updated; the
// output o = decay (q . S) + (q . k) d needs no second pass, and its gated norm
// is taken here because the workgroup holds the whole head.
struct StepArgs {
  const float* act;  // [B, C]: silu of the convolution, heads not yet normed
  const uint16_t *a, *b, *a_log, *dt_bias, *z, *norm;
  float* state;
  uint16_t* out;  // [B, hv, DV]
  int hk, hv, has_prev;
  float eps;
};

constexpr int kStepThreads = 512;

template <int DK, int DV>
__global__ void __launch_bounds__(kStepThreads) delta_step_kernel(const StepArgs p) {
  constexpr int CT = DV / 4;               // threads per state row
  constexpr int RG = kStepThreads / CT;    // rows at a time
  constexpr int N = DK / RG;               // rows per thread
  constexpr int EK = DK / 64;
  __shared__ __attribute__((aligned(16))) floatx4_t part[2][8][CT];
  __shared__ float delta[DV], squares[8];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int h = blockIdx.x, kh = h / (p.hv / p.hk);
  const int64_t b = blockIdx.y;
  const float* act = p.act + b * (2 * p.hk * DK + p.hv * DV);
  const float *qp = act + kh * DK, *kp = act + (p.hk + kh) * DK;
  float* sp = p.state + (b * p.hv + h) * DK * DV + 4 * (tid % CT);
  const int r0 = tid / CT;

  floatx4_t s[N];
#pragma unroll
  for (int i = 0; i < N; ++i)
    s[i] = p.has_prev ? *reinterpret_cast<const floatx4_t*>(sp + (r0 + RG * i) * DV) : floatx4_t{};
  float q[N], k[N];
#pragma unroll
  for (int i = 0; i < N; ++i) q[i] = qp[r0 + RG * i], k[i] = kp[r0 + RG * i];
  float sq = 0.f, sk = 0.f, qk = 0.f;
#pragma unroll
  for (int e = 0; e < EK; ++e) {
    const float x = qp[EK * lane + e], y = kp[EK * lane + e];
    sq = fmaf(x, x, sq), sk = fmaf(y, y, sk), qk = fmaf(x, y, qk);
  }
  const float rq = rsqrtf(wave_sum(sq) + 1e-6f) * rsqrtf(float(DK));
  const float rk = rsqrtf(wave_sum(sk) + 1e-6f);
  qk = wave_sum(qk) * rq * rk;
  const float ga = bf16_lo(p.a[b * p.hv + h]) + bf16_lo(p.dt_bias[h]);
  const float soft = ga > 20.f ? ga : log1pf(expf(ga));
  const float decay = expf(-expf(bf16_lo(p.a_log[h])) * soft);
  const float beta = sigmoid(bf16_lo(p.b[b * p.hv + h]));
  const int64_t at = (b * p.hv + h) * DV + min(tid, DV - 1);
  const float v = act[2 * p.hk * DK + h * DV + min(tid, DV - 1)];
  const float weight = bf16_lo(p.norm[min(tid, DV - 1)]), z = bf16_lo(p.z[at]);

  floatx4_t pk = {}, pq = {};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    k[i] *= rk, q[i] *= rq;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pk[e] = fmaf(k[i], s[i][e], pk[e]);
      pq[e] = fmaf(q[i], s[i][e], pq[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if constexpr (CT == 16) {
      pk[e] += xor_lanes<16>(pk[e], lane);
      pq[e] += xor_lanes<16>(pq[e], lane);
    }
    pk[e] += xor_lanes<32>(pk[e], lane);
    pq[e] += xor_lanes<32>(pq[e], lane);
  }
  if (lane < CT) part[0][w][lane] = pk, part[1][w][lane] = pq;
  __syncthreads();
  float o = 0.f;
  if (tid < DV) {
    const float* c = reinterpret_cast<const float*>(&part[0][0][0]) + tid;
    float dk = 0.f, dq = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) dk += c[i * DV], dq += c[(8 + i) * DV];
    const float d = beta * fmaf(-decay, dk, v);
    delta[tid] = d;
    o = fmaf(qk, d, decay * dq);
    const float ss = wave_sum(o * o);
    if (lane == 0) squares[w] = ss;
  }
  __syncthreads();
  const floatx4_t d = *reinterpret_cast<const floatx4_t*>(delta + 4 * (tid % CT));
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[i][e] = fmaf(k[i], d[e], decay * s[i][e]);
    *reinterpret_cast<floatx4_t*>(sp + (r0 + RG * i) * DV) = s[i];
  }
  if (tid < DV) {
    float ss = squares[0];
    if constexpr (DV == 128) ss += squares[1];
    p.out[at] = uint16_t(bf16_bits(o * rsqrtf(ss / DV + p.eps) * weight * silu(z)));
  }
}

constexpr int kMaxLds = 160 * 1024;

// Workgroups that are resident at once: more tiles are walked.
int resident_workgroups() {
  int device = 0, cus = 0;
  if (hipGetDevice(&device) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    return 768;
  return 3 * cus;
}

template <int kPro, int kEpi, int kForm, int kItems, bool kWalk = false>
int launch(TokenArgs& a, const char* what, pd_stream_t stream) {
  constexpr int waves = kPro == kNorm ? kNormWaves : kPlainWaves;
  constexpr int features = kForm == kWide ? 16 : 8;
  const int lds = 2 * waves * 1024 + 128 + (kPro == kNorm ? a.rows * (a.K + 8) * 2 : 0);
  if (lds > kMaxLds) return pd::fail(PD_EINVAL, "%s: the input rows exceed the LDS", what);
  int64_t tiles = 0;
  for (int i = 0; i < a.segments; ++i) tiles += (int64_t(a.m[i]) + features - 1) / features;
  a.tiles = int(tiles);
  const auto kernel = token_kernel<kPro, kEpi, kForm, kItems, kWalk>;
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                          hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds) != hipSuccess)
    return pd::fail(PD_ELAUNCH, "%s: LDS size", what);
  const int grid = kWalk ? std::min(resident_workgroups(), a.tiles) : a.tiles;
  hipLaunchKernelGGL(kernel, dim3(unsigned(grid)), dim3(64 * waves), unsigned(lds),
                     as_stream(stream), a);
  return launch_status(what);
}

template <int kEpi, int kForm, bool kWalk = false>
int launch_normed(TokenArgs& a, const char* what, pd_stream_t stream) {
  if (a.K > 512 * kNormWaves || a.rows > 8)
    return launch<kNorm, kEpi, kForm, 0, kWalk>(a, what, stream);
  if (a.rows == 1) return launch<kNorm, kEpi, kForm, 1, kWalk>(a, what, stream);
  if (a.rows <= 4) return launch<kNorm, kEpi, kForm, 4, kWalk>(a, what, stream);
  return launch<kNorm, kEpi, kForm, 8, kWalk>(a, what, stream);
}

int check_shape(int rows, int K) {
  if (rows < 1 || rows > kMaxRows) return pd::fail(PD_EINVAL, "1 to %d rows", kMaxRows);
  if (K < 64 || K % 64 || K > (1 << 20))
    return pd::fail(PD_EINVAL, "input features must be a multiple of 64");
  return PD_OK;
}

}  // namespace

extern "C" int pd_norm_linears(const void* x, const void* norm, double eps, int32_t rows, int32_t dim,
                               int32_t count, const void* const* weights, const int32_t* features,
                               void* const* outs, const void* taps, void* conv_state,
                               int32_t has_prev, pd_stream_t stream) {
  pd::clear_error();
  if (const int bad = check_shape(rows, dim)) return bad;
  if (count < 1 || count > kMaxSegments)
    return pd::fail(PD_EINVAL, "1 to %d weight matrices", kMaxSegments);
  if (!x || !norm || !weights || !features || !outs || !all_aligned16(x, norm, taps, conv_state) ||
      (taps == nullptr) != (conv_state == nullptr))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  TokenArgs a{};
  for (int i = 0; i < count; ++i) {
    if (!weights[i] || !outs[i] || !all_aligned16(weights[i], outs[i]) || features[i] < 1 ||
        int64_t(features[i]) * kMaxRows > 0x7fffffff)
      return pd::fail(PD_EINVAL, "weights and outputs must be present and 16-byte aligned");
    a.w[i] = u16(weights[i]), a.out[i] = outs[i], a.m[i] = features[i];
  }
  a.x = u16(x), a.norm = u16(norm), a.taps = u16(taps), a.conv_state = u16(conv_state);
  a.segments = count, a.rows = rows, a.K = dim, a.has_prev = has_prev, a.eps = float(eps);
  if (features[0] > 16 * 1024) {
    // Many tiles are walked by the resident workgroups, so that each norms the rows
    // once.  Walked, and with a workgroup a tile: 151936 features of 2048 for 16
    // rows 132 and 249 us, of 256 for one row 18 and 34.  Up to 8 rows of 2048 the
    // norm hides behind the weights and the walk is the slower: 30 and 26 us at
    // 32768 features for one row, 115 and 108 at 151936, 124 and 120 for 8 rows.
    // With few tiles it has nothing to share: 10.5 and 9.6 us at 8192 features of
    // 2048 for one row.
    if (!taps) return launch_normed<kStore, kWide, true>(a, "pd_norm_linears", stream);
  } else if (rows <= 4 && dim % 128 == 0) {
    // 8 features a workgroup spread over the CUs more evenly (8224 features of
    // 2048: 11.4 -> 9.7 us for one row), until the rows' norm, taken by every
    // workgroup, costs more (8 rows: 14.3 and 15.3 us).
    return taps ? launch_normed<kConv, kHalves>(a, "pd_norm_linears", stream)
                : launch_normed<kStore, kHalves>(a, "pd_norm_linears", stream);
  }
  return taps ? launch_normed<kConv, kWide>(a, "pd_norm_linears", stream)
              : launch_normed<kStore, kWide>(a, "pd_norm_linears", stream);
}

extern "C" int pd_norm_gate_up(const void* x, const void* norm, double eps, int32_t rows,
                               int32_t dim, const void* gate, const void* up, void* out,
                               int32_t features, pd_stream_t stream) {
  pd::clear_error();
  if (const int bad = check_shape(rows, dim)) return bad;
  if (!x || !norm || !gate || !up || !out || !all_aligned16(x, norm, gate, up, out) || features < 1)
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  TokenArgs a{};
  a.x = u16(x), a.norm = u16(norm), a.w[0] = u16(gate), a.w[1] = u16(up), a.out[0] = out;
  a.m[0] = features, a.segments = 1, a.rows = rows, a.K = dim, a.eps = float(eps);
  return launch_normed<kSiluMul, kPairs>(a, "pd_norm_gate_up", stream);
}

extern "C" int pd_linear_add(const void* h, const void* gate, int32_t head_dim, const void* weight,
                             void* x, int32_t rows, int32_t dim, int32_t features,
                             pd_stream_t stream) {
  pd::clear_error();
  if (const int bad = check_shape(rows, dim)) return bad;
  if (!h || !weight || !x || !all_aligned16(h, gate, weight, x) || features < 1)
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  if (gate && (!pd::valid_head_dim(head_dim) || dim % head_dim))
    return pd::fail(PD_EINVAL, "gated heads of 64, 128 or 256 that divide the input features");
  TokenArgs a{};
  a.x = u16(h), a.gate = u16(gate), a.head_shift = gate ? __builtin_ctz(unsigned(head_dim)) : 0, a.w[0] = u16(weight), a.out[0] = x;
  a.m[0] = features, a.segments = 1, a.rows = rows, a.K = dim;
  const bool halves = rows <= 8 && dim % 128 == 0;
  if (gate)
    return halves ? launch<kGated, kResidual, kHalves, 1>(a, "pd_linear_add", stream)
                  : launch<kGated, kResidual, kWide, 1>(a, "pd_linear_add", stream);
  return halves ? launch<kPlain, kResidual, kHalves, 1>(a, "pd_linear_add", stream)
                : launch<kPlain, kResidual, kWide, 1>(a, "pd_linear_add", stream);
}

extern "C" int pd_delta_step(const float* act, const void* a, const void* b, const void* a_log,
                             const void* dt_bias, const void* z, const void* norm, double eps,
                             float* state, void* out, int32_t batch, int32_t hk, int32_t hv,
                             int32_t dk, int32_t dv, int32_t has_prev, pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || batch > 65535 || hk < 1 || hv < 1 || hv % hk)
    return pd::fail(PD_EINVAL, "batch and heads must be positive, value heads a multiple");
  if ((dk != 64 && dk != 128) || (dv != 64 && dv != 128))
    return pd::fail(PD_EINVAL, "linear heads of 64 or 128 elements");
  if (!act || !a || !b || !a_log || !dt_bias || !z || !norm || !state || !out ||
      !all_aligned16(act, z, norm, state, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const StepArgs p{act, u16(a), u16(b), u16(a_log), u16(dt_bias), u16(z), u16(norm), state, u16(out),
                   hk, hv, has_prev, float(eps)};
  const dim3 grid{unsigned(hv), unsigned(batch)};
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kStepThreads), 0, as_stream(stream), p);
  };
  if (dk == 64)
    dv == 64 ? go(delta_step_kernel<64, 64>) : go(delta_step_kernel<64, 128>);
  else
    dv == 64 ? go(delta_step_kernel<128, 64>) : go(delta_step_kernel<128, 128>);
  return launch_status("pd_delta_step");
}
