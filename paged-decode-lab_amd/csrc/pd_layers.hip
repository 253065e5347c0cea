// The decoder layer's work between its matrix products, for MI355X (gfx950):
// norms, the gated delta rule with its convolution, rotary embedding with the
// K/V write, and the gates.  Activations are bf16 in memory between products;
// everything inside a kernel is float32.
//
// Each of these was a chain of separate elementwise and reduction launches
// over the same rows; here each reads its inputs once and writes its outputs
// once.  A 24-layer decoder (hidden 2048) on MI355X, these around library
// products: a prompt of 512 tokens 99.4 -> 7.0 ms, a captured decode step 8.1 ->
// 2.8 ms (4.7 and 1.09 with the delta rule in chunks, the products of one round
// and of few rows, all kernels of their own files).
#include <hip/hip_runtime.h>

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

// E consecutive bf16 (E = 1, 2 or 4) at element p.
template <int E>
__device__ __forceinline__ void load_bf16(const uint16_t* p, float (&x)[E]) {
  if constexpr (E == 1) {
    x[0] = bf16_lo(*p);
  } else if constexpr (E == 2) {
    const uint32_t t = *reinterpret_cast<const uint32_t*>(p);
    x[0] = bf16_lo(t), x[1] = bf16_hi(t);
  } else {
    const u32x2_t t = *reinterpret_cast<const u32x2_t*>(p);
    x[0] = bf16_lo(t.x), x[1] = bf16_hi(t.x), x[2] = bf16_lo(t.y), x[3] = bf16_hi(t.y);
  }
}
template <int E>
__device__ __forceinline__ void store_bf16(uint16_t* p, const float (&x)[E]) {
  if constexpr (E == 1)
    *p = uint16_t(bf16_bits(x[0]));
  else if constexpr (E == 2)
    *reinterpret_cast<uint32_t*>(p) = pack_bf16(x[0], x[1]);
  else
    *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])};
}
template <int E>
__device__ __forceinline__ void store_f32(float* p, const float (&x)[E]) {
  if constexpr (E == 1)
    *p = x[0];
  else
#pragma unroll
    for (int i = 0; i < E; i += 2) *reinterpret_cast<floatx2_t*>(p + i) = floatx2_t{x[i], x[i + 1]};
}

// ------------------------------------------------------------------- norms
// x += y (y optional, x rounded to bf16) and h = x rms(x)^-1 (1 + w): one
// workgroup a row, its elements held in registers between the two uses.
constexpr int kNormPieces = 4;  // 16-byte pieces per thread: rows of up to 8192

__global__ void __launch_bounds__(256)
add_rms_kernel(uint16_t* __restrict__ x, const uint16_t* __restrict__ y,
               const uint16_t* __restrict__ w, uint16_t* __restrict__ h, int dim, float eps) {
  __shared__ float sums[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, pieces = dim / 8;
  float v[kNormPieces][8], ss = 0.f;
#pragma unroll
  for (int i = 0; i < kNormPieces; ++i) {
    const int p = tid + 256 * i;
    if (p >= pieces) break;
    unpack8(load16(x + row * dim + 8 * p), v[i]);
    if (y) {
      float t[8];
      unpack8(load16(y + row * dim + 8 * p), t);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] += t[e];
      const u32x4_t sum = pack8(v[i]);
      *reinterpret_cast<u32x4_t*>(x + row * dim + 8 * p) = sum;
      unpack8(sum, v[i]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(v[i][e], v[i][e], ss);
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) sums[tid >> 6] = ss;
  __syncthreads();
  const float r = rsqrtf((sums[0] + sums[1] + sums[2] + sums[3]) / dim + eps);
#pragma unroll
  for (int i = 0; i < kNormPieces; ++i) {
    const int p = tid + 256 * i;
    if (p >= pieces) break;
    float t[8];
    unpack8(load16(w + 8 * p), t);
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = v[i][e] * r * (1.f + t[e]);
    *reinterpret_cast<u32x4_t*>(h + row * dim + 8 * p) = pack8(t);
  }
}

// y = o rms(o)^-1 w silu(z) per head: o float32, z and y bf16, one wavefront a
// (token, head).
template <int D>
__global__ void __launch_bounds__(256)
gated_norm_kernel(const float* __restrict__ o, const uint16_t* __restrict__ z,
                  const uint16_t* __restrict__ w, uint16_t* __restrict__ y, int64_t rows,
                  float eps) {
  constexpr int E = D / 64;
  const int lane = threadIdx.x & 63;
  const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  float v[E], g[E], c[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = o[row * D + E * lane + e];
  load_bf16<E>(z + row * D + E * lane, g);
  load_bf16<E>(w + E * lane, c);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) ss = fmaf(v[e], v[e], ss);
  const float r = rsqrtf(wave_sum(ss) / D + eps);
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = v[e] * r * c[e] * silu(g[e]);
  store_bf16<E>(y + row * D + E * lane, v);
}

// out = silu(a) b (gate and up projections), or with kSigmoid out = a
// sigmoid(b) where b's rows of `cols` are `b_stride` apart (attention and the
// gate half of the query projection's heads); 8 elements a thread.  out may be
// a: a thread has read its elements when it writes them.
template <bool kSigmoid>
__global__ void __launch_bounds__(256)
gate_kernel(const uint16_t* a, const uint16_t* __restrict__ b, uint16_t* out, int64_t pieces,
            int cols, int64_t b_stride) {
  const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (p >= pieces) return;
  float x[8], g[8];
  unpack8(load16(a + 8 * p), x);
  if constexpr (kSigmoid) {
    const int per_row = cols / 8;
    const int64_t r = p / per_row;
    unpack8(load16(b + r * b_stride + 8 * (p - r * per_row)), g);
  } else {
    unpack8(load16(b + 8 * p), g);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = kSigmoid ? x[e] * sigmoid(g[e]) : silu(x[e]) * g[e];
  *reinterpret_cast<u32x4_t*>(out + 8 * p) = pack8(x);
}

// ------------------------------------------------------------- convolution
// Causal depthwise convolution of 4 taps, silu, and the unit norm of the query
// and key heads (queries times dk^-1/2).  Units: 0 .. hk - 1 are a key head and
// its query head, the rest a value head; a wavefront serves one unit.  Lanes
// hold 8 channels of a head (16-byte loads), D / 8 lanes a row, and each lane
// group takes kConvTokens consecutive tokens with the three rows before them,
// all loaded before the first is used.  Channels: [hk dk queries | hk dk keys |
// hv dv].  512 tokens of 6144 channels: 27 us with a token loop per wavefront
// (4-byte loads, two 64-lane sums a token), 8.6 us in this form.
//
// conv_state [B, C, 4] receives the last four inputs; with `has_prev` it holds
// the four before this call, and the call's steps fit one wavefront's, so that
// the wavefront that reads a channel's state is the one that writes it.
constexpr int kConvTokens = 4;

struct ConvArgs {
  const uint16_t *x, *taps;
  uint16_t* conv_state;
  float* act;  // [B, S, C]
  int steps, hk, hv, has_prev;
};

// Sum over the N = 8 or 16 lanes of a group, in every lane, by DPP moves: row
// rotations, or for half rows lane ^ 1, lane ^ 2 and the mirrored half row.
template <int N>
__device__ __forceinline__ float group_sum(float x) {
  const auto dpp = [](float v, auto ctrl) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl.value, 0xF, 0xF, false));
  };
  if constexpr (N == 16) {
    x += dpp(x, std::integral_constant<int, 0x128>{});
    x += dpp(x, std::integral_constant<int, 0x124>{});
    x += dpp(x, std::integral_constant<int, 0x122>{});
    return x + dpp(x, std::integral_constant<int, 0x121>{});
  } else {
    static_assert(N == 8, "lanes of a group");
    x += dpp(x, std::integral_constant<int, 0xB1>{});
    x += dpp(x, std::integral_constant<int, 0x4E>{});
    return x + dpp(x, std::integral_constant<int, 0x141>{});
  }
}

// The convolved rows t0 .. t0 + kConvTokens - 1 of 8 channels from c.
struct ConvRows {
  u32x4_t x[kConvTokens + 3];
  float tap[8][4];

  __device__ __forceinline__ void load(const ConvArgs& p, int64_t b, int C, int c, int t0) {
#pragma unroll
    for (int i = 0; i < kConvTokens + 3; ++i) {
      const int t = t0 - 3 + i;
      x[i] = u32x4_t{};
      if (t >= 0 && t < p.steps) x[i] = load16(p.x + (b * p.steps + t) * C + c);
    }
    u32x4_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = load16(p.taps + 4 * c + 8 * i);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t lo = w[e / 2][2 * (e & 1)], hi = w[e / 2][2 * (e & 1) + 1];
      tap[e][0] = bf16_lo(lo), tap[e][1] = bf16_hi(lo), tap[e][2] = bf16_lo(hi), tap[e][3] = bf16_hi(hi);
    }
    if (p.has_prev && t0 < 3) {  // rows -3 .. -1 are elements 1 .. 3 of the state
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (t0 - 3 + i < 0) {
          uint16_t v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = p.conv_state[(b * C + c + e) * 4 + 4 + (t0 - 3 + i)];
#pragma unroll
          for (int e = 0; e < 4; ++e) x[i][e] = v[2 * e] | uint32_t(v[2 * e + 1]) << 16;
        }
    }
  }
  __device__ __forceinline__ void row(int i, float (&y)[8]) const {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s = fmaf(e & 1 ? bf16_hi(x[i + j][e / 2]) : bf16_lo(x[i + j][e / 2]), tap[e][j], s);
      y[e] = silu(s);
    }
  }
  // The four inputs up to row i as the channels' new state.
  __device__ __forceinline__ void finish(const ConvArgs& p, int64_t b, int C, int c, int i) const {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      u32x4_t s;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const auto at = [&](int j) {
          return k ? x[i + j][e / 2] >> 16 : x[i + j][e / 2] & 0xffffu;
        };
        s[2 * k] = at(0) | at(1) << 16;
        s[2 * k + 1] = at(2) | at(3) << 16;
      }
      *reinterpret_cast<u32x4_t*>(p.conv_state + (b * C + c + e) * 4) = s;
    }
  }
};

template <int DK, int DV>
__global__ void __launch_bounds__(256) conv_kernel(const ConvArgs p) {
  constexpr int kWaveTokens = 64 / (DK / 8) * kConvTokens;  // of a key head's unit
  const int lane = threadIdx.x & 63;
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= p.hk + p.hv) return;
  const int64_t b = blockIdx.z;
  const int C = 2 * p.hk * DK + p.hv * DV;
  const int begin = blockIdx.y * kWaveTokens;
  const auto store = [&](int t, int c, const float (&y)[8]) {
    float* out = p.act + (b * p.steps + t) * C + c;
    *reinterpret_cast<floatx4_t*>(out) = floatx4_t{y[0], y[1], y[2], y[3]};
    *reinterpret_cast<floatx4_t*>(out + 4) = floatx4_t{y[4], y[5], y[6], y[7]};
  };
  if (unit < p.hk) {
    constexpr int L = DK / 8;
    const int cq = unit * DK + 8 * (lane % L), ck = cq + p.hk * DK;
    const int t0 = begin + kConvTokens * (lane / L);
    ConvRows q, k;
    q.load(p, b, C, cq, t0);
    k.load(p, b, C, ck, t0);
#pragma unroll
    for (int i = 0; i < kConvTokens; ++i) {
      float yq[8], yk[8], sq = 0.f, sk = 0.f;
      q.row(i, yq);
      k.row(i, yk);
#pragma unroll
      for (int e = 0; e < 8; ++e) sq = fmaf(yq[e], yq[e], sq), sk = fmaf(yk[e], yk[e], sk);
      const float rq = rsqrtf(group_sum<L>(sq) + 1e-6f) * rsqrtf(float(DK));
      const float rk = rsqrtf(group_sum<L>(sk) + 1e-6f);
#pragma unroll
      for (int e = 0; e < 8; ++e) yq[e] *= rq, yk[e] *= rk;
      if (t0 + i < p.steps) {
        store(t0 + i, cq, yq);
        store(t0 + i, ck, yk);
      }
      if (t0 + i == p.steps - 1) {
        q.finish(p, b, C, cq, i);
        k.finish(p, b, C, ck, i);
      }
    }
  } else {
    // A value head's tokens of this block, in as many passes as its lane
    // groups need.
    constexpr int L = DV / 8, kPass = 64 / L * kConvTokens;
    const int c = 2 * p.hk * DK + (unit - p.hk) * DV + 8 * (lane % L);
    for (int t = begin; t < begin + kWaveTokens; t += kPass) {
      const int t0 = t + kConvTokens * (lane / L);
      ConvRows v;
      v.load(p, b, C, c, t0);
#pragma unroll
      for (int i = 0; i < kConvTokens; ++i) {
        float y[8];
        v.row(i, y);
        if (t0 + i < min(p.steps, begin + kWaveTokens)) store(t0 + i, c, y);
        if (t0 + i == p.steps - 1 && t0 + i < begin + kWaveTokens) v.finish(p, b, C, c, i);
      }
    }
  }
}

// ------------------------------------------------------------------- gates
// (log decay, beta) = (-exp(a_log) softplus(h wa + dt_bias), sigmoid(h wb)) of
// every token and value head: two products of few output features, 16 tokens a
// workgroup, whose wavefronts split K in units of 64 elements (weights the row
// operand, tokens the column operand).  Two library products took 21 us at 512
// tokens of 2048, 7.3 us here.
constexpr int kGateWaves = 8;

__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

__global__ void __launch_bounds__(64 * kGateWaves)
gates_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ wa,
             const uint16_t* __restrict__ wb, const uint16_t* __restrict__ a_log,
             const uint16_t* __restrict__ dt_bias, float* __restrict__ gates, int64_t rows, int K,
             int hv) {
  __shared__ __attribute__((aligned(16))) float part[2][kGateWaves][16][16];
  const int tid = threadIdx.x, lane = tid & 63, op = lane & 15, quad = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t r0 = int64_t(blockIdx.x) * 16;
  const int f0 = blockIdx.y * 16;
  const int64_t feature = int64_t(min(f0 + op, hv - 1)) * K + 8 * quad;
  const uint16_t* x = h + min(r0 + op, rows - 1) * K + 8 * quad;
  floatx4_t acc[2] = {};
#pragma unroll 4
  for (int k = 64 * w; k < K; k += 64 * kGateWaves) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const u32x4_t xv = load16(x + k + 32 * s);
      acc[0] = mfma16(load16(wa + feature + k + 32 * s), xv, acc[0]);
      acc[1] = mfma16(load16(wb + feature + k + 32 * s), xv, acc[1]);
    }
  }
  mfma_result_barrier(acc);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    *reinterpret_cast<floatx4_t*>(&part[i][w][op][4 * quad]) = acc[i];
  __syncthreads();
  const int f = tid & 15, row = tid >> 4;
  if (tid >= 256 || f0 + f >= hv || r0 + row >= rows) return;
  float a = 0.f, b = 0.f;
#pragma unroll
  for (int v = 0; v < kGateWaves; ++v) a += part[0][v][row][f], b += part[1][v][row][f];
  const float g = -expf(bf16_lo(a_log[f0 + f])) * softplus(a + bf16_lo(dt_bias[f0 + f]));
  *reinterpret_cast<floatx2_t*>(gates + ((r0 + row) * hv + f0 + f) * 2) = floatx2_t{g, sigmoid(b)};
}

// -------------------------------------------------------- gated delta rule
// Per value head and column j of its state S [dk, dv], over the tokens:
//   S_j *= decay;  d = beta (v_j - k . S_j);  S_j += d k;  o_j = q . S_j.
// The columns are independent, so each is one group of 16 lanes that hold
// DK / 16 of its elements in registers for the whole sequence; what is serial
// is the chain of a token's dot, its reduction over the 16 lanes (lane moves)
// and the update, 174 ns a token (32 lanes a column: no faster with one
// sequence, a third slower with eight).  For few tokens; more run in chunks
// (pd_delta_chunks).  A workgroup of two wavefronts stages kDeltaSteps tokens of k, q, v
// and the gates in LDS, the next ones loaded to registers meanwhile.
constexpr int kDeltaSteps = 16;

struct DeltaArgs {
  const float *act, *gates;
  float *state, *out;  // [B, hv, DK, DV], [B, S, hv, DV]
  int steps, hk, hv, has_prev;
};

template <int DK, int DV>
__global__ void __launch_bounds__(128) delta_kernel(const DeltaArgs p) {
  constexpr int L = 16, T = kDeltaSteps, N = DK / L, P = N / 4;  // elements, 16-byte pieces a lane
  constexpr int kCols = 128 / L;                         // columns per workgroup
  constexpr int kRowLoads = 2 * T * DK / 4 / 128;        // 16-byte pieces of q and k per thread
  static_assert(N % 4 == 0 && kCols * T <= 128, "one v element per thread");
  __shared__ __attribute__((aligned(16))) float qk[2][2][T][DK];
  __shared__ float vs[2][T][kCols];
  __shared__ floatx2_t gs[2][T];
  const int tid = threadIdx.x, lane = tid & 63, sub = lane % L;
  const int col = tid / L, c0 = blockIdx.x * kCols;
  const int h = blockIdx.y, kh = h / (p.hv / p.hk);
  const int64_t b = blockIdx.z;
  const int C = 2 * p.hk * DK + p.hv * DV;
  const float* base = p.act + b * p.steps * C;
  const int vcol = 2 * p.hk * DK + h * DV + c0;

  // Element 4 i + e of a lane is row 4 L i + 4 sub + e of the state, so that a
  // group's 16-byte reads of k and q are consecutive.
  float s[N];
  float* sp = p.state + ((b * p.hv + h) * DK + 4 * sub) * DV + c0 + col;
#pragma unroll
  for (int i = 0; i < N; ++i) s[i] = p.has_prev ? sp[(4 * L * (i / 4) + i % 4) * DV] : 0.f;

  floatx4_t fq[kRowLoads];
  float fv = 0.f;
  floatx2_t fg = {0.f, 0.f};
  const auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i) {
      const int idx = 128 * i + tid, which = idx / (T * DK / 4), r = idx % (T * DK / 4);
      const int t = min(t0 + r / (DK / 4), p.steps - 1);
      fq[i] = *reinterpret_cast<const floatx4_t*>(base + int64_t(t) * C + (which * p.hk + kh) * DK +
                                                  4 * (r % (DK / 4)));
    }
    if (tid < T * kCols) fv = base[int64_t(min(t0 + tid / kCols, p.steps - 1)) * C + vcol + tid % kCols];
    if (tid < T)
      fg = *reinterpret_cast<const floatx2_t*>(
          p.gates + ((b * p.steps + min(t0 + tid, p.steps - 1)) * p.hv + h) * 2);
  };
  const auto place = [&](int buf) {
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i)
      *reinterpret_cast<floatx4_t*>(&qk[buf][0][0][0] + 4 * (128 * i + tid)) = fq[i];
    if (tid < T * kCols) (&vs[buf][0][0])[tid] = fv;
    if (tid < T) gs[buf][tid] = floatx2_t{expf(fg.x), fg.y};
  };

  fetch(0);
  place(0);
  for (int t0 = 0; t0 < p.steps; t0 += T) {
    const int buf = (t0 / T) & 1;
    __syncthreads();
    if (t0 + T < p.steps) fetch(t0 + T);
    const int n = min(T, p.steps - t0);
    float keep = 0.f;
    const auto token = [&](int t) {
      floatx4_t k[P], q[P];
#pragma unroll
      for (int i = 0; i < P; ++i) {
        q[i] = *reinterpret_cast<const floatx4_t*>(&qk[buf][0][t][4 * L * i + 4 * sub]);
        k[i] = *reinterpret_cast<const floatx4_t*>(&qk[buf][1][t][4 * L * i + 4 * sub]);
      }
      const floatx2_t g = gs[buf][t];
      const float v = vs[buf][t][col];
      float d0 = 0.f, d1 = 0.f;
#pragma unroll
      for (int i = 0; i < N; i += 2) {
        d0 = fmaf(k[i / 4][i % 4], s[i], d0);
        d1 = fmaf(k[i / 4][i % 4 + 1], s[i + 1], d1);
      }
      const float d = g.y * fmaf(-g.x, group_sum<L>(d0 + d1), v);
      float o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int i = 0; i < N; ++i) s[i] = fmaf(k[i / 4][i % 4], d, g.x * s[i]);
#pragma unroll
      for (int i = 0; i < N; i += 2) {
        o0 = fmaf(q[i / 4][i % 4], s[i], o0);
        o1 = fmaf(q[i / 4][i % 4 + 1], s[i + 1], o1);
      }
      const float o = group_sum<L>(o0 + o1);
      if (sub == t) keep = o;
    };
    if (n == T) {
#pragma unroll
      for (int t = 0; t < T; ++t) token(t);
    } else {
      for (int t = 0; t < n; ++t) token(t);
    }
    if (sub < n)
      p.out[((b * p.steps + t0 + sub) * p.hv + h) * DV + c0 + col] = keep;
    if (t0 + T < p.steps) place(buf ^ 1);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) sp[(4 * L * (i / 4) + i % 4) * DV] = s[i];
}

// --------------------------------------------- rotary embedding, K/V write
// cos and sin of position x inverse frequency, float2 [steps, half].  The
// angle is reduced in float64: a float32 product is off by 1e-3 at 32768.
template <bool kBf16>
__global__ void __launch_bounds__(256)
rope_table_kernel(const int64_t* __restrict__ positions, const void* __restrict__ inv_freq,
                  floatx2_t* __restrict__ table, int64_t total, int half) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int j = int(i % half);
  const float f = kBf16 ? bf16_lo(static_cast<const uint16_t*>(inv_freq)[j])
                        : static_cast<const float*>(inv_freq)[j];
  constexpr double kTwoPi = 6.283185307179586476925;
  double angle = double(positions[i / half]) * double(f);
  angle -= rint(angle / kTwoPi) * kTwoPi;
  float s, c;
  sincosf(float(angle), &s, &c);
  table[i] = floatx2_t{c, s};
}

struct QkArgs {
  const uint16_t *q, *k, *v, *wq, *wk;  // [N, Hq, 2D] (query | gate), [N, Hkv, D]
  const floatx2_t* rope;
  uint16_t *q_out, *k_out, *k_pages, *v_pages;  // [N, Hq, D], [N, Hkv, D] or null
  const int32_t* table;
  const int64_t* positions;
  int64_t num_pages, tsb, rows;
  int width, steps, hq, hkv, half;
  float eps;
};

// Per token: query and key heads normed (times 1 + w) and rotated, keys and
// values written to their page slots (as store_pages_kernel: rows without a
// valid page are skipped).  One wavefront a head; partners of a rotation meet
// in LDS.
template <int D>
__global__ void __launch_bounds__(256) qk_rope_kernel(const QkArgs p) {
  constexpr int E = D / 64;
  __shared__ float rows[4][D];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int heads = p.hq + 2 * p.hkv;
  const int64_t id = int64_t(blockIdx.x) * 4 + w;
  if (id >= p.rows * heads) return;
  const int64_t n = id / heads;
  const int h = int(id - n * heads);
  const int step = int(n % p.steps);
  const int64_t b = n / p.steps;
  uint16_t *kp = nullptr, *vp = nullptr;
  if (h >= p.hq) {
    const int64_t pos = p.positions[step];
    if (pos >= 0 && (pos >> 8) < p.width) {
      const int32_t page = p.table[b * p.tsb + (pos >> 8)];
      if (page >= 0 && page < p.num_pages) {
        const int64_t at = (int64_t(page) * 256 + (pos & 255)) * p.hkv * D;
        kp = p.k_pages + at, vp = p.v_pages + at;
      }
    }
  }
  if (h >= p.hq + p.hkv) {
    const int64_t hv = h - p.hq - p.hkv;
    float x[E];
    load_bf16<E>(p.v + (n * p.hkv + hv) * D + E * lane, x);
    if (vp) store_bf16<E>(vp + hv * D + E * lane, x);
    return;
  }
  const bool query = h < p.hq;
  const int64_t hk = h - p.hq;
  float x[E], g[E];
  load_bf16<E>(query ? p.q + (n * p.hq + h) * 2 * D + E * lane
                     : p.k + (n * p.hkv + hk) * D + E * lane, x);
  load_bf16<E>((query ? p.wq : p.wk) + E * lane, g);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) ss = fmaf(x[e], x[e], ss);
  const float r = rsqrtf(wave_sum(ss) / D + p.eps);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    x[e] = x[e] * r * (1.f + g[e]);
    rows[w][E * lane + e] = x[e];
  }
  // A wavefront's own LDS writes are visible to it in order.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = E * lane + e;
    if (i < 2 * p.half) {
      const floatx2_t cs = p.rope[int64_t(step) * p.half + i % p.half];
      x[e] = i < p.half ? x[e] * cs.x - rows[w][i + p.half] * cs.y
                        : x[e] * cs.x + rows[w][i - p.half] * cs.y;
    }
  }
  if (query) {
    store_bf16<E>(p.q_out + (n * p.hq + h) * D + E * lane, x);
  } else {
    if (p.k_out) store_bf16<E>(p.k_out + (n * p.hkv + hk) * D + E * lane, x);
    if (kp) store_bf16<E>(kp + hk * D + E * lane, x);
  }
}

bool valid_linear_dims(int dk, int dv) {
  return (dk == 64 || dk == 128) && (dv == 64 || dv == 128);
}

}  // namespace

extern "C" int pd_add_rms_norm(void* x, const void* y, const void* weight, void* out, int64_t rows,
                               int32_t dim, double eps, pd_stream_t stream) {
  pd::clear_error();
  if (rows < 0 || rows > 0x7fffffff || dim < 8 || dim % 8 || dim > 2048 * kNormPieces)
    return pd::fail(PD_EINVAL, "rows of 8 to %d elements, a multiple of 8", 2048 * kNormPieces);
  if (rows == 0) return PD_OK;
  if (!x || !weight || !out || !all_aligned16(x, y, weight, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  hipLaunchKernelGGL(add_rms_kernel, dim3(unsigned(rows)), dim3(256), 0, as_stream(stream), u16(x),
                     u16(y), u16(weight), u16(out), dim, float(eps));
  return launch_status("pd_add_rms_norm");
}

extern "C" int pd_gated_norm(const float* o, const void* z, const void* weight, void* out,
                             int64_t rows, int32_t dim, double eps, pd_stream_t stream) {
  pd::clear_error();
  if (rows < 0 || rows > int64_t(0x7fffffff)) return pd::fail(PD_EINVAL, "row count out of range");
  if (dim != 64 && dim != 128) return pd::fail(PD_EINVAL, "value heads of 64 or 128 elements");
  if (rows == 0) return PD_OK;
  if (!o || !z || !weight || !out || !all_aligned16(o, z, weight, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const dim3 grid(unsigned((rows + 3) / 4));
  if (dim == 64)
    hipLaunchKernelGGL(gated_norm_kernel<64>, grid, dim3(256), 0, as_stream(stream), o, u16(z),
                       u16(weight), u16(out), rows, float(eps));
  else
    hipLaunchKernelGGL(gated_norm_kernel<128>, grid, dim3(256), 0, as_stream(stream), o, u16(z),
                       u16(weight), u16(out), rows, float(eps));
  return launch_status("pd_gated_norm");
}

extern "C" int pd_silu_mul(const void* gate, const void* up, void* out, int64_t elems,
                           pd_stream_t stream) {
  pd::clear_error();
  if (elems < 0 || elems % 8 || elems / 8 / 256 > 0x7ffffffe)
    return pd::fail(PD_EINVAL, "element count must be a multiple of 8");
  if (elems == 0) return PD_OK;
  if (!gate || !up || !out || !all_aligned16(gate, up, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const int64_t pieces = elems / 8;
  hipLaunchKernelGGL(gate_kernel<false>, dim3(unsigned((pieces + 255) / 256)), dim3(256), 0,
                     as_stream(stream), u16(gate), u16(up), u16(out), pieces, 8, int64_t(0));
  return launch_status("pd_silu_mul");
}

extern "C" int pd_sigmoid_gate(const void* x, const void* gate, int64_t gate_stride, void* out,
                               int64_t rows, int32_t cols, pd_stream_t stream) {
  pd::clear_error();
  if (rows < 0 || cols < 8 || cols % 8 || gate_stride % 8 || gate_stride < cols ||
      rows * (cols / 8) / 256 > 0x7ffffffe)
    return pd::fail(PD_EINVAL, "columns and the gate's row stride must be multiples of 8");
  if (rows == 0) return PD_OK;
  if (!x || !gate || !out || !all_aligned16(x, gate, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const int64_t pieces = rows * (cols / 8);
  hipLaunchKernelGGL(gate_kernel<true>, dim3(unsigned((pieces + 255) / 256)), dim3(256), 0,
                     as_stream(stream), u16(x), u16(gate), u16(out), pieces, cols, gate_stride);
  return launch_status("pd_sigmoid_gate");
}

extern "C" int pd_conv(const void* x, const void* taps, void* conv_state, float* act, int32_t batch,
                       int32_t steps, int32_t hk, int32_t hv, int32_t dk, int32_t dv,
                       int32_t has_prev, pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || batch > 65535 || steps < 1 || hk < 1 || hv < 1 || hv % hk)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive, value heads a multiple");
  if (!valid_linear_dims(dk, dv)) return pd::fail(PD_EINVAL, "linear heads of 64 or 128 elements");
  const int tokens = 64 / (dk / 8) * kConvTokens;  // of a wavefront
  if (has_prev && steps > 16)
    return pd::fail(PD_EINVAL, "at most 16 steps continue a state");
  const int64_t chunks = (int64_t(steps) + tokens - 1) / tokens;
  if (chunks > 65535) return pd::fail(PD_EINVAL, "too many steps");
  if (!x || !taps || !conv_state || !act || !all_aligned16(x, taps, conv_state, act))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const ConvArgs p{u16(x), u16(taps), u16(conv_state), act, steps, hk, hv, has_prev};
  const dim3 grid(unsigned((hk + hv + 3) / 4), unsigned(chunks), unsigned(batch));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, as_stream(stream), p);
  };
  if (dk == 64)
    dv == 64 ? go(conv_kernel<64, 64>) : go(conv_kernel<64, 128>);
  else
    dv == 64 ? go(conv_kernel<128, 64>) : go(conv_kernel<128, 128>);
  return launch_status("pd_conv");
}

extern "C" int pd_gates(const void* h, const void* wa, const void* wb, const void* a_log,
                        const void* dt_bias, float* gates, int64_t rows, int32_t dim, int32_t hv,
                        pd_stream_t stream) {
  pd::clear_error();
  if (rows < 0 || rows > 0x7fffffff || hv < 1 || hv > 16 * 65535 || dim < 64 || dim % 64)
    return pd::fail(PD_EINVAL, "input features must be a multiple of 64");
  if (rows == 0) return PD_OK;
  if (!h || !wa || !wb || !a_log || !dt_bias || !gates || !all_aligned16(h, wa, wb, gates))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const dim3 grid(unsigned((rows + 15) / 16), unsigned((hv + 15) / 16));
  hipLaunchKernelGGL(gates_kernel, grid, dim3(64 * kGateWaves), 0, as_stream(stream), u16(h), u16(wa),
                     u16(wb), u16(a_log), u16(dt_bias), gates, rows, dim, hv);
  return launch_status("pd_gates");
}

extern "C" int pd_delta_rule(const float* act, const float* gates, float* state, float* out,
                             int32_t batch, int32_t steps, int32_t hk, int32_t hv, int32_t dk,
                             int32_t dv, int32_t has_prev, pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || batch > 65535 || steps < 1 || hk < 1 || hv < 1 || hv > 65535 || hv % hk)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive, value heads a multiple");
  if (!valid_linear_dims(dk, dv)) return pd::fail(PD_EINVAL, "linear heads of 64 or 128 elements");
  if (!act || !gates || !state || !out || !all_aligned16(act, gates, state, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const DeltaArgs p{act, gates, state, out, steps, hk, hv, has_prev};
  const dim3 grid(unsigned(dv / 8), unsigned(hv), unsigned(batch));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(128), 0, as_stream(stream), p);
  };
  if (dk == 64)
    dv == 64 ? go(delta_kernel<64, 64>) : go(delta_kernel<64, 128>);
  else
    dv == 64 ? go(delta_kernel<128, 64>) : go(delta_kernel<128, 128>);
  return launch_status("pd_delta_rule");
}

extern "C" int pd_rope_table(const int64_t* positions, const void* inv_freq, int32_t is_bf16,
                             float* table, int32_t steps, int32_t half, pd_stream_t stream) {
  pd::clear_error();
  if (steps < 1 || half < 1) return pd::fail(PD_EINVAL, "steps and frequencies must be positive");
  if (!positions || !inv_freq || !table) return pd::fail(PD_EINVAL, "null tensor pointer");
  const int64_t total = int64_t(steps) * half;
  const dim3 grid(unsigned((total + 255) / 256));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, as_stream(stream), positions, inv_freq,
                       reinterpret_cast<floatx2_t*>(table), total, half);
  };
  is_bf16 ? go(rope_table_kernel<true>) : go(rope_table_kernel<false>);
  return launch_status("pd_rope_table");
}

extern "C" int pd_qk_rope(const void* q, const void* k, const void* v, const void* q_weight,
                          const void* k_weight, const float* rope, void* q_out, void* k_out,
                          void* k_pages, void* v_pages, int64_t num_pages, const int32_t* table,
                          int64_t table_stride_b, int32_t table_width, const int64_t* positions,
                          int32_t batch, int32_t steps, int32_t num_heads, int32_t num_kv_heads,
                          int32_t head_dim, int32_t half, double eps, pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || steps < 1 || num_heads < 1 || num_kv_heads < 1)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive");
  if (!pd::valid_head_dim(head_dim))
    return pd::fail(PD_EINVAL, "custom decode supports head_dim 64, 128, or 256");
  if (half < 1 || 2 * half > head_dim)
    return pd::fail(PD_EINVAL, "rotated dims must lie in [2, head_dim]");
  if (table_width < 1 || num_pages < 1) return pd::fail(PD_EINVAL, "empty table or page pool");
  if (!q || !k || !v || !q_weight || !k_weight || !rope || !q_out || !k_pages || !v_pages ||
      !table || !positions ||
      !all_aligned16(q, k, v, q_weight, k_weight, rope, q_out, k_out, k_pages, v_pages))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  QkArgs p;
  p.q = u16(q), p.k = u16(k), p.v = u16(v), p.wq = u16(q_weight), p.wk = u16(k_weight);
  p.rope = reinterpret_cast<const floatx2_t*>(rope);
  p.q_out = u16(q_out), p.k_out = u16(k_out), p.k_pages = u16(k_pages), p.v_pages = u16(v_pages);
  p.table = table, p.positions = positions;
  p.num_pages = num_pages, p.tsb = table_stride_b, p.rows = int64_t(batch) * steps;
  p.width = table_width, p.steps = steps, p.hq = num_heads, p.hkv = num_kv_heads, p.half = half;
  p.eps = float(eps);
  const int64_t waves = p.rows * (num_heads + 2 * num_kv_heads);
  if ((waves + 3) / 4 > 0x7fffffff)
    return pd::fail(PD_EINVAL, "grid dimension exceeds device limits");
  const dim3 grid(unsigned((waves + 3) / 4));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, as_stream(stream), p);
  };
  if (head_dim == 64)
    go(qk_rope_kernel<64>);
  else if (head_dim == 128)
    go(qk_rope_kernel<128>);
  else
    go(qk_rope_kernel<256>);
  return launch_status("pd_qk_rope");
}
