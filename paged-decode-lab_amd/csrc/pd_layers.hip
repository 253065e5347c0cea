// The decoder layer's work between its matrix products, for MI355X (gfx950):
// norms, the gated delta rule with its convolution, rotary embedding with the
// K/V write, and the gates.  Activations are bf16 in memory between products;
// everything inside a kernel is float32.
//
// Each of these was a chain of separate elementwise and reduction launches
// over the same rows; here each reads its inputs once and writes its outputs
// once.  A 24-layer decoder (hidden 2048) on MI355X: a prompt of 512 tokens
// 99.4 -> 7.0 ms, a captured decode step 8.1 -> 2.8 ms.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "pd_device.h"
#include "pd_internal.h"

namespace {

using namespace pdk;

__device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + exp_fast(-x)); }
__device__ __forceinline__ float silu(float x) { return x / (1.f + exp_fast(-x)); }

__device__ __forceinline__ void unpack8(u32x4_t t, float (&x)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) x[2 * i] = bf16_lo(t[i]), x[2 * i + 1] = bf16_hi(t[i]);
}
__device__ __forceinline__ u32x4_t pack8(const float (&x)[8]) {
  u32x4_t t;
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = pack_bf16(x[2 * i], x[2 * i + 1]);
  return t;
}

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
// gate half of the query projection's heads); 8 elements a thread.
template <bool kSigmoid>
__global__ void __launch_bounds__(256)
gate_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
            uint16_t* __restrict__ out, int64_t pieces, int cols, int64_t b_stride) {
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

// -------------------------------------------------- convolution and gates
// Causal depthwise convolution of 4 taps, silu, the unit norm of the query and
// key heads (queries times dk^-1/2), and the delta rule's decay and beta.  A
// wavefront runs kConvSteps tokens of one unit, the three earlier inputs in
// registers: units 0 .. hk - 1 are a key head and its query head, the rest a
// value head and its gates.  Channels: [hk dk queries | hk dk keys | hv dv].
//
// conv_state [B, C, 4] receives the last four inputs; with `has_prev` it holds
// the four before this call, and the call's steps fit one wavefront's, so that
// the wavefront that reads a channel's state is the one that writes it.
constexpr int kConvSteps = 16;

struct ConvArgs {
  const uint16_t *x, *taps, *a, *b, *a_log, *dt_bias;
  uint16_t* conv_state;
  float *act, *gates;  // [B, S, C], [B, S, hv, 2] = (decay, beta)
  int steps, hk, hv, has_prev;
};

template <int E>
struct ConvRun {  // E channels of a lane
  float tap[4][E], x[4][E];

  __device__ __forceinline__ void begin(const ConvArgs& p, int64_t b, int C, int c, int t0) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const u32x2_t w = *reinterpret_cast<const u32x2_t*>(p.taps + 4 * (c + e));
      tap[0][e] = bf16_lo(w.x), tap[1][e] = bf16_hi(w.x);
      tap[2][e] = bf16_lo(w.y), tap[3][e] = bf16_hi(w.y);
    }
#pragma unroll
    for (int j = 1; j < 4; ++j) {
      const int t = t0 - 4 + j;
      if (t >= 0) {
        load_bf16<E>(p.x + (b * p.steps + t) * C + c, x[j]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
          x[j][e] = p.has_prev ? bf16_lo(p.conv_state[(b * C + c + e) * 4 + 4 + t]) : 0.f;
      }
    }
  }
  __device__ __forceinline__ void step(const ConvArgs& p, int64_t row, int C, int c, float (&y)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) x[0][e] = x[1][e], x[1][e] = x[2][e], x[2][e] = x[3][e];
    load_bf16<E>(p.x + row * C + c, x[3]);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) s = fmaf(x[j][e], tap[j][e], s);
      y[e] = silu(s);
    }
  }
  __device__ __forceinline__ void finish(const ConvArgs& p, int64_t b, int C, int c) {
#pragma unroll
    for (int e = 0; e < E; ++e)
      *reinterpret_cast<u32x2_t*>(p.conv_state + (b * C + c + e) * 4) =
          u32x2_t{pack_bf16(x[0][e], x[1][e]), pack_bf16(x[2][e], x[3][e])};
  }
};

__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

template <int DK, int DV>
__global__ void __launch_bounds__(256) conv_gates_kernel(const ConvArgs p) {
  const int lane = threadIdx.x & 63;
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= p.hk + p.hv) return;
  const int t0 = blockIdx.y * kConvSteps, t1 = min(t0 + kConvSteps, p.steps);
  const int64_t b = blockIdx.z;
  const int C = 2 * p.hk * DK + p.hv * DV;
  if (unit < p.hk) {
    constexpr int E = DK / 64;
    const int cq = unit * DK + E * lane, ck = cq + p.hk * DK;
    ConvRun<E> q, k;
    q.begin(p, b, C, cq, t0);
    k.begin(p, b, C, ck, t0);
    for (int t = t0; t < t1; ++t) {
      const int64_t row = b * p.steps + t;
      float yq[E], yk[E], sq = 0.f, sk = 0.f;
      q.step(p, row, C, cq, yq);
      k.step(p, row, C, ck, yk);
#pragma unroll
      for (int e = 0; e < E; ++e) sq = fmaf(yq[e], yq[e], sq), sk = fmaf(yk[e], yk[e], sk);
      const float rq = rsqrtf(wave_sum(sq) + 1e-6f) * rsqrtf(float(DK));
      const float rk = rsqrtf(wave_sum(sk) + 1e-6f);
#pragma unroll
      for (int e = 0; e < E; ++e) yq[e] *= rq, yk[e] *= rk;
      store_f32<E>(p.act + row * C + cq, yq);
      store_f32<E>(p.act + row * C + ck, yk);
    }
    if (t1 == p.steps) {
      q.finish(p, b, C, cq);
      k.finish(p, b, C, ck);
    }
  } else {
    constexpr int E = DV / 64;
    const int h = unit - p.hk, c = 2 * p.hk * DK + h * DV + E * lane;
    ConvRun<E> v;
    v.begin(p, b, C, c, t0);
    for (int t = t0; t < t1; ++t) {
      const int64_t row = b * p.steps + t;
      float y[E];
      v.step(p, row, C, c, y);
      store_f32<E>(p.act + row * C + c, y);
    }
    if (t1 == p.steps) v.finish(p, b, C, c);
    if (t0 + lane < t1) {
      const int64_t at = (b * p.steps + t0 + lane) * p.hv + h;
      const float a = bf16_lo(p.a[at]) + bf16_lo(p.dt_bias[h]);
      const float g = -expf(bf16_lo(p.a_log[h])) * softplus(a);
      *reinterpret_cast<floatx2_t*>(p.gates + 2 * at) =
          floatx2_t{expf(g), sigmoid(bf16_lo(p.b[at]))};
    }
  }
}

// -------------------------------------------------------- gated delta rule
// Per value head and column j of its state S [dk, dv], over the tokens:
//   S_j *= decay;  d = beta (v_j - k . S_j);  S_j += d k;  o_j = q . S_j.
// The columns are independent, so each is one group of L lanes that hold
// DK / L of its elements in registers for the whole sequence; what is serial
// is the chain of a token's dot, its reduction over the L lanes (lane moves)
// and the update.  L = 32 halves the work of a token's chain, L = 16 the total
// work.  A workgroup of two wavefronts stages kDeltaSteps tokens of k, q, v
// and the gates in LDS, the next ones loaded to registers meanwhile.
constexpr int kDeltaSteps = 16;

struct DeltaArgs {
  const float *act, *gates;
  float *state, *out;  // [B, hv, DK, DV], [B, S, hv, DV]
  int steps, hk, hv, has_prev;
};

template <int L>
__device__ __forceinline__ float lanes_sum(float x) {
  const auto ror = [](float v, auto n) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + n.value, 0xF,
                                                      0xF, false));
  };
  x += ror(x, std::integral_constant<int, 8>{});
  x += ror(x, std::integral_constant<int, 4>{});
  x += ror(x, std::integral_constant<int, 2>{});
  x += ror(x, std::integral_constant<int, 1>{});
  if constexpr (L == 32) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
  return x;
}

template <int DK, int DV, int L>
__global__ void __launch_bounds__(128) delta_kernel(const DeltaArgs p) {
  constexpr int T = kDeltaSteps, N = DK / L, P = N / 4;  // elements, 16-byte pieces a lane
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
  floatx2_t fg = {1.f, 0.f};
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
    if (tid < T) gs[buf][tid] = fg;
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
      const float d = g.y * fmaf(-g.x, lanes_sum<L>(d0 + d1), v);
      float o0 = 0.f, o1 = 0.f;
#pragma unroll
      for (int i = 0; i < N; ++i) s[i] = fmaf(k[i / 4][i % 4], d, g.x * s[i]);
#pragma unroll
      for (int i = 0; i < N; i += 2) {
        o0 = fmaf(q[i / 4][i % 4], s[i], o0);
        o1 = fmaf(q[i / 4][i % 4 + 1], s[i + 1], o1);
      }
      const float o = lanes_sum<L>(o0 + o1);
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

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
template <typename... Ts>
bool all_aligned16(Ts... p) { return (aligned16(p) && ...); }

int launch_status(const char* what) {
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    return pd::fail(PD_ELAUNCH, "%s launch failed: %s", what, hipGetErrorString(err));
  return PD_OK;
}

hipStream_t as_stream(pd_stream_t s) { return reinterpret_cast<hipStream_t>(s); }
const uint16_t* u16(const void* p) { return static_cast<const uint16_t*>(p); }
uint16_t* u16(void* p) { return static_cast<uint16_t*>(p); }

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

extern "C" int pd_conv_gates(const void* x, const void* taps, const void* a, const void* b,
                             const void* a_log, const void* dt_bias, void* conv_state, float* act,
                             float* gates, int32_t batch, int32_t steps, int32_t hk, int32_t hv,
                             int32_t dk, int32_t dv, int32_t has_prev, pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || batch > 65535 || steps < 1 || hk < 1 || hv < 1 || hv % hk)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive, value heads a multiple");
  if (!valid_linear_dims(dk, dv)) return pd::fail(PD_EINVAL, "linear heads of 64 or 128 elements");
  if (has_prev && steps > kConvSteps)
    return pd::fail(PD_EINVAL, "at most %d steps continue a state", kConvSteps);
  const int64_t chunks = (int64_t(steps) + kConvSteps - 1) / kConvSteps;
  if (chunks > 65535) return pd::fail(PD_EINVAL, "too many steps");
  if (!x || !taps || !a || !b || !a_log || !dt_bias || !conv_state || !act || !gates ||
      !all_aligned16(x, taps, conv_state, act, gates))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const ConvArgs p{u16(x), u16(taps), u16(a), u16(b), u16(a_log), u16(dt_bias), u16(conv_state),
                   act, gates, steps, hk, hv, has_prev};
  const dim3 grid(unsigned((hk + hv + 3) / 4), unsigned(chunks), unsigned(batch));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, as_stream(stream), p);
  };
  if (dk == 64)
    dv == 64 ? go(conv_gates_kernel<64, 64>) : go(conv_gates_kernel<64, 128>);
  else
    dv == 64 ? go(conv_gates_kernel<128, 64>) : go(conv_gates_kernel<128, 128>);
  return launch_status("pd_conv_gates");
}

extern "C" int pd_delta_rule(const float* act, const float* gates, float* state, float* out,
                             int32_t batch, int32_t steps, int32_t hk, int32_t hv, int32_t dk,
                             int32_t dv, int32_t has_prev, int32_t lanes, pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || batch > 65535 || steps < 1 || hk < 1 || hv < 1 || hv > 65535 || hv % hk)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive, value heads a multiple");
  if (!valid_linear_dims(dk, dv)) return pd::fail(PD_EINVAL, "linear heads of 64 or 128 elements");
  if (!act || !gates || !state || !out || !all_aligned16(act, gates, state, out))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  if (lanes != 16 && (lanes != 32 || dk != 128))
    return pd::fail(PD_EINVAL, "16 lanes a column, or 32 at 128 elements");
  const DeltaArgs p{act, gates, state, out, steps, hk, hv, has_prev};
  const dim3 grid(unsigned(dv * lanes / 128), unsigned(hv), unsigned(batch));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(128), 0, as_stream(stream), p);
  };
  if (dk == 64)
    dv == 64 ? go(delta_kernel<64, 64, 16>) : go(delta_kernel<64, 128, 16>);
  else if (lanes == 16)
    dv == 64 ? go(delta_kernel<128, 64, 16>) : go(delta_kernel<128, 128, 16>);
  else
    dv == 64 ? go(delta_kernel<128, 64, 32>) : go(delta_kernel<128, 128, 32>);
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
