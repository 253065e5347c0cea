// The gated delta rule over many tokens, in chunks of 64, for MI355X (gfx950).
//
// The recurrence (per value head, state S [dk, dv])
//   S_t = a_t S_{t-1} + k_t u_t^T,   u_t = beta_t (v_t - a_t S_{t-1}^T k_t),
//   o_t = S_t^T q_t
// taken one token at a time is a serial chain of a dot, a reduction and an
// update per token (174 ns each on MI355X).  With G_t the product of the
// chunk's decays up to t, the u of a chunk solve a unit lower triangular
// system in the state before it (the WY form of a product of Householder-like
// factors; Yang et al., "Gated Delta Networks", 2024):
//   (I + A) U = beta V - (beta G K) S,   A_ti = beta_t (G_t / G_i) (k_t . k_i), i < t
//   O = (G Q) S + M U,                   M_ti = (G_t / G_i) (q_t . k_i), i <= t
//   S' = G_C S + K~^T U,                 K~_t = (G_C / G_t) k_t
// chunk_prepare_kernel solves for U0 = (I + A)^-1 beta V and W = (I + A)^-1
// beta G K of every chunk at once; what is left in sequence are four matrix
// products a chunk, whose columns of dv are independent: chunk_scan_kernel
// runs 16 of them a workgroup.
//
// Measured on MI355X, 16 heads of 128 x 128, against the recurrence: 20 and 14
// us for 64 tokens, 23 and 24 for 128, 44 and 88 for 512 (prepare 18, scan
// 26), 153 and 336 for 2049; eight sequences of 64 37 and 42, of 96 51 and 60,
// of 384 139 and 213.
//
// Everything is float32, products included (16x16x4 MFMAs, 64 flops a clock
// and SIMD: what bounds both kernels).  Ratios of decays are exponentials of
// differences of float64 sums of log decays, never quotients, so no chunk
// over- or underflows.
//
// Layout.  A product's row operand holds 16 bytes a lane: lane (r = L % 16, g =
// L / 16) has elements 16 b + 4 g .. + 3 of row r, and the four MFMAs of block b
// contract elements {4 g + e} of it.  The workspace keeps each 16 x 16 operand
// tile in lane order, 1 KB a wavefront's load: loads of 16 rows x 64 bytes
// instead held a CU to half the rate, and the scan to 4.6 us a chunk where its
// products take 2.3.  The column operand then wants
// element 4 g + e of the contraction in lane group g, which is how a result
// holds its rows: the state, U and the solve's intermediate columns go from one
// product into the next without moving.
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

constexpr int kChunk = 64;
static_assert(kChunk == 64, "four 16-token tiles");
constexpr int kPrepareThreads = 512;

struct ChunkArgs {
  const float *act, *gates;  // [B, S, C], [B, S, hv, 2] = (log decay, beta)
  // Operand tiles per (b, value head, chunk): -W and G Q [4 token tiles][DK /
  // 16], M [4][4], K~ and U0 transposed [DK / 16][4] and [DV / 16][4]; G_C.
  float *w, *q, *m, *k, *u, *total;
  float *state, *out;        // [B, hv, DK, DV], [B, S, hv, DV]
  int steps, hk, hv, chunks, has_prev;
};

__device__ __forceinline__ floatx4_t load4(const float* p) {
  return *reinterpret_cast<const floatx4_t*>(p);
}
__device__ __forceinline__ void store4(float* p, floatx4_t x) {
  *reinterpret_cast<floatx4_t*>(p) = x;
}
// acc += A B for 16 elements of the contraction.
__device__ __forceinline__ floatx4_t mfma4(floatx4_t a, floatx4_t b, floatx4_t acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
  return acc;
}

// The chunk's q, k, v and gates are loaded once, at the start, whole rows at a
// time; k and q pass through LDS to become row operands, v takes q's place
// there for its columns.
template <int DK, int DV>
__global__ void __launch_bounds__(kPrepareThreads) chunk_prepare_kernel(const ChunkArgs p) {
  constexpr int KB = DK / 16, VB = DV / 16, kWaves = kPrepareThreads / 64;
  constexpr int kPitch = (DK > DV ? DK : DV) + 4;
  constexpr int kLoadsK = kChunk * DK / 4 / kPrepareThreads;
  constexpr int kLoadsV = kChunk * DV / 4 / kPrepareThreads;
  __shared__ double sum[kChunk];  // log G
  __shared__ float beta[kChunk];
  __shared__ __attribute__((aligned(16))) float kl[kChunk][kPitch], ql[kChunk][kPitch];
  __shared__ __attribute__((aligned(16))) float a[kChunk][kChunk + 4];  // -A
  __shared__ __attribute__((aligned(16))) float inv[4][16][20];  // of I + A's 16 x 16 blocks
  __shared__ __attribute__((aligned(16))) float turn[kWaves][16][20];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chunk = blockIdx.y, h = blockIdx.x, kh = h / (p.hv / p.hk);
  const int64_t b = blockIdx.z, slot = (b * p.hv + h) * p.chunks + chunk;
  const int C = 2 * p.hk * DK + p.hv * DV, t0 = chunk * kChunk, n = min(kChunk, p.steps - t0);
  const float* act = p.act + (b * p.steps + t0) * C;
  const float *qs = act + kh * DK, *ks = act + (p.hk + kh) * DK, *vs = act + 2 * p.hk * DK + h * DV;

  // Tokens past the end neither decay nor write: their rows and gates are 0.
  floatx2_t gate = {0.f, 0.f};
  if (wave == 0 && lane < n)
    gate = *reinterpret_cast<const floatx2_t*>(p.gates + ((b * p.steps + t0 + lane) * p.hv + h) * 2);
  floatx4_t kv[kLoadsK], qv[kLoadsK], vv[kLoadsV];
  const auto rows_of = [&](const float* src, int D, int i) {
    const int at = kPrepareThreads * i + tid, t = at / (D / 4);
    return t < n ? load4(src + int64_t(t) * C + 4 * (at % (D / 4))) : floatx4_t{};
  };
#pragma unroll
  for (int i = 0; i < kLoadsK; ++i) kv[i] = rows_of(ks, DK, i);
#pragma unroll
  for (int i = 0; i < kLoadsK; ++i) qv[i] = rows_of(qs, DK, i);
#pragma unroll
  for (int i = 0; i < kLoadsV; ++i) vv[i] = rows_of(vs, DV, i);
  if (wave == 0) {
    // exp(-128) is 0 in float32: a stronger decay is no different, and sums
    // stay small enough for their differences to keep every bit that counts.
    double s = gate.x < -128.f ? -128.f : gate.x;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const double up = __shfl_up(s, d);
      if (lane >= d) s += up;
    }
    sum[lane] = s;
    beta[lane] = gate.y;
    if (lane == 63) p.total[slot] = expf(float(s));
  }
  const auto put = [&](float (*dst)[kPitch], int D, int i, floatx4_t x) {
    const int at = kPrepareThreads * i + tid;
    store4(&dst[at / (D / 4)][4 * (at % (D / 4))], x);
  };
#pragma unroll
  for (int i = 0; i < kLoadsK; ++i) put(kl, DK, i, kv[i]), put(ql, DK, i, qv[i]);
  __syncthreads();

  // A result tile's rows 4 g + e of column r, as the row operand of a later
  // product: element r of rows 4 g + e.  Through this wavefront's own LDS tile,
  // whose accesses are in order.
  const auto as_rows = [&](floatx4_t x) {
#pragma unroll
    for (int e = 0; e < 4; ++e) turn[wave][4 * g + e][r] = x[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const floatx4_t y = load4(&turn[wave][r][4 * g]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return y;
  };
  // G Q: eight wavefronts, half of a token tile's blocks each.
#pragma unroll
  for (int i = 0; i < KB / 2; ++i) {
    const int tile = wave / 2, block = wave % 2 * (KB / 2) + i;
    const float gt = expf(float(sum[16 * tile + r]));
    store4(p.q + (((slot * 4 + tile) * KB + block) * 64 + lane) * 4,
           load4(&ql[16 * tile + r][16 * block + 4 * g]) * gt);
  }
  // -A and M: the ten tiles on and below the diagonal, one a wavefront and two
  // for the first ones.
  for (int pair = wave; pair < 10; pair += kWaves) {
    const int ti = pair < 1 ? 0 : pair < 3 ? 1 : pair < 6 ? 2 : 3, tj = pair - ti * (ti + 1) / 2;
    floatx4_t kk[2] = {}, qk[2] = {};
    const int row = 16 * ti + r, other = 16 * tj + r;
#pragma unroll
    for (int i = 0; i < KB; i += 2) {
      floatx4_t ka[2], qa[2], kb[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        ka[j] = load4(&kl[row][16 * (i + j) + 4 * g]);
        qa[j] = load4(&ql[row][16 * (i + j) + 4 * g]);
        kb[j] = load4(&kl[other][16 * (i + j) + 4 * g]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          kk[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[j][e], kb[j][e], kk[j], 0, 0, 0);
          qk[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[j][e], kb[j][e], qk[j], 0, 0, 0);
        }
    }
    floatx4_t m = qk[0] + qk[1], c = kk[0] + kk[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * ti + 4 * g + i;
      const float ratio = expf(float(sum[t] - sum[other]));
      a[t][other] = other < t ? -beta[t] * ratio * c[i] : 0.f;
      m[i] = other <= t ? ratio * m[i] : 0.f;
    }
    store4(p.m + (((slot * 4 + ti) * 4 + tj) * 64 + lane) * 4, as_rows(m));
  }
  __syncthreads();  // -A is whole, and every wavefront is past its reads of q
#pragma unroll
  for (int i = 0; i < kLoadsV; ++i) put(ql, DV, i, vv[i]);
  if (wave < 4) {  // column r of the inverse of a diagonal block
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float s = t == r ? 1.f : 0.f;
#pragma unroll
      for (int i = 0; i < t; i += 4) {
        const floatx4_t c = load4(&a[16 * wave + t][16 * wave + i]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (i + e < t) s = fmaf(c[e], x[i + e], s);
      }
      x[t] = s;
    }
    if (g == 0)
#pragma unroll
      for (int t = 0; t < 16; ++t) inv[wave][t][r] = x[t];
  }
  __syncthreads();

  // Columns of U0 and W by block forward solve, 16 at a time.
  const auto solve = [&](floatx4_t (&rhs)[4], floatx4_t (&x)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < i; ++j) rhs[i] = mfma4(load4(&a[16 * i + r][16 * j + 4 * g]), x[j], rhs[i]);
      x[i] = mfma4(load4(&inv[i][r][4 * g]), rhs[i], floatx4_t{});
    }
  };
  for (int tile = wave; tile < VB; tile += kWaves) {
    floatx4_t x[4], rhs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 16 * i + 4 * g + e;
        rhs[i][e] = ql[t][16 * tile + r] * beta[t];
      }
    solve(rhs, x);
#pragma unroll
    for (int i = 0; i < 4; ++i) store4(p.u + (((slot * VB + tile) * 4 + i) * 64 + lane) * 4, x[i]);
  }
  float early[4][4], late[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * i + 4 * g + e;
      early[i][e] = -beta[t] * expf(float(sum[t]));
      late[i][e] = expf(float(sum[63] - sum[t]));
    }
  for (int tile = wave; tile < KB; tile += kWaves) {
    floatx4_t x[4], rhs[4], end;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float key = kl[16 * i + 4 * g + e][16 * tile + r];
        end[e] = key * late[i][e];
        rhs[i][e] = key * early[i][e];
      }
      store4(p.k + (((slot * KB + tile) * 4 + i) * 64 + lane) * 4, end);
    }
    solve(rhs, x);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      store4(p.w + (((slot * 4 + i) * KB + tile) * 64 + lane) * 4, as_rows(x[i]));
  }
}

// 16 columns of one value head's state.  Every wavefront holds all of them (as
// column operands) and multiplies its own 16 tokens by them; the chunk's U then
// meets in LDS, and wavefront w brings its quarter of the state's rows up to
// date, which meets in LDS again.  The next chunk's operands are loaded to
// registers a chunk ahead.
template <int DK, int DV>
__global__ void __launch_bounds__(256, 1) chunk_scan_kernel(const ChunkArgs p) {
  constexpr int KB = DK / 16, KW = KB / 4;
  __shared__ __attribute__((aligned(16))) floatx4_t us[4][64], ss[KB][64];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = 16 * blockIdx.y + r, h = blockIdx.x;
  const int64_t b = blockIdx.z, first = (b * p.hv + h) * p.chunks;
  float* state = p.state + ((b * p.hv + h) * DK + 4 * g) * DV + col;

  floatx4_t s[KB] = {};
  if (p.has_prev) {
#pragma unroll
    for (int i = 0; i < KB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[i][e] = state[(16 * i + e) * DV];
  }

  struct Operands {
    floatx4_t w[KB], q[KB], m[4], k[KW][4], u;
    float total;
  };
  const auto fetch = [&](int chunk, Operands& o) {
    const int64_t slot = first + chunk, tile = slot * 4 + wave;
#pragma unroll
    for (int i = 0; i < KB; ++i) {
      o.w[i] = load4(p.w + ((tile * KB + i) * 64 + lane) * 4);
      o.q[i] = load4(p.q + ((tile * KB + i) * 64 + lane) * 4);
    }
    o.u = load4(p.u + (((slot * (DV / 16) + blockIdx.y) * 4 + wave) * 64 + lane) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // Tiles past the diagonal hold nothing; they are loaded and not used, so
      // that the number of loads in flight is known.
      o.m[j] = load4(p.m + ((tile * 4 + j) * 64 + lane) * 4);
#pragma unroll
      for (int i = 0; i < KW; ++i)
        o.k[i][j] = load4(p.k + (((slot * KB + KW * wave + i) * 4 + j) * 64 + lane) * 4);
    }
    o.total = p.total[slot];
  };
  const auto run = [&](int chunk, const Operands& o) {
    floatx4_t u[2] = {o.u, floatx4_t{}}, y[2] = {};
    // Four sums in turn: a product is not issued right behind the one whose
    // result it adds to.
#pragma unroll
    for (int i = 0; i < KB; i += 2)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          u[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[i + j][e], s[i + j][e], u[j], 0, 0, 0);
          y[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[i + j][e], s[i + j][e], y[j], 0, 0, 0);
        }
    us[wave][lane] = u[0] + u[1];
    lds_barrier();
    floatx4_t all[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) all[j] = us[j][lane];
    floatx4_t mine[KW];
#pragma unroll
    for (int i = 0; i < KW; ++i) {
      mine[i] = floatx4_t{};
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (v == wave) mine[i] = s[KW * v + i] * o.total;
#pragma unroll
      for (int j = 0; j < 4; ++j) mine[i] = mfma4(o.k[i][j], all[j], mine[i]);
      ss[KW * wave + i][lane] = mine[i];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wave) y[j & 1] = mfma4(o.m[j], all[j], y[j & 1]);
    mfma_result_barrier(y);
    const floatx4_t sum = y[0] + y[1];
    const int t = chunk * kChunk + 16 * wave + 4 * g;
    float* out = p.out + ((b * p.steps + t) * p.hv + h) * DV + col;
    if ((chunk + 1) * kChunk <= p.steps) {
#pragma unroll
      for (int e = 0; e < 4; ++e) out[int64_t(e) * p.hv * DV] = sum[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (t + e < p.steps) out[int64_t(e) * p.hv * DV] = sum[e];
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < KB; ++i) s[i] = ss[i][lane];
  };

  Operands even, odd;
  fetch(0, even);
  // Past the last chunk its operands are loaded again: an unconditional load
  // lets each wait count the loads behind it.
  for (int chunk = 0;; chunk += 2) {
    fetch(min(chunk + 1, p.chunks - 1), odd);
    __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
    run(chunk, even);
    if (chunk + 1 == p.chunks) break;
    fetch(min(chunk + 2, p.chunks - 1), even);
    __builtin_amdgcn_sched_barrier(0);
    run(chunk + 1, odd);
    if (chunk + 2 == p.chunks) break;
  }
#pragma unroll
  for (int i = 0; i < KB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i / KW == wave) state[(16 * i + e) * DV] = s[i][e];
}

// Floats of workspace per (sequence, value head, chunk), G_C padded to 16 bytes.
int64_t chunk_floats(int dk, int dv) { return int64_t(kChunk) * (3 * dk + dv + kChunk) + 4; }

}  // namespace

extern "C" int pd_delta_workspace(int32_t batch, int32_t steps, int32_t hv, int32_t dk, int32_t dv,
                                  int64_t* floats) {
  pd::clear_error();
  if (batch < 1 || steps < 1 || hv < 1 || dk < 1 || dv < 1 || !floats)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive");
  *floats = int64_t(batch) * hv * ((int64_t(steps) + kChunk - 1) / kChunk) * chunk_floats(dk, dv);
  return PD_OK;
}

extern "C" int pd_delta_chunks(const float* act, const float* gates, float* state, float* out,
                               float* workspace, int32_t batch, int32_t steps, int32_t hk,
                               int32_t hv, int32_t dk, int32_t dv, int32_t has_prev,
                               pd_stream_t stream) {
  pd::clear_error();
  if (batch < 1 || batch > 65535 || steps < 1 || hk < 1 || hv < 1 || hv % hk)
    return pd::fail(PD_EINVAL, "batch, steps and heads must be positive, value heads a multiple");
  if ((dk != 64 && dk != 128) || (dv != 64 && dv != 128))
    return pd::fail(PD_EINVAL, "linear heads of 64 or 128 elements");
  if (!act || !gates || !state || !out || !workspace || !aligned16(act) || !aligned16(gates) ||
      !aligned16(state) || !aligned16(out) || !aligned16(workspace))
    return pd::fail(PD_EINVAL, "tensors must be present and 16-byte aligned");
  const int chunks = int((int64_t(steps) + kChunk - 1) / kChunk);
  const int64_t slots = int64_t(batch) * hv * chunks;
  if (chunks > 65535) return pd::fail(PD_EINVAL, "too many steps");
  ChunkArgs p;
  p.act = act, p.gates = gates, p.state = state, p.out = out;
  p.w = workspace;
  p.q = p.w + slots * kChunk * dk;
  p.k = p.q + slots * kChunk * dk;
  p.m = p.k + slots * kChunk * dk;
  p.u = p.m + slots * kChunk * kChunk;
  p.total = p.u + slots * kChunk * dv;
  p.steps = steps, p.hk = hk, p.hv = hv, p.chunks = chunks, p.has_prev = has_prev;
  // Heads first: the eight workgroups that read a head's chunks are then on one
  // XCD (with a multiple of eight heads) and share its L2.
  const dim3 prepare{unsigned(hv), unsigned(chunks), unsigned(batch)};
  const dim3 scan{unsigned(hv), unsigned(dv / 16), unsigned(batch)};
  const hipStream_t st = as_stream(stream);
  const auto go = [&](auto first, auto second) {
    hipLaunchKernelGGL(first, prepare, dim3(kPrepareThreads), 0, st, p);
    hipLaunchKernelGGL(second, scan, dim3(256), 0, st, p);
  };
  if (dk == 64)
    dv == 64 ? go(chunk_prepare_kernel<64, 64>, chunk_scan_kernel<64, 64>)
             : go(chunk_prepare_kernel<64, 128>, chunk_scan_kernel<64, 128>);
  else
    dv == 64 ? go(chunk_prepare_kernel<128, 64>, chunk_scan_kernel<128, 64>)
             : go(chunk_prepare_kernel<128, 128>, chunk_scan_kernel<128, 128>);
  return launch_status("pd_delta_chunks");
}
