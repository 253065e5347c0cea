// Causal prefill attention over packed or batched sequences for MI355X (gfx950):
// every new token of a sequence attends to the sequence's cached prefix, to
// the new tokens before it and to itself.
//
//   O[t, h] = softmax(scale * Q[t, h] . K[j, h / G], j <= nk - nq + t) V
//
// Bound: matrix cores.  Scores are bf16 x bf16 products accumulated in
// float32; the float32 probabilities go through the bf16 matrix cores as three
// bf16 terms whose sum is the probability itself (split3), so P V is a float32
// sum as well, at four matrix units per score where 16-bit probabilities
// would take two.
//
// Split of the work.  A workgroup of four wavefronts serves 128 packed rows (64
// at head_dim 256) of one kv head of one sequence; packed row r is query head r % G of the
// kv head's group and token r / G, so any group size fills the rows and all of
// a workgroup's rows read the same K and V.  A wavefront owns 32 rows and
// multiplies transposed: S^T = K Q^T and O^T = V^T P^T with 32 x 32 x 16 MFMAs.
// In both results lane L holds row L % 32, so the softmax state is one scalar
// a lane, and the score layout (keys 8 (i / 4) + 4 (L / 32) + i % 4 in element
// i) is the operand layout of P^T up to an order of the keys that the V reads
// follow: no probability crosses a lane or the LDS.
//
// At head_dim 256 the O and Q of 32 rows alone are 192 registers a lane, which
// leaves one wavefront a SIMD and nothing to run under its waits.  There two
// wavefronts share 32 rows: each takes half of D in the scores, whose halves
// are added through LDS, and half of the columns of O.
//
// K and V tiles of 16 KB each are double-buffered in LDS: the next tile's rows
// are loaded to registers before a tile's MFMAs and written after them, one
// barrier a tile.  The loads are buffer loads whose range ends at the last
// live row, so rows past the sequence, pages outside the pool and entries past
// the table's width read as zeros and never touch other memory.
//
// What bounds it: instructions.  A 32 x 32 tile of scores at head_dim 128 is 32
// MFMAs (1024 clocks) and, an element, an FMA, an exponential, an addition, half
// a maximum and 5.5 operations of the split, about 160 vector instructions (640
// clocks and the exponentials' 190); counters show half of the SIMDs' time in
// either, little of it at once.  So masks are a branch in the tiles that need
// them, and infinities and NaN of V are left to a second pass: a row tile whose
// sums are not finite is taken again with them outside the matrix products,
// where a zero probability (a masked key's among them) would make a NaN of
// them, and added for the rows that see their key.
//
// Measured on MI355X, K/V write included: four prompts of 17 to 2048 tokens, Hq
// 32 / Hkv 8 / D 128, 3964 -> 204 us (float32 products of the materialized
// scores before; 210 with a split of 7 operations and masks in line); 1000
// tokens after 3072 cached, Hq 16 / Hkv 4 / D 256, 1144 -> 168 us; 512 tokens,
// Hq 8 / Hkv 2 / D 256, 31 us in one span (45 with 32 whole rows a wavefront).
//
// Few rows leave CUs idle (128 rows of each kv head a workgroup): grid.y > 1
// cuts each row tile's keys into equal spans whose float32 (m, l, O) partials
// prefill_merge_kernel combines.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <cstdint>

#include "pd_check.h"
#include "pd_device.h"
#include "pd_internal.h"
#include "pd_launch.h"

namespace {

using namespace pdk;
using pd::aligned16;
using pd::as_stream;
using pd::launch_status;

struct PrefillArgs {
  const uint16_t *q, *k, *v;
  uint16_t* out;
  float *part_o, *part_ml;  // split partials: [split][row][D] and [split][row][2]
  const int32_t *cu_q, *cu_k, *table;
  int64_t qsb, qsn, qsh, ksb, ksn, ksh, vsb, vsn, vsh, osb, osn, osh, tsb;
  int64_t total_q, total_k, num_pages;
  int num_seqs, seq_len, table_width, page_size, num_kv_heads, G, splits;
  float scale;
  int32_t* verdicts;  // of the packed metadata, or null
};

template <int D>
struct Prefill {
  static constexpr int kTile = D == 256 ? 32 : 64;       // keys per tile
  static constexpr int kBlocks = kTile / 32;             // 32-key MFMA blocks
  static constexpr int kPieces = D / 8;                  // 16-byte pieces per row
  static constexpr int kLoads = kTile * kPieces / 256;   // pieces per thread, K or V
  static constexpr int kTileBytes = kTile * D * 2;
  // D = 256: two wavefronts share 32 rows, each with half of D (see above).
  static constexpr int kParts = D == 256 ? 2 : 1;
  static constexpr int kRows = 128 / kParts;             // packed rows per workgroup
  static constexpr int kCols = D / kParts;               // of a wavefront
  static constexpr int kSteps = kCols / 16;              // QK MFMAs per block
  static constexpr int kOut = kCols / 32;                // 32-column blocks of O
};

// Piece permutation of a V row: a transposed read takes 64 bytes of four
// consecutive rows at once, which must fall on distinct 64-byte bank groups.
// Rows of 256 bytes or more start on bank 0; 128-byte rows alternate halves.
template <int D>
__device__ __forceinline__ int v_swizzle(int row) {
  return D >= 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1);
}

// p = hi + mid + lo exactly, each a bf16 (the top 16 bits of a float32): every
// term takes the next eight significant bits, truncated.
struct Split3 {
  uint32_t hi, mid, lo;
};
__device__ __forceinline__ Split3 split3(float p) {
  Split3 s;
  s.hi = __float_as_uint(p) & 0xffff0000u;
  const float r = p - __uint_as_float(s.hi);
  s.mid = __float_as_uint(r) & 0xffff0000u;
  s.lo = __float_as_uint(r - __uint_as_float(s.mid));
  return s;
}
// 0xffff in each half of x that is an infinity or NaN.
__device__ __forceinline__ uint32_t odd_halves(uint32_t x) {
  const uint32_t ones = ((x & 0x7f807f80u) + 0x00800080u) >> 15 & 0x00010001u;
  return (ones << 16) - ones;
}
// The upper halves of (a, b) as one dword, a in the low half.
__device__ __forceinline__ uint32_t upper_halves(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// The sequence and row tile of grid tile `t` (counted from the last), for
// packed sequences: the tiles of 64 sequences at a time, one a lane, summed by
// a wavefront prefix.  Returns false past the last tile.
template <int kRows>
__device__ __forceinline__ bool find_tile(const PrefillArgs& a, int t, int lane, int& seq,
                                          int& tile) {
  for (int base = 0; base < a.num_seqs; base += 64) {
    const int i = base + lane;
    int n = 0;
    if (i < a.num_seqs) {
      const int64_t lo = max(0, a.cu_q[i]);
      const int64_t hi = min(int64_t(a.cu_q[i + 1]), a.total_q);
      n = hi > lo ? int(((hi - lo) * a.G + kRows - 1) / kRows) : 0;
    }
    int sum = n;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const int up = __shfl_up(sum, d);
      if (lane >= d) sum += up;
    }
    const int total = __shfl(sum, 63);
    if (t < total) {
      const int at = __popcll(__ballot(sum <= t));
      seq = base + at;
      tile = t - __shfl(sum - n, at);
      return true;
    }
    t -= total;
  }
  return false;
}

// kPaged: K and V are pages read through the table, page_size a multiple of
// the tile; else rows of the call's own tensors.
template <int D, bool kPaged>
__global__ void __launch_bounds__(256, 2) prefill_kernel(const PrefillArgs a) {
  using P = Prefill<D>;
  constexpr int kRows = P::kRows;
  __shared__ __attribute__((aligned(16))) char lds[2][2][P::kTileBytes];
  const int tid = threadIdx.x, lane = tid & 63;
  __shared__ __attribute__((aligned(16))) floatx4_t partial[P::kParts == 2 ? 4 : 1][4][64];
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = wave % (kRows / 32), part = wave / (kRows / 32);  // rows 32 w, columns of `part`
  const int half = lane >> 5, col = lane & 31;

  if (has_share(a.verdicts)) check_packed<kPaged>(a, tid);

  // Longest first: tiles are counted from the last, whose rows see most keys.
  const int id = blockIdx.x;
  const int kvh = id % a.num_kv_heads;
  const int grid_tiles = gridDim.x / a.num_kv_heads;
  const int t_rev = grid_tiles - 1 - id / a.num_kv_heads;
  int seq, tile;
  int64_t q0, k0;
  int nq, nk;
  if (a.cu_q) {
    if (!find_tile<kRows>(a, t_rev, lane, seq, tile)) return;
    seq = __builtin_amdgcn_readfirstlane(seq);
    tile = __builtin_amdgcn_readfirstlane(tile);
    q0 = max(0, a.cu_q[seq]);
    nq = int(min(int64_t(a.cu_q[seq + 1]), a.total_q) - q0);
    k0 = max(0, a.cu_k[seq]);
    const int64_t klim = kPaged ? int64_t(a.table_width) * a.page_size : a.total_k - k0;
    nk = int(min(max(int64_t(0), min(int64_t(a.cu_k[seq + 1]) - a.cu_k[seq], klim)),
                 int64_t(0x7fffffff)));
  } else {
    const int tiles = (int64_t(a.seq_len) * a.G + kRows - 1) / kRows;
    seq = t_rev / tiles;
    tile = t_rev % tiles;
    q0 = k0 = 0;
    nq = nk = a.seq_len;
  }

  // This lane's packed row (a clamped copy of the last one past the end).
  const int rows = nq * a.G;
  const int row = tile * kRows + 32 * w + col;
  const int at = min(row, rows - 1);
  const int token = at / a.G, head = kvh * a.G + at % a.G;
  const int limit = nk - nq + token;  // last key this row sees
  // Keys of the workgroup's and of the wavefront's last and first rows.
  const int last = min(tile * kRows + kRows, rows) - 1;
  const int wg_keys = max(0, nk - nq + last / a.G + 1);
  const int wave_first = min(tile * kRows + 32 * w, rows - 1) / a.G + nk - nq;
  const int wave_last = min(tile * kRows + 32 * w + 31, rows - 1) / a.G + nk - nq;
  int t_begin = 0, t_end = (wg_keys + P::kTile - 1) / P::kTile;
  if (a.splits > 1) {
    const int s = blockIdx.y, n = t_end;
    t_begin = int(int64_t(n) * s / a.splits);
    t_end = int(int64_t(n) * (s + 1) / a.splits);
  }

  // A negative scale is taken by Q's sign, which is exact, so that the largest
  // product is the largest score.
  const float c = fabsf(a.scale) * kLog2e;
  const uint32_t flip = a.scale < 0.f ? 0x80008000u : 0u;
  u32x4_t qf[P::kSteps];
  {
    const uint16_t* qrow = a.q + seq * a.qsb + (q0 + token) * a.qsn + head * a.qsh;
#pragma unroll
    for (int s = 0; s < P::kSteps; ++s) {
      qf[s] = load16(qrow + P::kCols * part + 16 * s + 8 * half);
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[s][e] ^= flip;
    }
  }

  // Piece i of this thread is piece 0 kStep rows further down; the swizzles
  // repeat within 16 rows, and 8 rows further down K's differs in one bit.
  constexpr int kStep = 256 / P::kPieces;
  static_assert(kStep % 16 == 0 || (kStep == 8 && D >= 128), "swizzles by up to four bits of the row");
  const int row0 = tid / P::kPieces, piece0 = tid % P::kPieces;
  const int src_k = int((row0 * a.ksn + 8 * piece0) * 2), src_v = int((row0 * a.vsn + 8 * piece0) * 2);
  const int dst_k = row0 * D * 2 + 16 * (piece0 ^ kswz<D>(row0));
  const int dst_v = row0 * D * 2 + 16 * (piece0 ^ v_swizzle<D>(row0));
  const uint16_t* k_first = a.k + kvh * a.ksh + (kPaged ? 0 : seq * a.ksb + k0 * a.ksn);
  const uint16_t* v_first = a.v + kvh * a.vsh + (kPaged ? 0 : seq * a.vsb + k0 * a.vsn);
  u32x4_t kr[P::kLoads], vr[P::kLoads];
  const auto fetch = [&](int t) {
    const int first = t * P::kTile;
    int live = min(P::kTile, nk - first), slot = first;
    const uint16_t *kp = k_first, *vp = v_first;
    if constexpr (kPaged) {
      int64_t page = a.table[seq * a.tsb + first / a.page_size];
      slot = first % a.page_size;
      if (page < 0 || page >= a.num_pages) live = 0, page = 0;
      kp += page * a.ksb, vp += page * a.vsb;
    }
    kp += slot * a.ksn, vp += slot * a.vsn;
    const auto rk = buffer_rsrc(kp, int(live * a.ksn * 2));
    const auto rv = buffer_rsrc(vp, int(live * a.vsn * 2));
    // Opaque to the compiler, which would keep every sum in a register.
    int step_k = int(kStep * a.ksn * 2), step_v = int(kStep * a.vsn * 2);
    asm volatile("" : "+s"(step_k), "+s"(step_v));
#pragma unroll
    for (int i = 0; i < P::kLoads; ++i) kr[i] = buffer_load16(rk, src_k + i * step_k);
#pragma unroll
    for (int i = 0; i < P::kLoads; ++i) vr[i] = buffer_load16(rv, src_v + i * step_v);
  };
  const auto place = [&](int b) {
#pragma unroll
    for (int i = 0; i < P::kLoads; ++i)
      *reinterpret_cast<u32x4_t*>(lds[b][0] + (dst_k ^ (kStep == 8 && i % 2 ? 128 : 0)) +
                                  i * kStep * D * 2) = kr[i];
#pragma unroll
    for (int i = 0; i < P::kLoads; ++i)
      *reinterpret_cast<u32x4_t*>(lds[b][1] + dst_v + i * kStep * D * 2) = vr[i];
  };

  floatx16_t o[P::kOut];
  float m, l;  // m in units of log2; l of this lane's keys

  // Transposed V reads: lane's row of a 16-key group and its byte in the row
  // for 32-column blocks j = 0..3 (mod 4).
  const int vrow = 4 * half + ((lane & 15) >> 2);
  int vat[P::kOut < 4 ? P::kOut : 4];
#pragma unroll
  for (int j = 0; j < (P::kOut < 4 ? P::kOut : 4); ++j) {
    const int piece = P::kCols / 8 * part + 4 * j + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    vat[j] = vrow * D * 2 + 16 * (piece ^ v_swizzle<D>(vrow)) + 8 * (lane & 1);
  }

  const auto sweep = [&](auto safe) {
    constexpr bool kSafe = decltype(safe)::value;
#pragma unroll
    for (int j = 0; j < P::kOut; ++j) o[j] = floatx16_t{};
    m = -INFINITY, l = 0.f;
    if (t_begin < t_end) {
      fetch(t_begin);
      place(0);
    }
    for (int t = t_begin; t < t_end; ++t) {
      const int b = (t - t_begin) & 1;
      __syncthreads();
      if (t + 1 < t_end) fetch(t + 1);
      const int first = t * P::kTile;
      if (P::kParts == 2 || first <= wave_last) {
        const char* ks = lds[b][0];
        const char* vs = lds[b][1];
        // Two sums in turn (32-key blocks, or halves of the contraction): a
        // product right behind the one it adds to waits for its result.
        floatx16_t s[2] = {};
        constexpr int kChain = P::kBlocks == 2 ? 1 : 2;
#pragma unroll
        for (int d = 0; d < P::kSteps; d += kChain)
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const int r = (P::kBlocks == 2 ? 32 * n : 0) + col, step = d + (kChain == 2 ? n : 0);
            const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(
                ks + r * D * 2 + P::kCols * 2 * part + 16 * ((2 * step + half) ^ kswz<D>(r)));
            s[n] = mfma32(kf, qf[step], s[n]);
          }
        if constexpr (P::kBlocks == 1) s[0] += s[1];
        if constexpr (P::kParts == 2) {
          // The two halves of the contraction meet in LDS; both wavefronts add
          // them in the same order and go on with the same scores.
#pragma unroll
          for (int g = 0; g < 4; ++g)
            partial[wave][g][lane] =
                floatx4_t{s[0][4 * g], s[0][4 * g + 1], s[0][4 * g + 2], s[0][4 * g + 3]};
          lds_barrier();
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const floatx4_t other = partial[wave ^ 2][g][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) s[0][4 * g + e] += other[e];
          }
        }
        // Keys past the row's limit, only in tiles that reach past the first
        // row's: their scores leave the maximum and their probabilities are 0.
        const bool edge = first + P::kTile - 1 > wave_first;
        if (edge) {
          asm volatile("");  // a branch, not selects in every tile
#pragma unroll
          for (int n = 0; n < P::kBlocks; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (first + 32 * n + 8 * (i / 4) + 4 * half + i % 4 > limit) s[n][i] = -INFINITY;
        }
        float top = s[0][0];
#pragma unroll
        for (int n = 0; n < P::kBlocks; ++n)
#pragma unroll
          for (int i = 0; i < 16; ++i) top = fmaxf(top, s[n][i]);
        top = fmaxf(top, xor_lanes<32>(top, lane));
        // A scale of 0 leaves a zero score where a masked row's top is -inf.
        const float mt = top == -INFINITY ? -INFINITY : top * c;
        // The running maximum moves only when a row's grows by more than 2^8:
        // the probabilities stay below 2^8 and the sums are the same.
        if (__any(mt > m + 8.f)) {
          const float up = fmaxf(m, mt);
          const float f = exp2_fast(m - (up == -INFINITY ? 0.f : up));
          m = up;
          l *= f;
#pragma unroll
          for (int j = 0; j < P::kOut; ++j)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[j][i] *= f;
        }
        const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int n = 0; n < P::kBlocks; ++n) {
#pragma unroll
          for (int i = 0; i < 16; ++i) s[n][i] = exp2_fast(fmaf(s[n][i], c, -base));
          if (edge) {
          asm volatile("");  // a branch, not selects in every tile
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (first + 32 * n + 8 * (i / 4) + 4 * half + i % 4 > limit) s[n][i] = 0.f;
          }
#pragma unroll
          for (int i = 0; i < 16; ++i) l += s[n][i];
#pragma unroll
          for (int g = 0; g < 2; ++g) {  // 16 keys a step
            u32x4_t hi, mid, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const Split3 x = split3(s[n][8 * g + 2 * e]), y = split3(s[n][8 * g + 2 * e + 1]);
              hi[e] = upper_halves(x.hi, y.hi);
              mid[e] = upper_halves(x.mid, y.mid);
              lo[e] = upper_halves(x.lo, y.lo);
            }
            const char* vg = vs + (32 * n + 16 * g) * D * 2;
            u32x4_t vf[P::kOut];
#pragma unroll
            for (int j = 0; j < P::kOut; ++j) {
              const char* p = vg + vat[j & 3] + 256 * (j >> 2);
              const short4_t v0 = lds_read_tr(p), v1 = lds_read_tr(p + 8 * D * 2);
              const uint64_t a0 = __builtin_bit_cast(uint64_t, v0), a1 = __builtin_bit_cast(uint64_t, v1);
              vf[j] = u32x4_t{uint32_t(a0), uint32_t(a0 >> 32), uint32_t(a1), uint32_t(a1 >> 32)};
            }
            // Infinities and NaN of V: not in the products, where a zero term makes a
            // NaN of them in every row, but added for the rows that see their key.
            uint32_t found[4] = {};
            if constexpr (kSafe) {
#pragma unroll
              for (int j = 0; j < P::kOut; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const uint32_t odd = odd_halves(vf[j][e]);
                  vf[j][e] &= ~odd;
                  found[e] |= odd;
                }
            }
#pragma unroll
            for (int j = 0; j < P::kOut; ++j) o[j] = mfma32(vf[j], lo, o[j]);
#pragma unroll
            for (int j = 0; j < P::kOut; ++j) o[j] = mfma32(vf[j], mid, o[j]);
#pragma unroll
            for (int j = 0; j < P::kOut; ++j) o[j] = mfma32(vf[j], hi, o[j]);
            if constexpr (kSafe) {
              if (__any(found[0] | found[1] | found[2] | found[3])) {
                // The products' results are read in another block: 24 wait states.
                asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
                for (int j = 0; j < P::kOut; ++j) asm volatile("" : "+v"(o[j]));
#pragma unroll 1
                for (int key = 0; key < 16; ++key) {
                  // Element of this key, in the lanes of one half.
                  const int e = 4 * (key / 8) + key % 4, r = 32 * n + 16 * g + key;
                  float p = 0.f;
#pragma unroll
                  for (int i = 0; i < 8; ++i)
                    if (i == e) p = s[n][8 * g + i];
                  const float other = xor_lanes<32>(p, lane);
                  if ((key / 4) % 2 != half) p = other;
                  if (first + r <= limit) {
#pragma unroll
                    for (int j = 0; j < P::kOut; ++j)
#pragma unroll
                      for (int i = 0; i < 16; i += 4) {
                        u32x2_t x = *reinterpret_cast<const u32x2_t*>(
                            vs + r * D * 2 + 8 * half +
                            16 * ((P::kCols / 8 * part + 4 * j + i / 4) ^ v_swizzle<D>(r)));
                        x.x &= odd_halves(x.x), x.y &= odd_halves(x.y);
                        o[j][i] = fmaf(p, bf16_lo(x.x), o[j][i]);
                        o[j][i + 1] = fmaf(p, bf16_hi(x.x), o[j][i + 1]);
                        o[j][i + 2] = fmaf(p, bf16_lo(x.y), o[j][i + 2]);
                        o[j][i + 3] = fmaf(p, bf16_hi(x.y), o[j][i + 3]);
                      }
                  }
                }
              }
            }
          }
        }
      }
      if (t + 1 < t_end) place(b ^ 1);
    }

    // The loop's last MFMAs and the reads below are in different blocks: 24 wait
    // states cover them.
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
    for (int j = 0; j < P::kOut; ++j) asm volatile("" : "+v"(o[j]));
  };
  sweep(std::false_type{});
  // A NaN may be a zero probability times an infinity or NaN: such row tiles are
  // taken again with those outside the products.
  float odd = 0.f;
#pragma unroll
  for (int j = 0; j < P::kOut; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) odd = fmaf(o[j][i], 0.f, odd);  // NaN of an infinity too
  int* flags = reinterpret_cast<int*>(&lds[0][0][0]);
  __syncthreads();
  const int any_odd = __any(odd != 0.f);
  if (lane == 0) flags[wave] = any_odd;
  __syncthreads();
  const bool again = flags[0] | flags[1] | flags[2] | flags[3];
  __syncthreads();
  if (again) sweep(std::true_type{});
  l += xor_lanes<32>(l, lane);

  if (a.splits > 1) {
    if (row < rows) {
      const int64_t r = ((int64_t(seq) * a.seq_len + q0 + token) * a.num_kv_heads * a.G) + head;
      const int64_t all = a.total_q * a.num_kv_heads * a.G;
      const int64_t pr = blockIdx.y * all + r;
      float* po = a.part_o + pr * D;
#pragma unroll
      for (int j = 0; j < P::kOut; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<floatx4_t*>(po + P::kCols * part + 32 * j + 8 * g + 4 * half) =
              floatx4_t{o[j][4 * g], o[j][4 * g + 1], o[j][4 * g + 2], o[j][4 * g + 3]};
      if (half == 0 && part == 0) {
        a.part_ml[2 * pr] = m;
        a.part_ml[2 * pr + 1] = l;
      }
    }
    return;
  }

  // Output rows through LDS (each wavefront its own 32, after every wavefront
  // has read its last tile), stored 16 bytes a lane.
  __syncthreads();
  char* stage = &lds[0][0][0] + wave * 32 * P::kCols * 2;
  const float inv = 1.f / l;
#pragma unroll
  for (int j = 0; j < P::kOut; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int piece = 4 * j + g;
      uint32_t* d = reinterpret_cast<uint32_t*>(stage + col * P::kCols * 2 +
                                                16 * (piece ^ (col & 7)) + 8 * half);
      d[0] = pack_bf16(o[j][4 * g] * inv, o[j][4 * g + 1] * inv);
      d[1] = pack_bf16(o[j][4 * g + 2] * inv, o[j][4 * g + 3] * inv);
    }
  // A wavefront's own LDS writes are visible to it in order.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  constexpr int kRowPieces = P::kCols / 8;
#pragma unroll
  for (int i = 0; i < 32 * kRowPieces / 64; ++i) {
    const int idx = 64 * i + lane, r = idx / kRowPieces, p = idx % kRowPieces;
    const int pr = tile * kRows + 32 * w + r;
    const u32x4_t x =
        *reinterpret_cast<const u32x4_t*>(stage + r * P::kCols * 2 + 16 * (p ^ (r & 7)));
    if (pr < rows)
      *reinterpret_cast<u32x4_t*>(a.out + seq * a.osb + (q0 + pr / a.G) * a.osn +
                                  (kvh * a.G + pr % a.G) * a.osh + P::kCols * part + 8 * p) = x;
  }
}

// Combines the splits of each row: one wavefront a row, D / 64 elements a lane.
template <int D>
__global__ void __launch_bounds__(256)
prefill_merge_kernel(const PrefillArgs a, int64_t all) {
  const int lane = threadIdx.x & 63;
  const int64_t r = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= all) return;
  constexpr int E = D / 64;
  float m = -INFINITY;
  for (int s = 0; s < a.splits; ++s) m = fmaxf(m, a.part_ml[2 * (s * all + r)]);
  const float base = m == -INFINITY ? 0.f : m;
  float l = 0.f, o[E] = {};
  for (int s = 0; s < a.splits; ++s) {
    const int64_t pr = s * all + r;
    const float f = exp2_fast(a.part_ml[2 * pr] - base);
    l += f * a.part_ml[2 * pr + 1];
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] += f * a.part_o[pr * D + E * lane + e];
  }
  const float inv = 1.f / l;
  const int heads = a.num_kv_heads * a.G;
  const int64_t n = r / heads;
  const int64_t seq = a.cu_q ? 0 : n / a.seq_len, t = a.cu_q ? n : n % a.seq_len;
  uint16_t* out = a.out + seq * a.osb + t * a.osn + (r % heads) * a.osh + E * lane;
#pragma unroll
  for (int e = 0; e < E; ++e) out[e] = uint16_t(bf16_bits(o[e] * inv));
}

template <int D>
void launch(const PrefillArgs& a, unsigned grid, hipStream_t stream) {
  const dim3 g(grid, unsigned(a.splits));
  if (a.table)
    hipLaunchKernelGGL((prefill_kernel<D, true>), g, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((prefill_kernel<D, false>), g, dim3(256), 0, stream, a);
  if (a.splits > 1) {
    const int64_t all = a.total_q * a.num_kv_heads * a.G;
    hipLaunchKernelGGL(prefill_merge_kernel<D>, dim3(unsigned((all + 3) / 4)), dim3(256), 0, stream,
                       a, all);
  }
}

int run_prefill(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                const void* v, const int64_t* v_strides, void* out, const int64_t* out_strides,
                const int32_t* cu_q, const int32_t* cu_k, int32_t num_seqs, int32_t seq_len,
                int64_t total_q, int64_t total_k, const int32_t* table, int64_t table_stride_b,
                int32_t table_width, int32_t page_size, int64_t num_pages, int32_t num_heads,
                int32_t num_kv_heads, int32_t head_dim, double scale, int32_t splits,
                float* part_o, float* part_ml, int32_t* verdicts, pd_stream_t stream) {
  pd::clear_error();
  if (num_seqs < 1 || num_heads < 1 || num_kv_heads < 1 || num_heads % num_kv_heads)
    return pd::fail(PD_EINVAL, "sequences and heads must be positive, heads divisible by kv heads");
  if (!pd::valid_head_dim(head_dim))
    return pd::fail(PD_EINVAL, "prefill supports head_dim 64, 128, or 256");
  if (total_q < 0 || total_q > 0x7fffffff || total_k < 0 || total_k > 0x7fffffff)
    return pd::fail(PD_EINVAL, "token counts must lie in [0, 2^31)");
  if (verdicts && !cu_q) return pd::fail(PD_EINVAL, "only packed metadata are checked");
  if (total_q == 0) {
    mark_absent(verdicts, 0);
    return PD_OK;
  }
  if (!q || !k || !v || !out || !q_strides || !k_strides || !v_strides || !out_strides)
    return pd::fail(PD_EINVAL, "null tensor pointer");
  if ((cu_q == nullptr) != (cu_k == nullptr) || (table && !cu_q))
    return pd::fail(PD_EINVAL, "packed sequences need both cumulative lengths");
  if (!cu_q && (seq_len < 1 || total_q != int64_t(num_seqs) * seq_len))
    return pd::fail(PD_EINVAL, "batched sequences need total_q = num_seqs * seq_len");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out))
    return pd::fail(PD_EINVAL, "q, k, v and out must be 16-byte aligned");
  const int64_t* all[4] = {q_strides, k_strides, v_strides, out_strides};
  for (const int64_t* s : all)
    for (int i = 0; i < 3; ++i)
      if (s[i] < 0 || s[i] % 8)
        return pd::fail(PD_EINVAL, "strides must be non-negative multiples of 8 elements");
  // A tile's rows are addressed with 32-bit offsets from its first row, and a
  // row stride below head_dim would end the range inside a row.
  for (int i = 1; i < 3; ++i)
    if (all[i][1] < head_dim || all[i][1] > (int64_t(1) << 23))
      return pd::fail(PD_EINVAL, "k and v token strides must lie in [head_dim, 2^23]");
  const int tile = head_dim == 256 ? 32 : 64, kRows = head_dim == 256 ? 64 : 128;
  if (table && (table_width < 1 || num_pages < 1 || page_size < tile || page_size % tile))
    return pd::fail(PD_EINVAL, "the page size must be a multiple of %d tokens", tile);
  const int G = num_heads / num_kv_heads;
  if (total_q * num_heads > 0x7fffffff)
    return pd::fail(PD_EINVAL, "tokens times heads must stay below 2^31");
  if (splits < 1 || splits > 64) return pd::fail(PD_EINVAL, "splits must lie in [1, 64]");
  if (splits > 1 && (!part_o || !part_ml || !aligned16(part_o)))
    return pd::fail(PD_EINVAL, "split prefill needs its 16-byte aligned workspace");

  PrefillArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.out = static_cast<uint16_t*>(out);
  a.part_o = part_o;
  a.part_ml = part_ml;
  a.cu_q = cu_q;
  a.cu_k = cu_k;
  a.table = table;
  a.qsb = q_strides[0], a.qsn = q_strides[1], a.qsh = q_strides[2];
  a.ksb = k_strides[0], a.ksn = k_strides[1], a.ksh = k_strides[2];
  a.vsb = v_strides[0], a.vsn = v_strides[1], a.vsh = v_strides[2];
  a.osb = out_strides[0], a.osn = out_strides[1], a.osh = out_strides[2];
  if (cu_q) {  // packed: one batch entry; pages keep their own stride
    a.qsb = a.osb = 0;
    if (!table) a.ksb = a.vsb = 0;
  }
  a.tsb = table_stride_b;
  a.total_q = total_q;
  a.total_k = total_k;
  a.num_pages = num_pages;
  a.num_seqs = num_seqs;
  a.seq_len = cu_q ? 0 : seq_len;
  a.table_width = table_width;
  a.page_size = page_size;
  a.num_kv_heads = num_kv_heads;
  a.G = G;
  a.splits = splits;
  a.scale = float(scale);
  // Packed: at most this many row tiles, whatever the lengths are.
  const int64_t tiles = cu_q ? total_q * G / kRows + num_seqs
                             : int64_t(num_seqs) * ((int64_t(seq_len) * G + kRows - 1) / kRows);
  const int64_t grid = tiles * num_kv_heads;
  if (grid > 0x7fffffff) return pd::fail(PD_EINVAL, "grid dimension exceeds device limits");
  a.verdicts = verdicts;
  mark_absent(verdicts, grid);
  const hipStream_t st = as_stream(stream);
  if (head_dim == 64)
    launch<64>(a, unsigned(grid), st);
  else if (head_dim == 128)
    launch<128>(a, unsigned(grid), st);
  else
    launch<256>(a, unsigned(grid), st);
  return launch_status("pd_prefill");
}

}  // namespace

extern "C" int pd_prefill(const void* q, const int64_t* q_strides, const void* k,
                          const int64_t* k_strides, const void* v, const int64_t* v_strides,
                          void* out, const int64_t* out_strides, const int32_t* cu_q,
                          const int32_t* cu_k, int32_t num_seqs, int32_t seq_len, int64_t total_q,
                          int64_t total_k, const int32_t* table, int64_t table_stride_b,
                          int32_t table_width, int32_t page_size, int64_t num_pages,
                          int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, double scale,
                          int32_t splits, float* part_o, float* part_ml, pd_stream_t stream) {
  return run_prefill(q, q_strides, k, k_strides, v, v_strides, out, out_strides, cu_q, cu_k, num_seqs,
                     seq_len, total_q, total_k, table, table_stride_b, table_width, page_size,
                     num_pages, num_heads, num_kv_heads, head_dim, scale, splits, part_o, part_ml,
                     nullptr, stream);
}

extern "C" int pd_prefill_checked(const void* q, const int64_t* q_strides, const void* k,
                       const int64_t* k_strides, const void* v, const int64_t* v_strides, void* out,
                       const int64_t* out_strides, const int32_t* cu_q, const int32_t* cu_k,
                       int32_t num_seqs, int32_t seq_len, int64_t total_q, int64_t total_k,
                       const int32_t* table, int64_t table_stride_b, int32_t table_width,
                       int32_t page_size, int64_t num_pages, int32_t num_heads,
                       int32_t num_kv_heads, int32_t head_dim, double scale, int32_t splits,
                       float* part_o, float* part_ml, int32_t* verdicts, pd_stream_t stream) {
  return run_prefill(q, q_strides, k, k_strides, v, v_strides, out, out_strides, cu_q, cu_k, num_seqs,
                     seq_len, total_q, total_k, table, table_stride_b, table_width, page_size,
                     num_pages, num_heads, num_kv_heads, head_dim, scale, splits, part_o, part_ml,
                     verdicts, stream);
}

extern "C" int pd_check_wait(const int32_t* verdicts, pd_stream_t stream, int32_t* found) {
  pd::clear_error();
  if (!verdicts || !found) return pd::fail(PD_EINVAL, "null pointer");
  *found = 0;
  // The stream is asked once a millisecond, which costs it a packet: when it has
  // ended, every write has been made.
  using Clock = std::chrono::steady_clock;
  auto ask = Clock::now() + std::chrono::milliseconds(1);
  bool done = false;
  for (int word = 0; word < PD_CHECK_WORDS; ++word) {
    int32_t v = 0;
    for (unsigned spin = 1;; ++spin) {
      v = __atomic_load_n(verdicts + word, __ATOMIC_ACQUIRE);
      if (v || done) break;
      if (spin % 64 == 0 && Clock::now() >= ask) {
        const hipError_t state = hipStreamQuery(as_stream(stream));
        if (state != hipSuccess && state != hipErrorNotReady)
          return pd::fail(PD_ELAUNCH, "pd_check_wait: %s", hipGetErrorString(state));
        done = state == hipSuccess;
        ask = Clock::now() + std::chrono::milliseconds(1);
      }
    }
    if (!v) return pd::fail(PD_ELAUNCH, "pd_check_wait: the check did not run");
    *found |= v & (PD_CHECK_ODD | PD_CHECK_OUTSIDE);
  }
  return PD_OK;
}
