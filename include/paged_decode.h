/*
 * paged_decode.h — C ABI of the MI355X (gfx950) paged decode operator.
 *
 * One query token per sequence attends over a paged KV cache:
 *   Q       bf16 [batch, num_heads, head_dim], innermost dim contiguous,
 *           rows 16-byte aligned (strides in elements are multiples of 8)
 *   K, V    bf16 [num_pages, 256, num_kv_heads, head_dim], contiguous (NHD pages)
 *   table   int32 [batch, width] block table, row stride table_stride_b,
 *           width = table_width (1 <= width < 2^22); logical token t of row b
 *           lives in page table[b, t / 256], slot t % 256.  Entries are read
 *           only inside the row's width: a length beyond width * 256 reads
 *           page 0 for the missing entries, never memory outside the table.
 *   lengths int32 [batch], 0 <= lengths[b] <= width * 256
 * Element offset of (page, slot, kv_head, d) is ((page*256+slot)*Hkv+kv_head)*D+d,
 * computed in 64-bit.  Query head h reads kv head h / (num_heads / num_kv_heads).
 *
 * Conventions of every entry point:
 *   - returns PD_OK (0) or a nonzero pd_status; pd_last_error() then holds a
 *     message for the calling thread;
 *   - pointers to tensors are device pointers; nothing is allocated, nothing
 *     synchronizes, no device memory is read on the host, so every launch can
 *     be recorded into a hipGraph on `stream` and replayed with new contents;
 *   - tensor CONTENTS are trusted (live table entries must name valid pages);
 *     use pd_validate_metadata on host copies to check them.
 * `pd_stream_t` is the same type as hipStream_t.
 */
#ifndef PAGED_DECODE_H_
#define PAGED_DECODE_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ihipStream_t* pd_stream_t;

enum pd_status { PD_OK = 0, PD_EINVAL = 1, PD_ELAUNCH = 2 };

#define PD_PAGE_SIZE 256      /* spec.py:6 */
#define PD_PARTITION_SIZE 1024 /* spec.py:7 */
#define PD_ABI_VERSION 7

/* Split-KV plan; field meanings follow SplitKVPlan (splitkv_plan.py:15-23). */
typedef struct pd_plan {
  int32_t splits;
  int32_t tile_tokens;
  int32_t tokens_per_split;
  int32_t table_capacity_tokens;
  int32_t lse_lanes;
  int32_t sm_count;
  int32_t is_explicit; /* 1 = policy "explicit", 0 = "pinned_geometry" */
} pd_plan;

/* Message describing the last failure on the calling thread ("" if none). */
const char* pd_last_error(void);

/* PD_ABI_VERSION of the built library. */
int pd_abi_version(void);

/* Replaces make_splitkv_plan (splitkv_plan.py:26-56), bit-exact including its
 * float32 rounding points.  max_context_len gives the table capacity through
 * ceil(max_context_len / 256) * 256 (spec.py:36-38).  num_splits = 0 selects
 * the pinned-geometry heuristic, 1..128 an explicit count. */
int pd_make_plan(int32_t max_batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                 int32_t max_context_len, int32_t sm_count, int32_t num_splits, pd_plan* out);

/* Host-memory content check; replaces validate_metadata (reference.py:10-21)
 * as used by validate_device_metadata (runtime.py:38-43): lengths within
 * [0, max_context_len], live pages ceil(len/256) <= width, live entries within
 * [0, num_pages).  `table` and `lengths` are HOST pointers. */
int pd_validate_metadata(const int32_t* table, int64_t table_stride_b, int32_t width,
                         const int32_t* lengths, int32_t batch, int64_t num_pages,
                         int32_t max_context_len);

/* Matched split-KV partition; replaces _normalized_partition
 * (matched_splitkv.py:52-98) as launched by matched_decode (:142-146).
 * Writes partials f32 [batch, num_heads, splits, head_dim] (normalized) and
 * lse f32 [batch, num_heads, splits] (-inf for an empty partition).
 * Partition p covers [p*tokens_per_split, min((p+1)*tokens_per_split, len)),
 * walked in tile_tokens tiles from the last to the first.  Requires
 * head_dim in {64,128,256}, tile_tokens == 16384/head_dim, tokens_per_split a
 * multiple of tile_tokens, num_heads/num_kv_heads <= 16, splits in [1,128].
 * splits * tokens_per_split < 2^31.
 * scale is applied to the scores (exp2 argument uses f32(scale*log2(e))). */
int pd_partition(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                 const void* k, const void* v,
                 const int32_t* table, int64_t table_stride_b, int32_t table_width,
                 const int32_t* lengths,
                 float* partials, float* lse,
                 int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                 int32_t splits, int32_t tokens_per_split, int32_t tile_tokens,
                 double scale, pd_stream_t stream);

/* Stable LSE merge; replaces _lse_merge (matched_splitkv.py:101-127) as
 * launched by matched_decode (:147-149).  Writes out bf16 [batch, num_heads,
 * head_dim].  lse_lanes is the plan's lane count, a power of two in [1, 64]
 * no larger than the next power of two of splits.  It sets the float32
 * summation order of the log-sum, as in the reference: lane j sums splits
 * j, j + lse_lanes, ... in order, then a halving tree adds the lanes. */
int pd_lse_merge(const float* partials, const float* lse, void* out,
                 int32_t batch, int32_t num_heads, int32_t head_dim, int32_t splits,
                 int32_t lse_lanes, pd_stream_t stream);

/* int32 counters per (sequence, kv head) in pd_matched_decode's `counters`. */
#define PD_FUSED_COUNTERS_PER_GROUP 128

/* Matched split-KV decode: the partition of pd_partition plus the LSE merge of
 * pd_lse_merge, bit-identical to pd_partition followed by pd_lse_merge.
 * Replaces the two launches of matched_decode (matched_splitkv.py:142-149).
 * Writes partials, lse and out bf16 [batch, num_heads, head_dim].  The merge
 * sums with the plan's lse_lanes, min(next_pow2(splits), 32 if
 * head_dim % 128 == 0 else 16).
 * With `counters` (non-NULL) it is one fused launch.  With splits of one tile
 * (tokens_per_split == tile_tokens) the merge of each GQA group is shared by
 * the last wavefront to finish each quarter of the head_dim columns;
 * otherwise the last workgroup of each (sequence, kv head) merges the whole
 * group.  `counters` is int32 [batch * num_kv_heads *
 * PD_FUSED_COUNTERS_PER_GROUP] (four counters per group, each on a 128-byte
 * line), all zero before the first call; every completed call leaves it all
 * zero again, so the launch can be replayed from a graph without a reset.
 * Calls that share `counters` must not run concurrently.  The partials are
 * published with device-scope stores and read with device-scope loads, so the
 * merge may run on any XCD.
 * With counters NULL it runs the partition and the merge as two launches,
 * except for a plan of one split of more than one tile (splits == 1,
 * tokens_per_split > tile_tokens): the merge of one split weighs it by exactly
 * 1, so the partition writes out = bf16(partial) itself (-0 as +0, 0 for an
 * empty sequence) and nothing else is launched. */
int pd_matched_decode(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                      const void* k, const void* v,
                      const int32_t* table, int64_t table_stride_b, int32_t table_width,
                      const int32_t* lengths,
                      float* partials, float* lse, int32_t* counters, void* out,
                      int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                      int32_t splits, int32_t tokens_per_split, int32_t tile_tokens,
                      double scale, pd_stream_t stream);

/* Bytes of the static device scratch of pd_matched_decode_noalloc. */
#define PD_NOALLOC_SCRATCH_BYTES (16 << 20)

/* Allocation-free matched split-KV decode.  This entry point has no
 * counterpart in the reference: it is for callers that cannot allocate device
 * memory or pass a workspace (code under hipGraph capture, tight serving
 * loops, harnesses that forbid hipMalloc).  Same arguments, output and
 * results (bit for bit) as pd_matched_decode without its partials, lse and
 * counters: the split workspace lives in a static device array of
 * PD_NOALLOC_SCRATCH_BYTES per GPU, held until the process ends, so
 * batch * num_heads * splits * (head_dim + 1) * 4 bytes (plus 256 for
 * alignment) must fit in it, or PD_EINVAL is returned.  It calls no
 * hipMalloc, hipFree or allocating library routine.  Every call on one GPU
 * shares that GPU's scratch, so calls that overlap on one GPU (two streams,
 * two threads) race; calls ordered on one stream do not. */
int pd_matched_decode_noalloc(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                              const void* k, const void* v,
                              const int32_t* table, int64_t table_stride_b, int32_t table_width,
                              const int32_t* lengths, void* out,
                              int32_t batch, int32_t num_heads, int32_t num_kv_heads,
                              int32_t head_dim, int32_t splits, int32_t tokens_per_split,
                              int32_t tile_tokens, double scale, pd_stream_t stream);

/* Base decode: FP32 online softmax over the whole context with FP32
 * probabilities, out = acc / denom (0 for an empty row), for every query head.
 * One workgroup per (kv head, sequence) serves the kv head's query heads (16 at
 * a time), so K/V is read once per kv head; at head_dim 64, one workgroup
 * serves four adjacent kv heads when num_kv_heads is a multiple of 4 and they
 * have at most 4 query heads each, else two when num_kv_heads is even and they
 * have at most 8 (a token's rows of those heads are one contiguous read).
 * Replaces _base (kernels.py:10-41) as launched by paged_decode
 * (runtime.py:109).  Writes out rows [0, batch). */
int pd_base(const void* q, int64_t q_stride_b, int64_t q_stride_h,
            const void* k, const void* v,
            const int32_t* table, int64_t table_stride_b, int32_t table_width,
            const int32_t* lengths,
            void* out, int32_t batch, int32_t num_heads, int32_t num_kv_heads,
            int32_t head_dim, double scale, pd_stream_t stream);

/* Fixed-size split-K partition: unnormalized (m, l, acc) per partition of
 * partition_size tokens, m in scaled units, every partition written (empty ones
 * as m = -inf, l = 0, acc = 0).  When the device has at least as many CUs as
 * pd_base has workgroups (one per kv head group and sequence), those
 * workgroups each walk their sequence's context and write every partition as
 * they pass it; with fewer, one workgroup runs per partition, as in the
 * reference's grid.  Both write the same bits.  Replaces _split
 * (kernels.py:44-80) as launched by paged_decode (runtime.py:111-113).
 * maxima/denoms f32 [batch, num_heads, partitions], accums f32 [batch,
 * num_heads, partitions, D] (16-byte aligned); the row stride of all three is
 * `partitions`; partition_size a positive multiple of 16384 / head_dim;
 * partitions * partition_size < 2^31. */
int pd_split_fixed(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                   const void* k, const void* v,
                   const int32_t* table, int64_t table_stride_b, int32_t table_width,
                   const int32_t* lengths,
                   float* maxima, float* denoms, float* accums,
                   int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                   int32_t partitions, int32_t partition_size, double scale,
                   pd_stream_t stream);

/* m/l/acc merge; replaces _merge (kernels.py:83-100) as launched by
 * paged_decode (runtime.py:114-116): M = max m_p (-inf -> 0), f_p =
 * exp(m_p - M), out = sum f_p acc_p / sum f_p l_p (a zero total divides by
 * 1), the sums in partition order.  Writes out rows [0, batch). */
int pd_ml_merge(const float* maxima, const float* denoms, const float* accums, void* out,
                int32_t batch, int32_t num_heads, int32_t head_dim, int32_t partitions,
                pd_stream_t stream);

/* The reference's fixed-split backend in one call (_split + _merge,
 * runtime.py:111-116): the workspace as pd_split_fixed writes it, and the
 * merged output in out.  When the walks fill the device, the walking
 * workgroups merge their sequence's partitions as they complete them (from
 * the last to the first, with a running maximum: the same formula as
 * pd_ml_merge in another order and float32 rounding) and write out directly,
 * in one launch; otherwise one workgroup runs per partition and a merge
 * kernel with the walk's order and arithmetic follows.  Both grids write the
 * same workspace and output bits. */
int pd_split_decode(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                    const void* k, const void* v,
                    const int32_t* table, int64_t table_stride_b, int32_t table_width,
                    const int32_t* lengths,
                    float* maxima, float* denoms, float* accums, void* out,
                    int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                    int32_t partitions, int32_t partition_size, double scale,
                    pd_stream_t stream);

/* Small-batch split of the base and fixed-split protocols; no counterpart in
 * the reference, whose _base and _split grids already spread a sequence over
 * (query heads[, partitions]) programs (runtime.py:109-113).  pd_base and
 * pd_split_fixed walk each sequence in one workgroup per kv head group, so a
 * batch of fewer walks than half of sm_count leaves CUs idle; the walks are
 * counted for `batch` rounded up to a power of two.  For such a batch this
 * returns a cut of a table of `table_width` pages into *chunks >= 2 partitions
 * of *chunk_tokens tokens (a multiple of 16384 / head_dim; about sm_count /
 * walks of them, at most 128): run pd_split_fixed(partitions, partition_size =
 * *chunk_tokens) and pd_ml_merge over partitions = ceil(w * 256 /
 * *chunk_tokens) for a call whose table has w <= table_width pages.  That
 * computes the same attention as pd_base or the 1024-token pd_split_fixed with
 * other float32 rounding.  Partitions past a sequence's length are empty and
 * leave the merge's bits unchanged, and each sequence's partitions are its own,
 * so a sequence's output does not depend on w, on the other sequences, or on
 * empty sequences padding the batch below its next power of two (a graph
 * bucket), as long as table_width is the same.  Otherwise *chunks = 1 and
 * *chunk_tokens = table_width * 256: run the backend itself.  Host only. */
int pd_plan_chunks(int32_t batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                   int32_t table_width, int32_t sm_count, int32_t* chunks,
                   int32_t* chunk_tokens);

/* Size of a chunk workspace for pd_plan_chunks (no counterpart in the
 * reference): *rows = the largest batch * num_heads * chunks it returns for any
 * batch <= max_batch and any table width (0 if none is cut), so maxima and
 * denoms of *rows floats and accums of *rows * head_dim floats serve every
 * call (batch <= max_batch, any w).  Host only. */
int pd_chunk_rows(int32_t max_batch, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                  int32_t sm_count, int64_t* rows);

/* KV-cache write of token rows through a flat slot mapping; replaces the
 * store_kvcache Triton kernel of the nano-vLLM overlay
 * (overlays/nano-vllm/nanovllm/layers/attention.py:10-38).  For token i with
 * slot = slot_mapping[i] >= 0, copies row_elems (= num_kv_heads * head_dim)
 * bf16 of key + i*key_stride to k_cache + slot*row_elems, and the same for
 * value/v_cache; slot -1 (a padded graph entry) is skipped.  Rows, caches and
 * strides must be 16-byte aligned (strides multiples of 8 elements, at least
 * row_elems).  Contents are trusted: slots must lie inside the caches. */
int pd_store_kv(const void* key, int64_t key_stride, const void* value, int64_t value_stride,
                void* k_cache, void* v_cache, const int32_t* slot_mapping, int64_t num_tokens,
                int32_t row_elems, pd_stream_t stream);

/* KV-cache write of a [batch, num_kv_heads, steps, head_dim] chunk into
 * 256-slot pages; replaces the index_copy_ of PagedHybridCache.update
 * (src/paged_decode/hybrid.py:63-72).  Element (b, h, s, d) goes to page
 * table[b, positions[s] / 256], slot positions[s] % 256, kv head h.  `positions`
 * is int64 [steps]; k_pages and v_pages hold num_pages pages each.  A negative
 * position, a page index at or past table_width, or a table entry outside
 * [0, num_pages) skips the row (the reference's index_copy_ rejects such an
 * index; here nothing is written outside the pool).  head_dim in
 * {64, 128, 256}; strides in elements, multiples of 8; pointers 16-byte
 * aligned. */
int pd_store_kv_pages(const void* key, int64_t key_stride_b, int64_t key_stride_h,
                      int64_t key_stride_s, const void* value, int64_t value_stride_b,
                      int64_t value_stride_h, int64_t value_stride_s, void* k_pages,
                      void* v_pages, int64_t num_pages, const int32_t* table,
                      int64_t table_stride_b,
                      int32_t table_width, const int64_t* positions, int32_t batch,
                      int32_t num_kv_heads, int32_t steps, int32_t head_dim, pd_stream_t stream);

/* Causal prefill attention: new token t of a sequence attends to keys
 * 0 .. nk - nq + t of it (nq new tokens, nk keys), in float32 up to the bf16
 * output.  Strides are host arrays {batch, token, head} in elements,
 * non-negative multiples of 8, tensors 16-byte aligned with a contiguous head.
 *   packed   (cu_q, cu_k int32 [num_seqs + 1] on the device): sequence i owns
 *            rows cu_q[i] .. cu_q[i+1] of q and out, [total_q, Hq, D], and rows
 *            cu_k[i] .. of k and v, [total_k, Hkv, D]; batch strides unused;
 *   paged    (packed, with a table): its keys are tokens 0 .. cu_k[i+1]-cu_k[i]
 *            of pages table[i, t / page_size]; k and v [num_pages, page_size,
 *            Hkv, D], page_size a multiple of 64 (of 32 at head_dim 256);
 *   batched  (no cu): num_seqs sequences of seq_len new tokens and no prefix.
 * Rows past total_q / total_k, pages outside [0, num_pages) and entries past
 * table_width are never read (their keys and values are zeros).
 * splits > 1 cuts the keys of every row into that many spans whose partials
 * (part_o float32 [splits, total_q, Hq, D], part_ml [splits, total_q, Hq, 2])
 * a second launch merges. */
int pd_prefill(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
               const void* v, const int64_t* v_strides, void* out, const int64_t* out_strides,
               const int32_t* cu_q, const int32_t* cu_k, int32_t num_seqs, int32_t seq_len,
               int64_t total_q, int64_t total_k, const int32_t* table, int64_t table_stride_b,
               int32_t table_width, int32_t page_size, int64_t num_pages, int32_t num_heads,
               int32_t num_kv_heads, int32_t head_dim, double scale, int32_t splits,
               float* part_o, float* part_ml, pd_stream_t stream);

/* pd_prefill of packed or paged sequences whose metadata are checked on the
 * device, and pd_store_kv (above) that checks them for the pd_prefill behind it.
 * verdicts: int32 [PD_CHECK_WORDS] of pinned host memory, zeroed by the caller
 * and kept until pd_check_wait returns, which waits for the check, not for the
 * kernel, and gives what was found:
 *   PD_CHECK_ODD      sequences are not rows of the tensors in order, or one of
 *                     new tokens has no keys or a page in [-num_pages, -1];
 *   PD_CHECK_OUTSIDE  a sequence has more keys than its table's entries hold,
 *                     or any other page outside the pool. */
#define PD_CHECK_WORDS 64
#define PD_CHECK_ODD 1
#define PD_CHECK_OUTSIDE 2
int pd_prefill_checked(const void* q, const int64_t* q_strides, const void* k,
                       const int64_t* k_strides, const void* v, const int64_t* v_strides, void* out,
                       const int64_t* out_strides, const int32_t* cu_q, const int32_t* cu_k,
                       int32_t num_seqs, int32_t seq_len, int64_t total_q, int64_t total_k,
                       const int32_t* table, int64_t table_stride_b, int32_t table_width,
                       int32_t page_size, int64_t num_pages, int32_t num_heads,
                       int32_t num_kv_heads, int32_t head_dim, double scale, int32_t splits,
                       float* part_o, float* part_ml, int32_t* verdicts, pd_stream_t stream);
int pd_store_kv_checked(const void* key, int64_t key_stride, const void* value,
                        int64_t value_stride, void* k_cache, void* v_cache,
                        const int32_t* slot_mapping, int64_t num_tokens, int32_t row_elems,
                        const int32_t* cu_q, const int32_t* cu_k, int32_t num_seqs, int64_t total_q,
                        int64_t total_k, const int32_t* table, int64_t table_stride_b,
                        int32_t table_width, int32_t page_size, int64_t num_pages,
                        int32_t* verdicts, pd_stream_t stream);
int pd_check_wait(const int32_t* verdicts, pd_stream_t stream, int32_t* found);

/* The decoder layer between its matrix products.  bf16 tensors are contiguous
 * and 16-byte aligned unless strides are given; arithmetic is float32. */

/* x [rows, dim] += y (y may be null), out = x rms(x)^-1 (1 + weight). */
int pd_add_rms_norm(void* x, const void* y, const void* weight, void* out, int64_t rows,
                    int32_t dim, double eps, pd_stream_t stream);

/* out = o rms(o)^-1 weight silu(z) per row of dim (64 or 128); o float32. */
int pd_gated_norm(const float* o, const void* z, const void* weight, void* out, int64_t rows,
                  int32_t dim, double eps, pd_stream_t stream);

/* out = silu(gate) up; out may be gate. */
int pd_silu_mul(const void* gate, const void* up, void* out, int64_t elems, pd_stream_t stream);

/* out = x sigmoid(gate), gate's rows gate_stride elements apart. */
int pd_sigmoid_gate(const void* x, const void* gate, int64_t gate_stride, void* out, int64_t rows,
                    int32_t cols, pd_stream_t stream);

/* Gated delta rule inputs of x [batch, steps, C], C = 2 hk dk + hv dv channels
 * (queries, keys, values): causal convolution with taps [C, 4], silu, unit
 * query (times dk^-1/2) and key heads -> act float32 [batch, steps, C].
 * conv_state [batch, C, 4] receives the last four inputs; with has_prev (at
 * most 16 steps) it holds the four before them. */
int pd_conv(const void* x, const void* taps, void* conv_state, float* act, int32_t batch,
            int32_t steps, int32_t hk, int32_t hv, int32_t dk, int32_t dv, int32_t has_prev,
            pd_stream_t stream);

/* gates float32 [rows, hv, 2] = (-exp(a_log) softplus(h wa^T + dt_bias),
 * sigmoid(h wb^T)): the log decay and beta of h [rows, dim]. */
int pd_gates(const void* h, const void* wa, const void* wb, const void* a_log, const void* dt_bias,
             float* gates, int64_t rows, int32_t dim, int32_t hv, pd_stream_t stream);

/* S = decay S; S += k (beta (v - S^T k))^T; out = S^T q per value head and
 * token, one after the other; state float32 [batch, hv, dk, dv], read with has_prev, written;
 * out float32 [batch, steps, hv, dv]. */
int pd_delta_rule(const float* act, const float* gates, float* state, float* out, int32_t batch,
                  int32_t steps, int32_t hk, int32_t hv, int32_t dk, int32_t dv, int32_t has_prev,
                  pd_stream_t stream);

/* The same in chunks of 64 tokens; workspace of pd_delta_workspace floats. */
int pd_delta_chunks(const float* act, const float* gates, float* state, float* out,
                    float* workspace, int32_t batch, int32_t steps, int32_t hk, int32_t hv,
                    int32_t dk, int32_t dv, int32_t has_prev, pd_stream_t stream);
int pd_delta_workspace(int32_t batch, int32_t steps, int32_t hv, int32_t dk, int32_t dv,
                       int64_t* floats);

/* table float32 [steps, half, 2]: cos and sin of positions x inv_freq. */
int pd_rope_table(const int64_t* positions, const void* inv_freq, int32_t is_bf16, float* table,
                  int32_t steps, int32_t half, pd_stream_t stream);

/* Query and key heads normed (weights as 1 + w) and rotated (2 half leading
 * elements), keys and values written to their page slots as
 * pd_store_kv_pages does.  q [batch, steps, Hq, 2, D] (query, gate), k and v
 * [batch, steps, Hkv, D] -> q_out [batch, steps, Hq, D], k_out (may be null). */
int pd_qk_rope(const void* q, const void* k, const void* v, const void* q_weight,
               const void* k_weight, const float* rope, void* q_out, void* k_out, void* k_pages,
               void* v_pages, int64_t num_pages, const int32_t* table, int64_t table_stride_b,
               int32_t table_width, const int64_t* positions, int32_t batch, int32_t steps,
               int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, int32_t half, double eps,
               pd_stream_t stream);

/* Products of x [rows, dim] with `count` <= 4 weight matrices [features[i],
 * dim], dim a multiple of 64, features of 4; the arrays are host arrays.  form
 * 0: outs[i] = x weights[i]^T; form 1 (two matrices of one size): outs[0] =
 * silu(x weights[0]^T) (x weights[1]^T).  tile: 128 or 256 weight rows a
 * workgroup. */
int pd_linears(const void* x, int32_t rows, int32_t dim, int32_t count, const void* const* weights,
               const int32_t* features, void* const* outs, int32_t form, int32_t tile,
               pd_stream_t stream);

/* One token per sequence: products of 1 to 16 rows whose norms, gates,
 * convolution and residual run in the same launch.  dim (the input features)
 * is a multiple of 64; weights are bf16 [features, dim]. */

/* h = x rms(x)^-1 (1 + norm); outs[i] = h weights[i]^T, bf16 [rows,
 * features[i]].  With taps, outs[0] is instead float32 silu of the causal
 * convolution of its channels, whose conv_state [rows, features[0], 4] moves
 * one step (from zeros without has_prev).  The three arrays are host arrays of
 * `count` <= 4. */
int pd_norm_linears(const void* x, const void* norm, double eps, int32_t rows, int32_t dim,
                    int32_t count, const void* const* weights, const int32_t* features,
                    void* const* outs, const void* taps, void* conv_state, int32_t has_prev,
                    pd_stream_t stream);

/* out = silu(h gate^T) (h up^T), h as above. */
int pd_norm_gate_up(const void* x, const void* norm, double eps, int32_t rows, int32_t dim,
                    const void* gate, const void* up, void* out, int32_t features,
                    pd_stream_t stream);

/* x [rows, features] += h weight^T; with gate (rows of heads [dim / head_dim,
 * 2, head_dim], pointing at the second half of the first), h sigmoid(gate) in
 * the place of h. */
int pd_linear_add(const void* h, const void* gate, int32_t head_dim, const void* weight, void* x,
                  int32_t rows, int32_t dim, int32_t features, pd_stream_t stream);

/* One token of pd_delta_rule and pd_gated_norm from act float32 [batch, C]
 * (silu of the convolution; heads are normed here): out bf16 [batch, hv, dv]. */
int pd_delta_step(const float* act, const void* a, const void* b, const void* a_log,
                  const void* dt_bias, const void* z, const void* norm, double eps, float* state,
                  void* out, int32_t batch, int32_t hk, int32_t hv, int32_t dk, int32_t dv,
                  int32_t has_prev, pd_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* PAGED_DECODE_H_ */
