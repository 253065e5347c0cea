"""ctypes binding of libpaged_decode.so (declared in include/paged_decode.h).

torch is imported before the library is opened so that the library's
``libamdhip64.so.7`` dependency resolves to the HIP runtime torch already
loaded: streams, graphs and device pointers are then shared with torch.

There is no fallback: if the library is missing, every entry point raises.
"""
import ctypes
import os

import torch  # noqa: F401  (must precede the CDLL load, see module docstring)

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libpaged_decode.so")

PD_OK, PD_EINVAL, PD_ELAUNCH = 0, 1, 2

_i32, _i64, _dbl, _vp = ctypes.c_int32, ctypes.c_int64, ctypes.c_double, ctypes.c_void_p


class Plan(ctypes.Structure):
    _fields_ = [("splits", _i32), ("tile_tokens", _i32), ("tokens_per_split", _i32),
                ("table_capacity_tokens", _i32), ("lse_lanes", _i32), ("sm_count", _i32),
                ("is_explicit", _i32)]


# Exported symbol -> argtypes.  Kept in the order of include/paged_decode.h.
SIGNATURES = {
    "pd_last_error": [],
    "pd_abi_version": [],
    "pd_make_plan": [_i32, _i32, _i32, _i32, _i32, _i32, _i32, ctypes.POINTER(Plan)],
    "pd_validate_metadata": [_vp, _i64, _i32, _vp, _i32, _i64, _i32],
    "pd_partition": [_vp, _i64, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _vp,
                     _i32, _i32, _i32, _i32, _i32, _i32, _i32, _dbl, _vp],
    "pd_lse_merge": [_vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _vp],
    "pd_matched_decode": [_vp, _i64, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _vp, _vp, _vp,
                          _i32, _i32, _i32, _i32, _i32, _i32, _i32, _dbl, _vp],
    "pd_matched_decode_noalloc": [_vp, _i64, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp,
                                  _i32, _i32, _i32, _i32, _i32, _i32, _i32, _dbl, _vp],
    "pd_base": [_vp, _i64, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _i32, _i32, _i32, _i32,
                _dbl, _vp],
    "pd_split_fixed": [_vp, _i64, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _vp, _vp,
                       _i32, _i32, _i32, _i32, _i32, _i32, _dbl, _vp],
    "pd_ml_merge": [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _vp],
    "pd_split_decode": [_vp, _i64, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _vp, _vp, _vp,
                        _i32, _i32, _i32, _i32, _i32, _i32, _dbl, _vp],
    "pd_plan_chunks": [_i32, _i32, _i32, _i32, _i32, _i32, ctypes.POINTER(_i32),
                       ctypes.POINTER(_i32)],
    "pd_chunk_rows": [_i32, _i32, _i32, _i32, _i32, ctypes.POINTER(_i64)],
    "pd_store_kv": [_vp, _i64, _vp, _i64, _vp, _vp, _vp, _i64, _i32, _vp],
    "pd_store_kv_pages": [_vp, _i64, _i64, _i64, _vp, _i64, _i64, _i64, _vp, _vp, _i64, _vp, _i64,
                          _i32, _vp, _i32, _i32, _i32, _i32, _vp],
    "pd_prefill": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i32, _i32, _i64, _i64, _vp,
                   _i64, _i32, _i32, _i64, _i32, _i32, _i32, _dbl, _i32, _vp, _vp, _vp],
    "pd_prefill_checked": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i32, _i32, _i64, _i64,
                           _vp, _i64, _i32, _i32, _i64, _i32, _i32, _i32, _dbl, _i32, _vp, _vp, _vp,
                           _vp],
    "pd_store_kv_checked": [_vp, _i64, _vp, _i64, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _i32, _i64,
                            _i64, _vp, _i64, _i32, _i32, _i64, _vp, _vp],
    "pd_check_wait": [_vp, _vp, ctypes.POINTER(_i32)],
    "pd_add_rms_norm": [_vp, _vp, _vp, _vp, _i64, _i32, _dbl, _vp],
    "pd_gated_norm": [_vp, _vp, _vp, _vp, _i64, _i32, _dbl, _vp],
    "pd_silu_mul": [_vp, _vp, _vp, _i64, _vp],
    "pd_sigmoid_gate": [_vp, _vp, _i64, _vp, _i64, _i32, _vp],
    "pd_conv": [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    "pd_gates": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _vp],
    "pd_delta_rule": [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    "pd_delta_chunks": [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    "pd_delta_workspace": [_i32, _i32, _i32, _i32, _i32, ctypes.POINTER(_i64)],
    "pd_rope_table": [_vp, _vp, _i32, _vp, _i32, _i32, _vp],
    "pd_qk_rope": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _vp, _i64, _i32, _vp,
                   _i32, _i32, _i32, _i32, _i32, _i32, _dbl, _vp],
    "pd_linears": [_vp, _i32, _i32, _i32, _vp, _vp, _vp, _i32, _i32, _vp],
    "pd_norm_linears": [_vp, _vp, _dbl, _i32, _i32, _i32, _vp, _vp, _vp, _vp, _vp, _i32, _vp],
    "pd_norm_gate_up": [_vp, _vp, _dbl, _i32, _i32, _vp, _vp, _vp, _i32, _vp],
    "pd_linear_add": [_vp, _vp, _i32, _vp, _vp, _i32, _i32, _i32, _vp],
    "pd_delta_step": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _dbl, _vp, _vp, _i32, _i32, _i32, _i32,
                      _i32, _i32, _vp],
}

_lib = None


def load_library(path):
    """A ctypes handle of a libpaged_decode.so build at ``path``, with the signatures set.
    Every entry point below takes ``library=`` to run through such a handle instead of
    the package's own build (an A/B of two builds in one process)."""
    if not os.path.exists(path):
        raise RuntimeError(
            f"{path} is not built: run `make -C paged-decode-lab_amd/csrc` "
            "(or __graft_entry__.build()); there is no fallback implementation")
    handle = ctypes.CDLL(path)
    for name, argtypes in SIGNATURES.items():
        try:
            fn = getattr(handle, name)
        except AttributeError:
            if path == LIB_PATH:
                raise
            continue  # an older build compared in an A/B run: calls to it raise
        fn.argtypes = argtypes
        fn.restype = ctypes.c_char_p if name == "pd_last_error" else ctypes.c_int
    return handle


def lib():
    """The loaded library; raises RuntimeError when it has not been built."""
    global _lib
    if _lib is None:
        _lib = load_library(LIB_PATH)
    return _lib


def check(status, library=None):
    if status == PD_OK:
        return
    message = (library or lib()).pd_last_error().decode()
    if status == PD_EINVAL:
        raise ValueError(message)
    raise RuntimeError(message)


def make_plan(max_batch, num_heads, num_kv_heads, head_dim, max_context_len, sm_count,
              num_splits):
    plan = Plan()
    check(lib().pd_make_plan(max_batch, num_heads, num_kv_heads, head_dim, max_context_len,
                             sm_count, num_splits, ctypes.byref(plan)))
    return plan


def validate_metadata(table, lengths, num_pages, max_context_len):
    """``table``/``lengths``: contiguous int32 CPU tensors."""
    check(lib().pd_validate_metadata(table.data_ptr(), table.stride(0) if table.dim() else 0,
                                     table.shape[1], lengths.data_ptr(), lengths.shape[0],
                                     num_pages, max_context_len))


# torch's raw lookup of the current stream returns the handle without building a Stream
# object (a few microseconds of host time per launch); current_stream is the fallback.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_handle(device):
    if _raw_stream is not None and device.index is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


def partition(q, k, v, tables, lengths, partials, lse, num_kv_heads, splits, tokens_per_split,
              tile_tokens, scale, library=None):
    b, h, d = q.shape
    L = library or lib()
    check(L.pd_partition(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), v.data_ptr(),
                         tables.data_ptr(), tables.stride(0), tables.shape[1],
                         lengths.data_ptr(), partials.data_ptr(), lse.data_ptr(), b, h,
                         num_kv_heads, d, splits,
                         tokens_per_split, tile_tokens, scale, stream_handle(q.device)), L)


def matched_decode(q, k, v, tables, lengths, partials, lse, counters, out, num_kv_heads, splits,
                   tokens_per_split, tile_tokens, scale, library=None):
    """pd_matched_decode: the fused launch with ``counters``; without (None) the partition
    and the LSE merge, or the partition alone for a plan of one multi-tile split."""
    b, h, d = q.shape
    L = library or lib()
    check(L.pd_matched_decode(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(),
                              v.data_ptr(), tables.data_ptr(), tables.stride(0),
                              tables.shape[1], lengths.data_ptr(), partials.data_ptr(),
                              lse.data_ptr(),
                              None if counters is None else counters.data_ptr(),
                              out.data_ptr(), b, h, num_kv_heads, d,
                              splits, tokens_per_split, tile_tokens, scale,
                              stream_handle(q.device)), L)


def matched_decode_noalloc(q, k, v, tables, lengths, out, num_kv_heads, splits,
                           tokens_per_split, tile_tokens, scale, library=None):
    """pd_matched_decode with the split workspace in the library's static device scratch."""
    b, h, d = q.shape
    L = library or lib()
    check(L.pd_matched_decode_noalloc(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(),
                                      v.data_ptr(), tables.data_ptr(), tables.stride(0),
                                      tables.shape[1], lengths.data_ptr(), out.data_ptr(), b,
                                      h, num_kv_heads, d, splits, tokens_per_split,
                                      tile_tokens, scale, stream_handle(q.device)), L)


def lse_merge(partials, lse, out, lse_lanes, library=None):
    b, h, splits, d = partials.shape
    L = library or lib()
    check(L.pd_lse_merge(partials.data_ptr(), lse.data_ptr(), out.data_ptr(), b, h, d, splits,
                         lse_lanes, stream_handle(partials.device)), L)


def base(q, k, v, tables, lengths, out, num_kv_heads, scale, library=None):
    b, h, d = q.shape
    L = library or lib()
    check(L.pd_base(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), v.data_ptr(),
                    tables.data_ptr(), tables.stride(0), tables.shape[1], lengths.data_ptr(),
                    out.data_ptr(),
                    b, h, num_kv_heads, d, scale, stream_handle(q.device)), L)


def split_fixed(q, k, v, tables, lengths, maxima, denoms, accums, num_kv_heads, partitions,
                partition_size, scale, library=None):
    b, h, d = q.shape
    L = library or lib()
    check(L.pd_split_fixed(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), v.data_ptr(),
                           tables.data_ptr(), tables.stride(0), tables.shape[1],
                           lengths.data_ptr(), maxima.data_ptr(), denoms.data_ptr(),
                           accums.data_ptr(), b, h, num_kv_heads, d, partitions, partition_size,
                           scale, stream_handle(q.device)), L)


def ml_merge(maxima, denoms, accums, out, batch, library=None):
    _, h, parts, d = accums.shape
    L = library or lib()
    check(L.pd_ml_merge(maxima.data_ptr(), denoms.data_ptr(), accums.data_ptr(),
                        out.data_ptr(), batch, h, d, parts, stream_handle(out.device)), L)


def split_decode(q, k, v, tables, lengths, maxima, denoms, accums, out, num_kv_heads,
                 partitions, partition_size, scale, library=None):
    """pd_split_decode: the fixed-split partitions and their merge into ``out``."""
    b, h, d = q.shape
    L = library or lib()
    check(L.pd_split_decode(q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), v.data_ptr(),
                            tables.data_ptr(), tables.stride(0), tables.shape[1],
                            lengths.data_ptr(), maxima.data_ptr(), denoms.data_ptr(),
                            accums.data_ptr(), out.data_ptr(), b, h, num_kv_heads, d,
                            partitions, partition_size, scale, stream_handle(q.device)), L)


def plan_chunks(batch, num_heads, num_kv_heads, head_dim, table_width, sm_count):
    """(chunks, chunk_tokens) of pd_plan_chunks: the small-batch split of the base and
    fixed-split protocols, chunks == 1 when the backend runs as it is."""
    chunks, tokens = _i32(0), _i32(0)
    check(lib().pd_plan_chunks(batch, num_heads, num_kv_heads, head_dim, table_width, sm_count,
                               ctypes.byref(chunks), ctypes.byref(tokens)))
    return chunks.value, tokens.value


def chunk_rows(max_batch, num_heads, num_kv_heads, head_dim, sm_count):
    """Chunk-workspace rows that serve every call of pd_plan_chunks (pd_chunk_rows)."""
    rows = _i64(0)
    check(lib().pd_chunk_rows(max_batch, num_heads, num_kv_heads, head_dim, sm_count,
                              ctypes.byref(rows)))
    return rows.value


def store_kv(key, value, k_cache, v_cache, slot_mapping):
    """key/value [N, Hkv, D] (rows 16-byte aligned); caches [..., Hkv, D] flat over slots."""
    n, hkv, d = key.shape
    check(lib().pd_store_kv(key.data_ptr(), key.stride(0), value.data_ptr(), value.stride(0),
                            k_cache.data_ptr(), v_cache.data_ptr(), slot_mapping.data_ptr(), n,
                            hkv * d, stream_handle(key.device)))


def store_kv_checked(key, value, k_cache, v_cache, slot_mapping, metadata):
    """store_kv that checks the packed prefill behind it: ``metadata`` is its (cu_q, cu_k,
    sequences, total_q, total_k, tables or None, page_size, num_pages, verdicts)."""
    n, hkv, d = key.shape
    cu_q, cu_k, seqs, total_q, total_k, tables, page_size, num_pages, verdicts = metadata
    check(lib().pd_store_kv_checked(
        key.data_ptr(), key.stride(0), value.data_ptr(), value.stride(0), k_cache.data_ptr(),
        v_cache.data_ptr(), slot_mapping.data_ptr(), n, hkv * d, cu_q.data_ptr(), cu_k.data_ptr(),
        seqs, total_q, total_k, None if tables is None else tables.data_ptr(),
        0 if tables is None else tables.stride(0), 0 if tables is None else tables.shape[1],
        page_size, num_pages, verdicts.data_ptr(), stream_handle(key.device)))


def store_kv_pages(key, value, k_pages, v_pages, tables, positions):
    """key/value [B, Hkv, S, D]; pages [P, 256, Hkv, D]; tables int32 [B, W]; positions int64 [S]."""
    b, hkv, steps, d = key.shape
    check(lib().pd_store_kv_pages(key.data_ptr(), key.stride(0), key.stride(1), key.stride(2),
                                  value.data_ptr(), value.stride(0), value.stride(1),
                                  value.stride(2), k_pages.data_ptr(), v_pages.data_ptr(),
                                  k_pages.shape[0], tables.data_ptr(), tables.stride(0),
                                  tables.shape[1],
                                  positions.data_ptr(), b, hkv, steps, d,
                                  stream_handle(key.device)))


_Strides = _i64 * 3


def prefill(q, q_strides, k, k_strides, v, v_strides, out, out_strides, cu_q, cu_k, num_seqs,
            seq_len, total_q, total_k, tables, page_size, num_pages, heads, kv_heads, head_dim,
            scale, splits, part_o, part_ml, verdicts=None):
    """pd_prefill, or with verdicts (int32 [CHECK_WORDS] pinned, zero) pd_prefill_checked;
    strides are (batch, token, head) in elements."""
    args = (q.data_ptr(), _Strides(*q_strides), k.data_ptr(), _Strides(*k_strides), v.data_ptr(),
            _Strides(*v_strides), out.data_ptr(), _Strides(*out_strides),
            None if cu_q is None else cu_q.data_ptr(), None if cu_k is None else cu_k.data_ptr(),
            num_seqs, seq_len, total_q, total_k, None if tables is None else tables.data_ptr(),
            0 if tables is None else tables.stride(0), 0 if tables is None else tables.shape[1],
            page_size, num_pages, heads, kv_heads, head_dim, scale, splits,
            None if part_o is None else part_o.data_ptr(),
            None if part_ml is None else part_ml.data_ptr())
    if verdicts is None:
        check(lib().pd_prefill(*args, stream_handle(q.device)))
    else:
        check(lib().pd_prefill_checked(*args, verdicts.data_ptr(), stream_handle(q.device)))


CHECK_WORDS, CHECK_ODD, CHECK_OUTSIDE = 64, 1, 2


def check_wait(verdicts, device):
    """The bits that a checked prefill found, launched on the current stream of ``device``."""
    found = _i32(0)
    check(lib().pd_check_wait(verdicts.data_ptr(), stream_handle(device), ctypes.byref(found)))
    return found.value


def add_rms_norm(x, y, weight, out, eps):
    """x [N, H] += y (or y None), out = x rms(x)^-1 (1 + weight)."""
    check(lib().pd_add_rms_norm(x.data_ptr(), None if y is None else y.data_ptr(),
                                weight.data_ptr(), out.data_ptr(), x.shape[0], x.shape[1], eps,
                                stream_handle(x.device)))


def gated_norm(o, z, weight, out, rows, dim, eps):
    """out = o rms(o)^-1 weight silu(z) over `rows` rows of `dim`; o float32."""
    check(lib().pd_gated_norm(o.data_ptr(), z.data_ptr(), weight.data_ptr(), out.data_ptr(), rows,
                              dim, eps, stream_handle(o.device)))


def silu_mul(gate, up, out):
    check(lib().pd_silu_mul(gate.data_ptr(), up.data_ptr(), out.data_ptr(), gate.numel(),
                            stream_handle(gate.device)))


def sigmoid_gate(x, gate, out, rows, cols):
    """out = x sigmoid(gate), x and out [rows, cols], gate's rows gate.stride(0) apart."""
    check(lib().pd_sigmoid_gate(x.data_ptr(), gate.data_ptr(), gate.stride(0), out.data_ptr(), rows,
                                cols, stream_handle(x.device)))


def conv(x, taps, conv_state, act, batch, steps, hk, hv, dk, dv, has_prev):
    check(lib().pd_conv(x.data_ptr(), taps.data_ptr(), conv_state.data_ptr(), act.data_ptr(), batch,
                        steps, hk, hv, dk, dv, int(has_prev), stream_handle(x.device)))


def gates(h, wa, wb, a_log, dt_bias, out):
    """out float32 [N, hv, 2] = (log decay, beta) of h [N, dim]."""
    check(lib().pd_gates(h.data_ptr(), wa.data_ptr(), wb.data_ptr(), a_log.data_ptr(),
                         dt_bias.data_ptr(), out.data_ptr(), h.shape[0], h.shape[1], wa.shape[0],
                         stream_handle(h.device)))


def delta_workspace(batch, steps, hv, dk, dv):
    floats = _i64(0)
    check(lib().pd_delta_workspace(batch, steps, hv, dk, dv, ctypes.byref(floats)))
    return floats.value


def delta_chunks(act, gates, state, out, workspace, batch, steps, hk, hv, dk, dv, has_prev):
    check(lib().pd_delta_chunks(act.data_ptr(), gates.data_ptr(), state.data_ptr(), out.data_ptr(),
                                workspace.data_ptr(), batch, steps, hk, hv, dk, dv, int(has_prev),
                                stream_handle(act.device)))


def delta_rule(act, gates, state, out, batch, steps, hk, hv, dk, dv, has_prev):
    check(lib().pd_delta_rule(act.data_ptr(), gates.data_ptr(), state.data_ptr(), out.data_ptr(),
                              batch, steps, hk, hv, dk, dv, int(has_prev),
                              stream_handle(act.device)))


def rope_table(positions, inv_freq, table):
    """table float32 [steps, half, 2] = (cos, sin) of positions x inv_freq (bf16 or float32)."""
    check(lib().pd_rope_table(positions.data_ptr(), inv_freq.data_ptr(),
                              int(inv_freq.dtype == torch.bfloat16), table.data_ptr(),
                              table.shape[0], table.shape[1], stream_handle(table.device)))


def qk_rope(q, k, v, q_weight, k_weight, rope, q_out, k_out, k_pages, v_pages, tables, positions,
            batch, steps, hq, hkv, d, half, eps):
    check(lib().pd_qk_rope(q.data_ptr(), k.data_ptr(), v.data_ptr(), q_weight.data_ptr(),
                           k_weight.data_ptr(), rope.data_ptr(), q_out.data_ptr(),
                           None if k_out is None else k_out.data_ptr(), k_pages.data_ptr(),
                           v_pages.data_ptr(), k_pages.shape[0], tables.data_ptr(),
                           tables.stride(0), tables.shape[1], positions.data_ptr(), batch, steps,
                           hq, hkv, d, half, eps, stream_handle(q.device)))


LINEAR_STORE, LINEAR_SILU_MUL = 0, 1


def linears(x, weights, outs, form=LINEAR_STORE, tile=128):
    """outs[i] = x weights[i]^T, or outs[0] = silu(x gate^T) (x up^T); ``tile`` weight rows a
    workgroup."""
    n = len(weights)
    check(lib().pd_linears(x.data_ptr(), x.shape[0], x.shape[1], n,
                           (_vp * n)(*[w.data_ptr() for w in weights]),
                           (_i32 * n)(*[w.shape[0] for w in weights]),
                           (_vp * n)(*[outs[i % len(outs)].data_ptr() for i in range(n)]), form, tile,
                           stream_handle(x.device)))


def norm_linears(x, norm, eps, weights, outs, taps=None, conv_state=None, has_prev=False):
    """outs[i] = norm(x) weights[i]^T; with taps outs[0] (float32) is convolved."""
    n = len(weights)
    check(lib().pd_norm_linears(
        x.data_ptr(), norm.data_ptr(), eps, x.shape[0], x.shape[1], n,
        (_vp * n)(*[w.data_ptr() for w in weights]), (_i32 * n)(*[w.shape[0] for w in weights]),
        (_vp * n)(*[o.data_ptr() for o in outs]), None if taps is None else taps.data_ptr(),
        None if conv_state is None else conv_state.data_ptr(), int(has_prev),
        stream_handle(x.device)))


def norm_gate_up(x, norm, eps, gate, up, out):
    check(lib().pd_norm_gate_up(x.data_ptr(), norm.data_ptr(), eps, x.shape[0], x.shape[1],
                                gate.data_ptr(), up.data_ptr(), out.data_ptr(), gate.shape[0],
                                stream_handle(x.device)))


def linear_add(h, weight, x, gate=None, head_dim=0):
    """x += h weight^T, or (h sigmoid(gate)) weight^T."""
    check(lib().pd_linear_add(h.data_ptr(), None if gate is None else gate.data_ptr(), head_dim,
                              weight.data_ptr(), x.data_ptr(), x.shape[0], weight.shape[1],
                              weight.shape[0], stream_handle(x.device)))


def delta_step(act, a, b, a_log, dt_bias, z, norm, eps, state, out, batch, hk, hv, dk, dv, has_prev):
    check(lib().pd_delta_step(act.data_ptr(), a.data_ptr(), b.data_ptr(), a_log.data_ptr(),
                              dt_bias.data_ptr(), z.data_ptr(), norm.data_ptr(), eps,
                              state.data_ptr(), out.data_ptr(), batch, hk, hv, dk, dv,
                              int(has_prev), stream_handle(act.device)))
