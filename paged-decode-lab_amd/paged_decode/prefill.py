"""Causal prefill attention: the HIP kernel (pd_prefill) and the float32 PyTorch form.

The kernel serves what an engine on this GPU passes: bf16 tensors with head_dim 64, 128
or 256, 16-byte rows, int32 device metadata, a page size that is a whole number of key
tiles.  Everything else (other types and head dims, CPU tensors, tensors that autograd or
a functorch transform follows, odd layouts, host metadata) keeps the PyTorch form, which
materializes the scores of one sequence at a time.  An infinity or NaN in a later token's V
leaves earlier rows alone in the kernel; the PyTorch form multiplies it by their zero
probabilities, a NaN.
"""
import functools
import math
import numbers

import torch

from . import _native

HEAD_DIMS = (64, 128, 256)


def _plain(*tensors):
    """Ordinary device tensors whose memory a kernel may read: no subclass, no autograd
    or forward-mode graph to keep, no functorch wrapper, no tracer watching."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing():
        return False
    if torch.autograd.forward_ad._current_level >= 0:
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if (type(t) not in (torch.Tensor, torch.nn.Parameter) or not t.is_cuda
                or (grad and t.requires_grad)
                or torch._C._functorch.is_functorch_wrapped_tensor(t)):
            return False
    return True


def _rows_ok(t, token, head, least):
    """bf16 rows a kernel can read 16 bytes at a time: a contiguous head, other strides
    multiples of 8 elements, tokens at least ``least`` elements apart."""
    strides = t.stride()
    return (t.dtype == torch.bfloat16 and strides[-1] == 1 and t.data_ptr() % 16 == 0
            and all(s % 8 == 0 for s in strides[:-1]) and strides[head] >= 0
            and least <= strides[token] <= 1 << 23)


def _heads_ok(hq, hkv, dim, scale):
    return (dim in HEAD_DIMS and hkv > 0 and hq % hkv == 0 and isinstance(scale, (int, float))
            and math.isfinite(scale))


def _rows(dim):
    """Packed (token, query head of the group) rows of a workgroup."""
    return 64 if dim == 256 else 128


@functools.lru_cache(maxsize=None)
def device_cus(device):
    return torch.cuda.get_device_properties(device).multi_processor_count


def _splits(workgroups, max_keys, dim, device):
    """Key spans per row tile, of 256 keys or more each: as many as fill the device's slots
    (two workgroups a CU), and at head_dim 256, where a workgroup's rows are few and its
    spans uneven, twice that.  Measured, one span against the rule's: 108 and 79 us (2049
    rows, Hq 8 / Hkv 2, D 256, 258 workgroups, 4 spans; 2 spans 91), 176 and 42 us (100 rows
    after 3072, Hq 16 / Hkv 4, D 256, 12 spans; 8 spans 40), 80 and 26 us (128 after 2048, Hq
    8 / Hkv 2, D 128, 8 spans), 30 and 25 us (512 rows, Hq 8 / Hkv 2, D 256, 2 spans; 4 spans
    22); two spans where the workgroups fill the slots alone: 103 instead of 87 us (2048
    rows, Hq 32 / Hkv 8, D 128)."""
    if not isinstance(max_keys, numbers.Integral):
        return 1
    cus = device_cus(device)
    slots = 4 * cus if dim == 256 else 2 * cus
    return max(1, min((slots + workgroups // 2) // workgroups, max_keys // 256, 16))


def _workspace(splits, total_q, heads, dim, device):
    if splits == 1:
        return None, None
    return (torch.empty((splits, total_q, heads, dim), device=device, dtype=torch.float32),
            torch.empty((splits, total_q, heads, 2), device=device, dtype=torch.float32))


def packed_prefill(q, k, v, cu_q, cu_k, scale, *, tables=None, max_keys=0, group=None):
    """Attention of packed sequences; q [N, Hq, D], returns a tensor like it.

    ``cu_q``/``cu_k``: cumulative new and visible tokens per sequence.  Without ``tables``
    k and v are the packed rows [M, Hkv, D]; with them the paged caches
    [blocks, block_size, Hkv, D], which hold every visible token already.  ``max_keys`` is
    a hint of the longest sequence's visible tokens (0 or no whole number: unknown).
    ``group``: query heads per kv head of the layer (None: what the tensors have); tensors
    with other head counts fail in the PyTorch form.

    The metadata are checked on the device as the attention starts, which reads nothing
    outside its tensors whatever they hold, and the host waits for that check alone: what does
    not fit the tensors is left to the PyTorch form, which fails on it, and pages outside the
    cache raise.  A captured call has no such check: there such rows read as zeros.
    """
    return PackedPrefill(q, k, v, cu_q, cu_k, scale, tables, max_keys, group).run()


class PackedPrefill:
    """One packed_prefill call, so that the K/V write ahead of it can check its metadata:
    ``check`` is what that launch takes (None: nothing for it to check), then ``run``."""

    def __init__(self, q, k, v, cu_q, cu_k, scale, tables=None, max_keys=0, group=None):
        self.call = q, k, v, cu_q, cu_k, scale, tables
        self.max_keys = max_keys
        self.out = torch.empty_like(q)
        self.group = q.shape[1] // k.shape[-2] if group is None else group
        self.kernel = (_packed_ok(q, k, v, self.out, cu_q, cu_k, scale, tables)
                       and q.shape[1] == self.group * k.shape[-2])
        self.check = None
        if (self.kernel and q.shape[0] and cu_q.shape[0] > 1
                and not torch.cuda.is_current_stream_capturing()):
            page_size, num_pages = (k.shape[1], k.shape[0]) if tables is not None else (0, 0)
            self.check = (cu_q, cu_k, cu_q.shape[0] - 1, q.shape[0],
                          0 if tables is not None else k.shape[0], tables, page_size, num_pages,
                          torch.zeros(_native.CHECK_WORDS, dtype=torch.int32, pin_memory=True))

    def run(self, checking=False):
        """The attention; ``checking``: a launch with ``check`` is under way."""
        q, k, v, cu_q, cu_k, scale, tables = self.call
        if not self.kernel:
            return self._general()
        n, hq, d = q.shape
        hkv, seqs = k.shape[-2], cu_q.shape[0] - 1
        if self.check is None:
            if seqs < 1 or n == 0:
                empty = seqs < 1 or torch.cuda.is_current_stream_capturing()
                return self.out if empty else self._general()
            verdicts = None
        else:
            verdicts = self.check[-1]
        try:
            splits = _splits((n * (hq // hkv) // _rows(d) + seqs) * hkv, self.max_keys, d, q.device)
            part_o, part_ml = _workspace(splits, n, hq, d, q.device)
            rows = lambda t: (t.stride(0) if t.dim() == 4 else 0, t.stride(-3), t.stride(-2))  # noqa: E731
            paged = tables is not None
            _native.prefill(q, rows(q), k, rows(k), v, rows(v), self.out, rows(self.out), cu_q, cu_k,
                            seqs, 0, n, 0 if paged else k.shape[0], tables,
                            k.shape[1] if paged else 0, k.shape[0] if paged else 0, hq, hkv, d,
                            float(scale), splits, part_o, part_ml, None if checking else verdicts)
            checking = verdicts is not None
        finally:        # until it has been waited for, a check writes to ``verdicts``
            found = _native.check_wait(verdicts, q.device) if checking else 0
        if found & _native.CHECK_OUTSIDE:
            raise IndexError("a sequence reaches past its block table or to a page outside the cache")
        return self._general() if found & _native.CHECK_ODD else self.out

    def _general(self):
        return _packed_torch(*self.call, self.out, self.group)


def _packed_ok(q, k, v, out, cu_q, cu_k, scale, tables):
    meta = (cu_q, cu_k) if tables is None else (cu_q, cu_k, tables)
    if not all(isinstance(t, torch.Tensor) for t in (q, k, v, *meta)) or not _plain(q, k, v, *meta):
        return False
    if any(t.device != q.device for t in (k, v, *meta)) or q.dim() != 3:
        return False
    if k.shape != v.shape or k.dim() != (3 if tables is None else 4) or k.shape[-1] != q.shape[-1]:
        return False
    if not _heads_ok(q.shape[1], k.shape[-2], q.shape[2], scale):
        return False
    if k.shape[0] == 0 or max(q.shape[0], k.shape[0]) * q.shape[1] >= 1 << 31:
        return False
    if not (_rows_ok(q, 0, 1, 0) and _rows_ok(out, 0, 1, 0)):
        return False
    d = q.shape[2]
    if not (_rows_ok(k, -3, -2, d) and _rows_ok(v, -3, -2, d)):
        return False
    if any(t.dtype != torch.int32 or t.stride(-1) != 1 for t in meta):
        return False
    if cu_q.dim() != 1 or cu_k.dim() != 1 or cu_k.shape[0] < cu_q.shape[0]:
        return False
    if tables is not None:
        tile = 32 if d == 256 else 64
        if tables.dim() != 2 or tables.shape[0] < cu_q.shape[0] - 1 or tables.shape[1] < 1:
            return False
        if k.shape[1] == 0 or k.shape[1] % tile or k.stride(0) < 0 or v.stride(0) < 0:
            return False
    return True


def _packed_torch(q, k, v, cu_q, cu_k, scale, tables, out, group):
    cu_q, cu_k = cu_q.tolist(), cu_k.tolist()
    for i in range(len(cu_q) - 1):
        nq, nk = cu_q[i + 1] - cu_q[i], cu_k[i + 1] - cu_k[i]
        if tables is None:
            keys, vals = k[cu_k[i]:cu_k[i + 1]], v[cu_k[i]:cu_k[i + 1]]
        else:  # prefix cache: the whole context is in the paged cache already
            pos = torch.arange(nk, device=q.device)
            blocks = tables[i, pos // k.shape[1]].long()
            keys, vals = k[blocks, pos % k.shape[1]], v[blocks, pos % k.shape[1]]
        qf = q[cu_q[i]:cu_q[i + 1]].float().transpose(0, 1)                   # [Hq, nq, D]
        kf = keys.float().repeat_interleave(group, dim=1).transpose(0, 1)     # [Hq, nk, D]
        vf = vals.float().repeat_interleave(group, dim=1).transpose(0, 1)
        scores = torch.matmul(qf, kf.transpose(1, 2).contiguous()) * scale
        qpos = torch.arange(nk - nq, nk, device=q.device)[:, None]
        scores.masked_fill_(torch.arange(nk, device=q.device)[None, :] > qpos, float("-inf"))
        out[cu_q[i]:cu_q[i + 1]] = torch.matmul(scores.softmax(-1), vf).transpose(0, 1).to(q.dtype)
    return out


def batched_prefill(query, key, value, scale):
    """Attention of equally long sequences without a prefix; query [B, Hq, S, D], key and
    value [B, Hkv, S, D], returns [B, S, Hq, D], contiguous in either form: the decoder's
    kernels read it by its address."""
    if not _batched_ok(query, key, value, scale):
        return _batched_torch(query, key, value, scale)
    b, hq, s, d = query.shape
    hkv = key.shape[1]
    out = torch.empty((b, s, hq, d), device=query.device, dtype=query.dtype)
    splits = _splits(b * -(-s * (hq // hkv) // _rows(d)) * hkv, s, d, query.device)
    part_o, part_ml = _workspace(splits, b * s, hq, d, query.device)
    rows = lambda t: (t.stride(0), t.stride(2), t.stride(1))  # noqa: E731
    _native.prefill(query, rows(query), key, rows(key), value, rows(value), out,
                    (out.stride(0), out.stride(1), out.stride(2)), None, None, b, s, b * s, b * s,
                    None, 0, 0, hq, hkv, d, float(scale), splits, part_o, part_ml)
    return out


def _batched_ok(query, key, value, scale):
    if not _plain(query, key, value) or any(t.device != query.device for t in (key, value)):
        return False
    if query.dim() != 4 or key.shape != value.shape or key.dim() != 4:
        return False
    b, hq, s, d = query.shape
    if key.shape[0] != b or key.shape[2:] != (s, d) or not _heads_ok(hq, key.shape[1], d, scale):
        return False
    if b == 0 or s == 0 or b * s * hq >= 1 << 31:
        return False
    return (_rows_ok(query, 2, 1, 0) and _rows_ok(key, 2, 1, d) and _rows_ok(value, 2, 1, d)
            and min(t.stride(0) for t in (query, key, value)) >= 0)


def _batched_torch(query, key, value, scale):
    s = query.shape[2]
    group = query.shape[1] // key.shape[1]
    q = query.float()
    k = key.float().repeat_interleave(group, dim=1).transpose(-1, -2).contiguous()
    v = value.float().repeat_interleave(group, dim=1).contiguous()
    scores = torch.matmul(q, k) * scale
    future = torch.ones(s, s, dtype=torch.bool, device=query.device).triu(1)
    probs = scores.masked_fill(future, float("-inf")).softmax(-1)
    return torch.matmul(probs, v).transpose(1, 2).to(query.dtype).contiguous()
