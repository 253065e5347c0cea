"""GPU parity of the prefill attention kernel (pd_prefill) with attention in 64 bits.

The gate is derived per output: half a bf16 ulp, plus what float32 leaves in the scores
(a dot product of D terms) and in the sums over the keys (and their three bf16 terms).
"""
import numpy as np
import pytest
import torch

if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)

from paged_decode import prefill as PF
from paged_decode.engine_attention import Attention, reset_context, set_context

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def rows(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)


def check(out, q, k, v, first, scale, where):
    """out/q [n, Hq, D] at positions first.. against keys k, v [m, Hkv, D]."""
    n, hq, d = q.shape
    m, group = k.shape[0], hq // k.shape[1]
    q64, k64, v64 = (t.double().cpu().transpose(0, 1) for t in (q, k, v))
    k64, v64 = k64.repeat_interleave(group, 0), v64.repeat_interleave(group, 0)
    masked = torch.arange(m)[None, :] > first + torch.arange(n)[:, None]
    s = (torch.matmul(q64, k64.transpose(1, 2)) * scale).masked_fill(masked, float("-inf"))
    p = s.softmax(-1)
    ref = torch.matmul(p, v64)
    spread = torch.matmul(p, v64.abs())
    size = torch.matmul(q64.abs(), k64.abs().transpose(1, 2)).amax(-1, keepdim=True) * abs(scale)
    # half an ulp of 8 significant bits is at most 2^-8 of the value
    bound = 2.0 ** -8 * ref.abs() + (2 * (d + 4) * size + m + 16) * 2 * EPS * spread
    diff = (out.double().cpu().transpose(0, 1) - ref).abs()
    worst = (diff / (bound + 1e-30)).max()
    assert worst <= 1, (where, float(worst), float(diff.max()))


def packed(lens, prefix, hq, hkv, d, page, seed, scale=None, splits=None, monkeypatch=None):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if splits:
        monkeypatch.setattr(PF, "_splits", lambda *a: splits)
    total = [n + prefix for n in lens]
    cu = lambda ns: torch.tensor(np.cumsum([0] + ns), dtype=torch.int32, device="cuda")  # noqa: E731
    q = rows(gen, sum(lens), hq, d)
    # keys and values as slices of one fused row, like a model's projection
    kv = rows(gen, sum(total), 2 * hkv, d)
    k, v = kv[:, :hkv], kv[:, hkv:]
    scale = d ** -0.5 if scale is None else scale
    if page:
        width = max(-(-n // page) for n in total)
        blocks = sum(-(-n // page) for n in total) + 1
        order = list(np.random.default_rng(seed).permutation(blocks))
        cache = torch.full((2, blocks, page, hkv, d), float("nan"), device="cuda",
                           dtype=torch.bfloat16)
        tables = torch.full((len(lens), width), -1, dtype=torch.int32)
        at = 0
        for i, n in enumerate(total):
            for j in range(0, n, page):
                b = int(order.pop())
                tables[i, j // page] = b
                take = min(page, n - j)
                cache[0, b, :take], cache[1, b, :take] = k[at + j:at + j + take], v[at + j:at + j + take]
            at += n
        args = (q, cache[0], cache[1], cu(lens), cu(total), scale)
        kwargs = dict(tables=tables.cuda(), max_keys=max(total))
    else:
        args, kwargs = (q, k, v, cu(lens), cu(total), scale), dict(max_keys=max(total))
    assert PF._packed_ok(args[0], args[1], args[2], torch.empty_like(q), args[3], args[4], scale,
                         kwargs.get("tables"))
    out = PF.packed_prefill(*args, **kwargs)
    a = b = 0
    for n, m in zip(lens, total):
        if n:
            check(out[a:a + n], q[a:a + n], k[b:b + m], v[b:b + m], prefix, scale, (n, m))
        a, b = a + n, b + m


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 256), (8, 2, 128), (4, 4, 64), (6, 2, 128), (16, 1, 64)])
@pytest.mark.parametrize("lens,prefix", [([1], 0), ([31, 1, 65], 0), ([127, 129, 2], 0), ([300, 33], 0),
                                         ([1, 70], 64), ([40], 1000)])
def test_packed_rows(hq, hkv, d, lens, prefix):
    packed(lens, prefix, hq, hkv, d, None, sum(lens) + d)


@pytest.mark.parametrize("hq,hkv,d,page", [(8, 2, 256, 256), (8, 2, 256, 32), (8, 8, 128, 64),
                                           (4, 1, 64, 256)])
@pytest.mark.parametrize("lens,prefix", [([1, 5, 257], 0), ([64, 31], 256), ([3], 700)])
def test_paged_keys_with_nan_beyond_the_live_rows(hq, hkv, d, page, lens, prefix):
    packed(lens, prefix, hq, hkv, d, page, sum(lens) + page)


@pytest.mark.parametrize("splits", [2, 3, 8])
@pytest.mark.parametrize("d,page", [(256, 256), (128, None), (64, 256)])
def test_split_keys(monkeypatch, splits, d, page):
    packed([200, 1, 33], 130, 8, 2, d, page, splits, splits=splits, monkeypatch=monkeypatch)


@pytest.mark.parametrize("scale", [0.0, -0.09, 1.0, 3.0])
def test_scales(scale):
    packed([150], 20, 4, 2, 128, None, 7, scale=scale)


def test_more_than_a_wavefront_of_sequences():
    packed([(5 * i) % 23 for i in range(140)], 3, 4, 2, 64, None, 9)


@pytest.mark.parametrize("b,hq,hkv,s,d", [(1, 8, 2, 513, 256), (3, 8, 2, 65, 256), (2, 4, 4, 200, 128)])
def test_batched(b, hq, hkv, s, d):
    gen = torch.Generator(device="cuda").manual_seed(s)
    q = rows(gen, b, s, hq, d).transpose(1, 2)
    k = rows(gen, b, s, hkv, d).transpose(1, 2)
    v = rows(gen, b, s, hkv, d).transpose(1, 2)
    assert PF._batched_ok(q, k, v, d ** -0.5)
    out = PF.batched_prefill(q, k, v, d ** -0.5)
    for i in range(b):
        check(out[i], q[i].transpose(0, 1), k[i].transpose(0, 1), v[i].transpose(0, 1), 0,
              d ** -0.5, i)


@pytest.mark.parametrize("special", ["v_inf", "k_inf", "q_nan"])
def test_infinities_and_nans_as_in_float32(special):
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = rows(gen, 1, 2, 70, 128), rows(gen, 1, 2, 70, 128), rows(gen, 1, 2, 70, 128)
    if special == "v_inf":
        v[0, 0, 0, 5], v[0, 1, 0, 7] = float("inf"), float("-inf")
    elif special == "k_inf":
        k[0, 0, 0, 3] = float("inf")
    else:
        q[0, 1, 40, 9] = float("nan")
    out = PF.batched_prefill(q, k, v, 0.1).float()
    ref = PF._batched_torch(q, k, v, 0.1).float()
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    ok = ref.isfinite()
    assert (out[ok] - ref[ok]).abs().max() < 2.0 ** -6
    assert torch.equal(out[ref.isinf()], ref[ref.isinf()])


def test_general_form_serves_what_the_kernel_does_not():
    gen = torch.Generator(device="cuda").manual_seed(4)
    q, k, v = (rows(gen, 37, 4, 80) for _ in range(3))
    cu = torch.tensor([0, 20, 37], dtype=torch.int64, device="cuda")
    out = PF.packed_prefill(q, k, v, cu, cu, 0.1)
    for a, b in ((0, 20), (20, 37)):
        check(out[a:b], q[a:b], k[a:b], v[a:b], 0, 0.1, a)
    x = torch.randn(9, 2, 64, requires_grad=True)
    cu = torch.tensor([0, 9], dtype=torch.int32)
    PF.packed_prefill(x, x, x, cu, cu, 0.1).sum().backward()
    assert x.grad.abs().sum() > 0


def metadata(d=64, page=None, lens=(20, 1, 37), prefix=64):
    """A packed call (paged with `page`) as (q, k, v, cu_q, cu_k, scale), keywords, host lists."""
    gen = torch.Generator(device="cuda").manual_seed(d)
    total = [n + (prefix if page else 0) for n in lens]
    q = rows(gen, sum(lens), 4, d)
    cu = [list(np.cumsum([0, *ns])) for ns in (lens, total)]
    if page is None:
        return q, rows(gen, sum(total), 2, d), rows(gen, sum(total), 2, d), *cu, None
    used = [-(-n // page) for n in total]
    order = list(np.random.default_rng(d).permutation(sum(used) + 2))
    table = [[int(order.pop()) for _ in range(n)] + [-1] * (max(used) - n) for n in used]
    k, v = (rows(gen, sum(used) + 2, page, 2, d) for _ in range(2))
    return q, k, v, *cu, table


def call(q, k, v, cu_q, cu_k, table, form=PF.packed_prefill):
    device = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    args = (q, k, v, device(cu_q), device(cu_k), 0.1)
    tables = None if table is None else device(table)
    if form is PF.packed_prefill:
        out = torch.empty_like(q)
        assert q.shape[0] == 0 or PF._packed_ok(*args[:3], out, *args[3:], tables)
        return form(*args, tables=tables, max_keys=3000)
    return form(*args, tables, torch.zeros_like(q), 2)


@pytest.mark.parametrize("d,page", [(64, None), (256, 32)])
@pytest.mark.parametrize("fault", ["q_end", "q_order", "q_start", "k_order", "no_rows"])
def test_sequences_that_are_not_the_tensors_fail(d, page, fault):
    q, k, v, cu_q, cu_k, table = metadata(d, page)
    if fault == "q_end":
        cu_q[-1] += 1
    elif fault == "q_order":
        cu_q[1], cu_q[2] = cu_q[2] + 3, cu_q[1]
    elif fault == "q_start":
        cu_q[0] = -3
    elif fault == "k_order":
        cu_k[2:] = [n - (cu_k[2] - cu_k[1] + 2) for n in cu_k[2:]]
    else:
        q = q[:0]
    for form in (PF.packed_prefill, PF._packed_torch):
        with pytest.raises(RuntimeError):
            call(q, k, v, cu_q, cu_k, table, form)


@pytest.mark.parametrize("fault", ["k_end", "k_start"])
def test_keys_that_are_not_the_tensors_fail(fault):
    q, k, v, cu_q, cu_k, _ = metadata()
    cu_k[0 if fault == "k_start" else -1] += -2 if fault == "k_start" else 2
    for form in (PF.packed_prefill, PF._packed_torch):
        with pytest.raises(RuntimeError):
            call(q, k, v, cu_q, cu_k, None, form)


@pytest.mark.parametrize("fault", ["width", "page", "below"])
@pytest.mark.parametrize("sequences", [3, 300])
def test_pages_outside_the_cache_fail(fault, sequences):
    q, k, v, cu_q, cu_k, table = metadata(256, 32, lens=(5,) * sequences)
    if fault == "width":
        cu_k[-1] += 32
    else:
        table[-1][1] = k.shape[0] if fault == "page" else -k.shape[0] - 1
    with pytest.raises(IndexError, match="outside the cache"):
        call(q, k, v, cu_q, cu_k, table)
    table[-1][1] = 0     # and the process goes on
    cu_k[-1] = cu_k[-2] + 69
    call(q, k, v, cu_q, cu_k, table)


@pytest.mark.parametrize("d,page", [(64, 64), (256, 32), (128, None)])
def test_unusual_metadata_as_in_the_general_form(d, page):
    """Pages counted from the pool's end, and a sequence of new tokens without keys."""
    q, k, v, cu_q, cu_k, table = metadata(d, page)
    if page:
        table[0][0], table[2][1] = -1, -3
    cu_k[2:] = [n - (cu_k[2] - cu_k[1]) for n in cu_k[2:]]
    if not page:
        k, v = k[:cu_k[-1]], v[:cu_k[-1]]
    got, want = (call(q, k, v, cu_q, cu_k, table, form) for form in (PF.packed_prefill, PF._packed_torch))
    assert torch.equal(got, want) and not got[cu_q[1]:cu_q[2]].any()


def test_captured_packed_prefill():
    q, k, v, cu_q, cu_k, table = metadata(256, 32)
    device = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    args = (q, k, v, device(cu_q), device(cu_k), 0.1)
    tables = device(table)
    PF.packed_prefill(*args, tables=tables, max_keys=3000)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = PF.packed_prefill(*args, tables=tables, max_keys=3000)
    for seed in range(3):
        q.copy_(rows(torch.Generator(device="cuda").manual_seed(seed), *q.shape))
        graph.replay()
        assert torch.equal(out, PF.packed_prefill(*args, tables=tables, max_keys=3000))


@pytest.mark.parametrize("d,page,splits", [(64, None, 1), (64, 64, 3), (128, None, 1), (128, 64, 2),
                                           (256, None, 1), (256, 32, 1), (256, 256, 3)])
@pytest.mark.parametrize("special", ["v_inf", "v_both", "v_nan", "k_nan"])
def test_later_tokens_never_reach_earlier_rows(monkeypatch, d, page, splits, special):
    """Infinities and NaN in the keys' rows: rows that see their token get them, as the
    softmax's products do; rows before it are what they are without it."""
    monkeypatch.setattr(PF, "_splits", lambda *a: splits)
    gen = torch.Generator(device="cuda").manual_seed(d)
    n, hq, prefix = 150, 4, 70 if page else 0
    m = n + prefix
    q, k, v = rows(gen, n, hq, d), rows(gen, m, 2, d), rows(gen, m, 2, d)
    inf = float("inf")
    for at, sign in ((prefix + 2, 1), (prefix + 97, -1), (m - 1, 1)):
        if special == "k_nan":
            k[at, 1, 3] = float("nan")
        else:
            v[at, 0, d - 7] = float("nan") if special == "v_nan" else sign * inf
            if special == "v_both":
                v[at, 0, 5], v[at, 1, 33] = inf, sign * inf
    keys, vals, tables = k, v, None
    if page:
        used = -(-m // page)
        order = np.random.default_rng(d).permutation(used + 1)[:used]
        keys, vals = (torch.full((used + 1, page, 2, d), float("nan"), device="cuda").bfloat16() for _ in "kv")
        for i, b in enumerate(order):
            part = slice(page * i, min(page * (i + 1), m))
            keys[b, :part.stop - part.start], vals[b, :part.stop - part.start] = k[part], v[part]
        tables = torch.tensor(order[None], dtype=torch.int32, device="cuda")
    cu = lambda x: torch.tensor([0, x], dtype=torch.int32, device="cuda")  # noqa: E731
    assert PF._packed_ok(q, keys, vals, torch.empty_like(q), cu(n), cu(m), 0.1, tables)
    out = PF.packed_prefill(q, keys, vals, cu(n), cu(m), 0.1, tables=tables).double().cpu()
    q, k, v = (t.double().cpu() for t in (q, k, v))
    for t in range(n):
        seen = prefix + t + 1
        for h in range(hq):
            p = (k[:seen, h // 2] @ q[t, h] * 0.1).softmax(-1)
            # a product and a sum a key, as a matrix product's zero terms are none of them
            want = (p[:, None] * v[:seen, h // 2]).sum(0)
            got = out[t, h]
            assert torch.equal(got.isnan(), want.isnan()), (t, h)
            assert torch.equal(got[want.isinf()], want[want.isinf()]), (t, h)
            ok = want.isfinite()
            assert not ok.any() or (got[ok] - want[ok]).abs().max() < 2.0 ** -6, (t, h)


@pytest.mark.parametrize("prefix", [0, 96])
@pytest.mark.parametrize("fault", [None, "q_end", "k_order", "page", "width", "wrapped"])
def test_layers_check_the_metadata_with_the_write(prefix, fault):
    """The engine's layer: what does not fit fails as in packed_prefill, the rows are written
    first, and the next call is a plain one."""
    page, d, lens = 32, 256, (40, 1, 300)
    q, k, v, cu_q, cu_k, table = metadata(d, page, lens, prefix)
    if not prefix and fault in ("page", "width", "wrapped"):
        pytest.skip("no pages to read")
    layer = Attention(4, d, 0.1, 2)
    layer.k_cache, layer.v_cache = k, v
    gen = torch.Generator(device="cuda").manual_seed(1)
    key, value = rows(gen, sum(lens), 2, d), rows(gen, sum(lens), 2, d)
    slots = torch.cat([torch.tensor([table[i][t // page] * page + t % page
                                     for t in range(prefix, prefix + n)]) for i, n in enumerate(lens)])
    if not prefix:
        cu_k = list(cu_q)
    good = list(cu_q), list(cu_k), [list(t) for t in table]
    if fault == "q_end":
        cu_q[-1] += 1
    elif fault == "k_order":
        cu_k[2:] = [n - (cu_k[2] - cu_k[1] + 2) for n in cu_k[2:]]
    elif fault == "page":
        table[2][0] = k.shape[0]
    elif fault == "width":
        cu_k[-1] += page
    elif fault == "wrapped":
        table[2][0] -= k.shape[0]
    device = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731

    def run(cu_q, cu_k, table):
        set_context(True, device(cu_q), device(cu_k), 300, 500, slots.int().cuda(),
                    block_tables=device(table) if prefix else None)
        try:
            return layer(q, key, value)
        finally:
            reset_context()

    want = run(*good)
    flat = k.view(-1, 2, d)
    flat[slots.cuda()] = 0
    if fault in (None, "wrapped"):
        assert (run(cu_q, cu_k, table) - want).abs().max() < 2.0 ** -6
    else:
        with pytest.raises(IndexError if fault in ("page", "width") else RuntimeError):
            run(cu_q, cu_k, table)
    assert torch.equal(flat[slots.cuda()], key)
    assert torch.equal(run(*good), want)
