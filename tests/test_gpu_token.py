"""GPU parity of the one-token layer kernels with the same formulas in 64 bits.

A product's inputs are rounded to bf16 after the norm or gate, its float32 sums once more
at the end.  The reference rounds the inputs alike; where float32 may round one the other
way (within 2^-19 of a tie), the difference is allowed.  A sum is a chain of at most K / 8
+ 24 float32 additions (its terms shared by four wavefronts or more with two sums each,
then the wavefronts' partial sums and the residual).
"""
import pytest
import torch
import torch.nn.functional as F

if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)

from paged_decode import _native

pytestmark = pytest.mark.gpu


def bf16(gen, *shape, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)


def normed(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1 + w.double())


def rounded(h):
    """(h in bf16, how far the other rounding of values near a tie is)."""
    low, high = ((h * (1 + s * 2.0 ** -19)).to(torch.bfloat16).double() for s in (-1, 1))
    return h.to(torch.bfloat16).double(), (high - low).abs()


def product(h, w):
    """(h w^T, bound of a float32 sum of it), h [rows, K] before its rounding to bf16."""
    h, tie = rounded(h.double())
    w = w.double()
    chain = (h.shape[1] / 8 + 24) * 2.0 ** -24
    return h @ w.T, chain * (h.abs() @ w.abs().T) + tie @ w.abs().T


def within(got, ref, bound):
    """got (bf16) is ref, known to `bound`, rounded."""
    bound = bound + 2.0 ** -8 * (ref.abs() + bound) + 1e-30
    worst = ((got.double() - ref).abs() / bound).max()
    assert worst <= 1, float(worst)


def check(got, h, w):
    within(got, *product(h, w))


def check_sum(got, held, h, w):
    ref, bound = product(h, w)
    within(got, held.double() + ref, bound)


@pytest.mark.parametrize("rows", [1, 2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("dim,features", [(64, (3, 20)), (256, (40, 8, 4)), (2048, (48, 16)),
                                          (2112, (16,)), (4096, (24,))])
def test_norm_linears(rows, dim, features):
    gen = torch.Generator(device="cuda").manual_seed(rows * dim)
    x, norm = bf16(gen, rows, dim), bf16(gen, dim, scale=0.1)
    weights = [bf16(gen, f, dim, scale=0.05) for f in features]
    outs = [torch.empty(rows, f, device="cuda", dtype=torch.bfloat16) for f in features]
    _native.norm_linears(x, norm, 1e-6, weights, outs)
    for w, out in zip(weights, outs):
        check(out, normed(x, norm), w)


@pytest.mark.parametrize("rows", [1, 3, 8])
def test_a_vocabulary_walks_its_tiles(rows):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    for dim, features in ((256, 40007), (2048, 16392), (2176, 17000)):
        x, norm, w = bf16(gen, rows, dim), bf16(gen, dim, scale=0.1), bf16(gen, features, dim, scale=0.05)
        out = torch.empty(rows, features, device="cuda", dtype=torch.bfloat16)
        _native.norm_linears(x, norm, 1e-6, (w,), (out,))
        check(out, normed(x, norm), w)


@pytest.mark.parametrize("rows", [1, 4, 7, 16])
@pytest.mark.parametrize("dim", [64, 256, 2048])
def test_gate_up_and_residual(rows, dim):
    gen = torch.Generator(device="cuda").manual_seed(rows + dim)
    mid = 200
    x, norm = bf16(gen, rows, dim), bf16(gen, dim, scale=0.1)
    gate, up = bf16(gen, mid, dim, scale=dim ** -0.5), bf16(gen, mid, dim, scale=dim ** -0.5)
    out = torch.empty(rows, mid, device="cuda", dtype=torch.bfloat16)
    _native.norm_gate_up(x, norm, 1e-6, gate, up, out)
    (a, da), (b, db) = product(normed(x, norm), gate), product(normed(x, norm), up)
    # silu's slope is at most 1.1, its float32 value good to 2^-19
    within(out, F.silu(a) * b, 1.1 * da * (b.abs() + db) + F.silu(a).abs() * (db + 2.0 ** -19 * b.abs()))
    h, w, held = bf16(gen, rows, dim), bf16(gen, 72, dim, scale=0.05), bf16(gen, rows, 72)
    y = held.clone()
    _native.linear_add(h, w, y)
    check_sum(y, held, h, w)


@pytest.mark.parametrize("rows", [1, 4, 8, 9, 16])
@pytest.mark.parametrize("dim,d", [(64, 64), (256, 64), (256, 128), (256, 256), (768, 256),
                                   (2048, 128), (2048, 256)])
def test_gated_residual(rows, dim, d):
    gen = torch.Generator(device="cuda").manual_seed(rows + dim + d)
    h, w, held = bf16(gen, rows, dim), bf16(gen, 72, dim, scale=0.05), bf16(gen, rows, 72)
    q, y = bf16(gen, rows, dim // d, 2 * d, scale=2), held.clone()
    _native.linear_add(h, w, y, q[..., d:], d)
    check_sum(y, held, h.double() * torch.sigmoid(q[..., d:].double()).reshape(rows, dim), w)


@pytest.mark.parametrize("dim", [6144, 1088])
def test_long_inputs_take_several_rounds(dim):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    for rows in (1, 8, 9):
        h, w, held = bf16(gen, rows, dim), bf16(gen, 40, dim, scale=0.05), bf16(gen, rows, 40)
        y = held.clone()
        _native.linear_add(h, w, y)
        check_sum(y, held, h, w)


@pytest.mark.parametrize("rows,held", [(1, True), (3, False), (8, True), (11, True)])
def test_convolved_projection(rows, held):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    dim, c = 256, 56
    x, norm, w = bf16(gen, rows, dim), bf16(gen, dim, scale=0.1), bf16(gen, c, dim, scale=0.05)
    z, taps, state = bf16(gen, 9, dim, scale=0.05), bf16(gen, c, 1, 4, scale=0.5), bf16(gen, rows, c, 4)
    before = state.clone() if held else torch.zeros_like(state)
    act = torch.empty(rows, c, device="cuda")
    gate = torch.empty(rows, 9, device="cuda", dtype=torch.bfloat16)
    _native.norm_linears(x, norm, 1e-6, (w, z), (act, gate), taps, state, held)
    assert torch.equal(state[..., :3], before[..., 1:])
    check(state[..., 3], normed(x, norm), w)
    check(gate, normed(x, norm), z)
    ref = F.silu((state.double() * taps.double()[:, 0]).sum(-1))
    assert ((act.double() - ref).abs() <= 1e-6 * (1 + ref.abs())).all()


@pytest.mark.parametrize("hk,hv,dk,dv", [(4, 4, 64, 64), (2, 4, 128, 128), (1, 2, 64, 128), (3, 3, 128, 64)])
@pytest.mark.parametrize("batch,held", [(1, True), (3, False)])
def test_delta_step(hk, hv, dk, dv, batch, held):
    gen = torch.Generator(device="cuda").manual_seed(dk + dv)
    act = torch.randn((batch, 2 * hk * dk + hv * dv), generator=gen, device="cuda")
    state = torch.randn((batch, hv, dk, dv), generator=gen, device="cuda") * 0.1
    a, b, z = bf16(gen, batch, hv, scale=3), bf16(gen, batch, hv), bf16(gen, batch, hv * dv, scale=2)
    a_log, dt, norm = bf16(gen, hv), bf16(gen, hv, scale=2), bf16(gen, dv)
    out = torch.empty(batch, hv, dv, device="cuda", dtype=torch.bfloat16)
    ref = state.double() if held else torch.zeros_like(state).double()
    _native.delta_step(act, a, b, a_log, dt, z, norm, 1e-6, state, out, batch, hk, hv, dk, dv, held)
    q, k, v = act.double().split([hk * dk, hk * dk, hv * dv], -1)
    unit = lambda y: y * torch.rsqrt(y.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = (unit(q.view(batch, hk, dk)) * dk ** -0.5).repeat_interleave(hv // hk, 1)
    k, v = unit(k.view(batch, hk, dk)).repeat_interleave(hv // hk, 1), v.view(batch, hv, dv)
    decay = torch.exp(-a_log.double().exp() * F.softplus(a.double() + dt.double()))
    beta = torch.sigmoid(b.double())
    ref = ref * decay[..., None, None]
    d = (v - (k[..., None] * ref).sum(-2)) * beta[..., None]
    ref = ref + k[..., None] * d[:, :, None]
    assert ((state.double() - ref).abs() <= 4e-6 * (1 + ref.abs())).all()
    o = (q[..., None] * ref).sum(-2)
    y = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-6) * norm.double()
    y = y * F.silu(z.double().view(batch, hv, dv))
    assert ((out.double() - y).abs() <= 2.0 ** -8 * y.abs() + 1e-4).all()
