"""GPU parity of the one-token layer kernels with the same formulas in 64 bits.

A product's inputs are rounded to bf16 after the norm or gate (2^-9 relative, at random
over its terms: bounded by 2^-8 of the products' 2-norm times 4), its result once more.
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


def check(got, h, w, ref=None, slack=1.0):
    """got ~ ref, a product of h [rows, K] and w [features, K] by default."""
    plain = h @ w.double().T
    ref = plain if ref is None else ref
    spread = (h.square() @ w.double().square().T).sqrt()
    bound = 2.0 ** -6 * slack * spread + 2.0 ** -8 * ref.abs() + 1e-30
    worst = ((got.double() - ref).abs() / bound).max()
    assert worst <= 1, float(worst)


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
    h = normed(x, norm)
    ref = F.silu(h @ gate.double().T) * (h @ up.double().T)
    check(out, h, gate, ref, slack=4.0)
    h, w, held = bf16(gen, rows, dim), bf16(gen, 72, dim, scale=0.05), bf16(gen, rows, 72)
    y = held.clone()
    _native.linear_add(h, w, y)
    check(y, h.double(), w, held.double() + h.double() @ w.double().T)
    d = 64
    q, y = bf16(gen, rows, dim // d, 2 * d, scale=2), held.clone()
    _native.linear_add(h, w, y, q[..., d:], d)
    g = h.double() * torch.sigmoid(q[..., d:].double()).reshape(rows, dim)
    check(y, g, w, held.double() + g @ w.double().T)


@pytest.mark.parametrize("dim", [6144, 1088])
def test_long_inputs_take_several_rounds(dim):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    for rows in (1, 8, 9):
        h, w, held = bf16(gen, rows, dim), bf16(gen, 40, dim, scale=0.05), bf16(gen, rows, 40)
        y = held.clone()
        _native.linear_add(h, w, y)
        check(y, h.double(), w, held.double() + h.double() @ w.double().T)


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
