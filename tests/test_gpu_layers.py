"""GPU parity of the decoder-layer kernels with the same formulas in 64 bits.

float32 results are held to a few float32 ulps of the largest terms of their sums, bf16
results to half a bf16 ulp (2^-8 of the value) more.
"""
import copy

import numpy as np
import pytest
import torch
import torch.nn.functional as F

if not torch.cuda.is_available():
    pytest.skip("needs an MI355X GPU", allow_module_level=True)

from paged_decode import _native
from paged_decode import decoder_layers as DL
from paged_decode import hybrid as H
from paged_decode import prefill as PF

pytestmark = pytest.mark.gpu


def bf16(gen, *shape, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(torch.bfloat16)


def close(got, ref, absolute, bf16_out=False):
    bound = absolute + (2.0 ** -8 * ref.abs() if bf16_out else 0)
    worst = ((got.double() - ref).abs() / bound).max()
    assert worst <= 1, float(worst)


@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 2040), (5, 2048), (2, 2056), (2, 8192)])
@pytest.mark.parametrize("add", [False, True])
def test_add_rms_norm(rows, dim, add):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    x, y, w = bf16(gen, rows, dim), bf16(gen, rows, dim), bf16(gen, dim, scale=0.1)
    out, held = torch.empty_like(x), x.clone()
    _native.add_rms_norm(x, y if add else None, w, out, 1e-6)
    total = (held.float() + y.float()).to(torch.bfloat16) if add else held
    assert torch.equal(x, total)
    t = total.double()
    ref = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * (1 + w.double())
    close(out, ref, 2.0 ** -18 * ref.abs() + 1e-9, bf16_out=True)


@pytest.mark.parametrize("dim", [64, 128])
def test_gates_and_gated_norm(dim):
    gen = torch.Generator(device="cuda").manual_seed(dim)
    rows = 9
    o = torch.randn((rows, dim), generator=gen, device="cuda")
    z, w, out = bf16(gen, rows, dim, scale=4), bf16(gen, dim), bf16(gen, rows, dim)
    _native.gated_norm(o, z, w, out, rows, dim, 1e-6)
    ref = o.double() * torch.rsqrt(o.double().square().mean(-1, keepdim=True) + 1e-6) * w.double()
    ref = ref * F.silu(z.double())
    close(out, ref, 2.0 ** -18 * ref.abs() + 1e-9, bf16_out=True)
    a, b = bf16(gen, rows, dim, scale=30), bf16(gen, rows, 2 * dim, scale=30)
    _native.sigmoid_gate(a, b[:, dim:], out, rows, dim)
    ref = a.double() * torch.sigmoid(b[:, dim:].double())
    close(out, ref, 2.0 ** -18 * ref.abs() + 1e-30, bf16_out=True)
    ref = F.silu(a.double()) * z.double()
    _native.silu_mul(a, z, a)
    close(a, ref, 2.0 ** -18 * ref.abs() + 1e-30, bf16_out=True)


def linear_case(batch, steps, hk, hv, dk, dv, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    c = 2 * hk * dk + hv * dv
    return dict(x=bf16(gen, batch, steps, c), taps=bf16(gen, c, 1, 4, scale=0.3),
                decay=-3 * torch.rand((batch, steps, hv), generator=gen, device="cuda") ** 3,
                beta=torch.rand((batch, steps, hv), generator=gen, device="cuda"),
                conv=bf16(gen, batch, c, 4),
                state=torch.randn((batch, hv, dk, dv), generator=gen, device="cuda") * 0.1)


def conv_exact(t, hk, hv, dk, dv, held):
    x, taps = t["x"].double(), t["taps"].double()[:, 0]
    batch, steps, c = x.shape
    prev = t["conv"].double().transpose(1, 2) if held else torch.zeros(batch, 4, c, device="cuda").double()
    full = torch.cat([prev, x], 1)
    act = F.silu(sum(full[:, 1 + j:1 + j + steps] * taps[:, j] for j in range(4)))
    unit = lambda y: y * torch.rsqrt(y.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k, v = act.split([hk * dk, hk * dk, hv * dv], -1)
    q, k = unit(q.reshape(batch, steps, hk, dk)) * dk ** -0.5, unit(k.reshape(batch, steps, hk, dk))
    return q, k, v.reshape(batch, steps, hv, dv), full[:, -4:].transpose(1, 2)


def delta_exact(q, k, v, decay, beta, state):
    """The recurrence in 64 bits: (outputs, last state)."""
    group = v.shape[2] // q.shape[2]
    q, k = q.repeat_interleave(group, 2), k.repeat_interleave(group, 2)
    out = torch.empty_like(v)
    for i in range(q.shape[1]):
        state = state * decay[:, i, :, None, None].exp()
        d = (v[:, i] - (k[:, i, :, :, None] * state).sum(-2)) * beta[:, i, :, None]
        state = state + k[:, i, :, :, None] * d[:, :, None]
        out[:, i] = (q[:, i, :, :, None] * state).sum(-2)
    return out, state


HEADS = pytest.mark.parametrize("hk,hv,dk,dv", [(4, 4, 64, 64), (2, 4, 128, 128), (1, 2, 64, 128),
                                                (3, 3, 128, 64)])


@HEADS
@pytest.mark.parametrize("batch,steps,held", [(1, 1, False), (2, 1, True), (2, 2, False), (2, 3, True),
                                              (1, 16, True), (2, 17, False), (1, 63, False),
                                              (1, 64, False), (2, 70, False), (1, 300, False)])
def test_conv_and_delta_rule(hk, hv, dk, dv, batch, steps, held):
    t = linear_case(batch, steps, hk, hv, dk, dv, steps + dk)
    q, k, v, conv = conv_exact(t, hk, hv, dk, dv, held)
    act = torch.empty(batch, steps, t["x"].shape[-1], device="cuda")
    gates = torch.stack([t["decay"], t["beta"]], -1).contiguous()
    _native.conv(t["x"], t["taps"], t["conv"], act, batch, steps, hk, hv, dk, dv, held)
    assert torch.equal(t["conv"].double(), conv)
    ref = torch.cat([q.flatten(2), k.flatten(2), v.flatten(2)], -1)
    close(act, ref, 1e-6 * (ref.abs() + 1))
    q, k, v = (a.double().reshape(batch, steps, -1, d) for a, d in
               zip(act.split([hk * dk, hk * dk, hv * dv], -1), (dk, dk, dv)))
    start = t["state"].double() if held else torch.zeros_like(t["state"]).double()
    want, ref = delta_exact(q, k, v, t["decay"].double(), t["beta"].double(), start)
    work = torch.full((_native.delta_workspace(batch, steps, hv, dk, dv),), float("nan"), device="cuda")
    forms = [lambda s, o: _native.delta_chunks(act, gates, s, o, work, batch, steps, hk, hv, dk, dv, held)]
    forms.append(lambda s, o: _native.delta_rule(act, gates, s, o, batch, steps, hk, hv, dk, dv, held))
    for form in forms:
        s, out = t["state"].clone(), torch.empty(batch, steps, hv, dv, device="cuda")
        form(s, out)
        # values of order 1, sums of up to 128 terms, remembered for some tens of tokens
        close(s, ref, 4e-6 * (1 + ref.abs()))
        close(out, want, 4e-6 * (1 + want.abs()))


def test_delta_rule_forgets_without_overflow():
    """Log decays from 0 to -1000 in one chunk: ratios of decays neither over- nor underflow
    into the tokens that remember, and infinite decay clears the state."""
    t = linear_case(1, 130, 2, 2, 128, 128, 5)
    t["decay"][0, :, 0] = torch.where(torch.arange(130, device="cuda") % 9 == 4, -1000.0, -1e-3)
    t["decay"][0, 70, 1] = -1e30
    q, k, v, _ = conv_exact(t, 2, 2, 128, 128, False)
    act = torch.cat([q.flatten(2), k.flatten(2), v.flatten(2)], -1).float()
    gates = torch.stack([t["decay"], t["beta"]], -1).contiguous()
    q, k, v = (a.double().reshape(1, 130, 2, 128) for a in act.split(256, -1))
    want, ref = delta_exact(q, k, v, t["decay"].double(), t["beta"].double(),
                            torch.zeros_like(t["state"]).double())
    work = torch.empty(_native.delta_workspace(1, 130, 2, 128, 128), device="cuda")
    s, out = t["state"].clone(), torch.empty(1, 130, 2, 128, device="cuda")
    _native.delta_chunks(act, gates, s, out, work, 1, 130, 2, 2, 128, 128, False)
    close(s, ref, 4e-6 * (1 + ref.abs()))
    close(out, want, 4e-6 * (1 + want.abs()))


@pytest.mark.parametrize("rows,dim,hv", [(1, 64, 4), (17, 256, 16), (40, 2048, 16), (33, 576, 20)])
def test_gates(rows, dim, hv):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    h, wa, wb = bf16(gen, rows, dim), bf16(gen, hv, dim, scale=0.05), bf16(gen, hv, dim, scale=0.05)
    a_log, dt = bf16(gen, hv), bf16(gen, hv, scale=3)
    out = torch.empty(rows, hv, 2, device="cuda")
    _native.gates(h, wa, wb, a_log, dt, out)
    a, b = h.double() @ wa.double().T, h.double() @ wb.double().T
    # float32 products of up to 2048 terms of size about 0.05
    ref = -a_log.double().exp() * F.softplus(a + dt.double())
    close(out[..., 0], ref, 2e-5 * (0.1 + ref.abs()) * a_log.double().exp().clamp(min=1))
    close(out[..., 1], torch.sigmoid(b), 1e-5 + 0 * b)


@pytest.mark.parametrize("d,half", [(64, 8), (128, 64), (256, 32)])
def test_rope_and_page_write(d, half):
    gen = torch.Generator(device="cuda").manual_seed(d)
    batch, steps, hq, hkv, start = 2, 5, 4, 2, 254
    q, k, v = bf16(gen, batch, steps, hq, 2, d), bf16(gen, batch, steps, hkv, d), bf16(gen, batch, steps, hkv, d)
    wq, wk = bf16(gen, d, scale=0.1), bf16(gen, d, scale=0.1)
    inv = (10000.0 ** (-torch.arange(half, device="cuda") / half)).to(torch.bfloat16)
    positions = torch.arange(start, start + steps, device="cuda")
    tables = torch.tensor([[3, 1], [0, -1]], dtype=torch.int32, device="cuda")
    pages = torch.full((2, 4, 256, hkv, d), 7.0, device="cuda", dtype=torch.bfloat16)
    rope = torch.empty(steps, half, 2, device="cuda")
    _native.rope_table(positions, inv, rope)
    angle = positions.double()[:, None] * inv.double()
    close(rope[..., 0], angle.cos(), 2e-7 + 0 * angle)
    close(rope[..., 1], angle.sin(), 2e-7 + 0 * angle)
    q_out, k_out = torch.empty(batch, steps, hq, d, device="cuda").bfloat16(), torch.empty_like(k)
    _native.qk_rope(q, k, v, wq, wk, rope, q_out, k_out, pages[0], pages[1], tables, positions, batch,
                    steps, hq, hkv, d, half, 1e-6)

    def turned(x, w):
        x = x.double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1 + w.double())
        a, b, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
        c, s = angle.cos()[:, None], angle.sin()[:, None]
        return torch.cat([a * c - b * s, b * c + a * s, rest], -1)

    for got, x, w in ((q_out, q[..., 0, :], wq), (k_out, k, wk)):
        ref = turned(x, w)
        close(got, ref, 1e-5 + 0 * ref, bf16_out=True)
    want = torch.full_like(pages, 7.0)
    for i, at in enumerate(positions.tolist()):
        for b in range(batch):
            page = int(tables[b, at // 256])
            if page >= 0:
                want[0, page, at % 256], want[1, page, at % 256] = k_out[b, i], v[b, i]
    assert torch.equal(pages, want)


@pytest.mark.parametrize("hk,hv,dk,dv,length", [(4, 4, 64, 64, 1), (2, 4, 128, 128, 8), (2, 4, 128, 128, 19),
                                                (2, 2, 64, 128, 300)])
def test_layers_agree_with_the_modules(hk, hv, dk, dv, length):
    """One model on the kernels and, with a hook on a layer, on transformers' modules."""
    cfg = H.decoder_config(num_hidden_layers=4, hidden_size=256, intermediate_size=512,
                           vocab_size=512, linear_num_key_heads=hk, linear_key_head_dim=dk,
                           linear_num_value_heads=hv, linear_value_head_dim=dv)
    model = H.random_init_model(cfg, "cuda", seed=1)
    prompt = [[(7 * i + j) % 512 for i in range(length)] for j in range(2)]
    results = []
    for hooked in (False, True):
        handle = model.model.layers[1].mlp.register_forward_hook(lambda *a: None) if hooked else None
        runner = H.HybridRunner(model=model, backend="hip_matched", batch=2, max_context=400)
        assert (DL.decoder_weights(model, runner.cache.pool.block.device) is None) == hooked
        logits = [runner.prefill(prompt)]
        for s in range(3):
            logits.append(runner.decode_step(torch.tensor([5 + s, 9 + s], device="cuda"), length + s))
        states = [t.float().clone() for t in runner.cache.state_tensors()]
        pages = runner.cache.pool.tables[:, 0].long()
        results.append((logits, states, runner.cache.pool.block[:, :, pages, :min(length, 256)].float()))
        if handle:
            handle.remove()
    # bf16 roundings at different places, through four layers
    for a, b in zip(results[0][0] + results[0][1] + [results[0][2]],
                    results[1][0] + results[1][1] + [results[1][2]]):
        assert (a.float() - b.float()).norm() <= 0.03 * b.float().norm()


@pytest.mark.parametrize("rows", [1, 127, 128, 129, 300])
@pytest.mark.parametrize("dim,features", [(64, (4, 100)), (128, (128,)), (192, (260, 4, 128)),
                                          (256, (384,)), (320, (36, 64)), (2048, (132,)),
                                          (384, (252, 516)), (448, (256,))])
@pytest.mark.parametrize("tile", [128, 256])
def test_linears(rows, dim, features, tile):
    gen = torch.Generator(device="cuda").manual_seed(rows + dim)
    x = bf16(gen, rows, dim)
    weights = [bf16(gen, f, dim, scale=dim ** -0.5) for f in features]
    outs = [torch.empty(rows, f, device="cuda", dtype=torch.bfloat16) for f in features]
    _native.linears(x, weights, outs, tile=tile)
    for w, out in zip(weights, outs):
        # float32 sums of dim products of order dim^-1/2
        close(out, x.double() @ w.double().T, 1e-5, bf16_out=True)


@pytest.mark.parametrize("rows,dim,features", [(1, 64, 4), (130, 192, 68), (257, 2048, 200), (129, 448, 132)])
@pytest.mark.parametrize("tile", [128, 256])
def test_linears_of_gate_and_up(rows, dim, features, tile):
    gen = torch.Generator(device="cuda").manual_seed(rows + dim)
    x = bf16(gen, rows, dim)
    gate, up = (bf16(gen, features, dim, scale=2 * dim ** -0.5) for _ in range(2))
    out = torch.empty(rows, features, device="cuda", dtype=torch.bfloat16)
    _native.linears(x, (gate, up), (out,), _native.LINEAR_SILU_MUL, tile)
    a, b = x.double() @ gate.double().T, x.double() @ up.double().T
    close(out, F.silu(a) * b, 1e-4, bf16_out=True)


def test_other_batches_are_refused_as_before():
    cfg = H.decoder_config(num_hidden_layers=4, hidden_size=256, intermediate_size=512,
                           vocab_size=512, linear_num_key_heads=4, linear_key_head_dim=64,
                           linear_num_value_heads=4, linear_value_head_dim=64)
    model = H.random_init_model(cfg, "cuda", seed=1)
    for rows in (1, 3):
        runner = H.HybridRunner(model=model, backend="hip_matched", batch=2, max_context=300)
        with pytest.raises((RuntimeError, ValueError)):
            runner.prefill([[1, 2, 3]] * rows)


def small_model(layers=4, **overrides):
    sizes = dict(hidden_size=256, intermediate_size=512, vocab_size=512, linear_num_key_heads=4,
                 linear_key_head_dim=64, linear_num_value_heads=4, linear_value_head_dim=64)
    return H.random_init_model(H.decoder_config(num_hidden_layers=layers, **{**sizes, **overrides}),
                               "cuda", seed=1)


@pytest.mark.parametrize("length", [5, 40])
def test_layers_read_the_general_prefill_form(length):
    """A scale that the prefill kernel does not take sends the attention to its PyTorch form,
    in the few-row and in the row layers; outputs differ by the attention's roundings."""
    model = small_model()
    prompt = [[(7 * i + 3 * j) % 512 for i in range(length)] for j in range(2)]
    runner = H.HybridRunner(model=model, backend="hip_matched", batch=2, max_context=300)
    want = runner.prefill(prompt).float()
    module = runner.attention_modules[0]
    q = torch.zeros(1, 8, 4, 256, device="cuda", dtype=torch.bfloat16)
    assert not PF._batched_ok(q, q[:, :2], q[:, :2], np.float32(module.scaling))
    module.scaling = np.float32(module.scaling)
    assert DL.decoder_weights(model, runner.cache.pool.block.device) is not None
    got = runner.prefill(prompt).float()
    assert (got - want).norm() <= 0.01 * want.norm()


def generation(model, batch, length, modules, steps=3, mode="eager"):
    """Logits of a prompt and of decode steps, then states and pages; phase 0 is the prompt,
    phase i decode step i, and `modules` the phases that run on transformers' modules."""
    vocab = model.config.vocab_size
    runner = H.HybridRunner(model=model, backend="hip_matched", batch=batch, mode=mode,
                            max_context=length + steps + 1)
    runner.cache.pool.block.zero_()
    prompt = [[(7 * i + 31 * j + 3) % vocab for i in range(length)] for j in range(batch)]
    fed = [torch.tensor([(5 + 13 * s + 7 * j) % vocab for j in range(batch)], device="cuda")
           for s in range(steps)]
    logits = []
    for phase in range(steps + 1):
        handle = (model.model.layers[1].mlp.register_forward_hook(lambda *a: None)
                  if phase in modules else None)
        assert (DL.decoder_weights(model, runner.cache.pool.block.device) is None) == bool(handle)
        logits.append((runner.prefill(prompt) if phase == 0 else
                       runner.decode_step(fed[phase - 1], length + phase - 1)).float().clone())
        if handle:
            handle.remove()
    return logits + [t.float() for t in runner.cache.state_tensors()] + [runner.cache.pool.block.float()]


def agree(got, want, rel):
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).norm() <= rel * b.norm(), (i, float((a - b).norm() / b.norm()))


ALL = (0, 1, 2, 3)


@pytest.mark.parametrize("batch", [1, 3, 8, 16, 17, 20])
@pytest.mark.parametrize("length", [1, 5])
def test_batches_agree_with_the_modules(batch, length):
    """Few-row, one-token and row forms of the prompt and of the steps: up to 16 rows the
    one-token products, more the row form, whose steps continue held states."""
    model = small_model()
    # bf16 roundings at different places, through four layers
    agree(generation(model, batch, length, ()), generation(model, batch, length, ALL), 0.03)


@pytest.mark.parametrize("modules", [(1, 2, 3), (0,), (2,), (0, 2)])
@pytest.mark.parametrize("batch", [2, 18])
def test_kernels_and_modules_take_turns(batch, modules):
    """States, pages and lengths are the same to either, in mid-generation too."""
    model = small_model()
    agree(generation(model, batch, 9, modules), generation(model, batch, 9, ()), 0.03)


@pytest.mark.parametrize("batch", [4, 18])
def test_captured_steps_of_batches(batch):
    model = small_model()
    runs = [generation(model, batch, 6, (), mode=mode) for mode in ("graph", "eager")]
    for a, b in zip(*runs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("batch,length", [(1, 300), (2, 130), (1, 40), (3, 4), (16, 1), (20, 3)])
def test_full_width_is_as_exact_as_the_modules(batch, length):
    """The decoder's own widths (hidden 2048, 16 linear heads of 128, vocabulary 151936): the
    logits are no further from those of the same weights in float64 than transformers' bf16
    modules leave them, but for a fifth, as both are draws of the same roundings."""
    model = H.random_init_model(H.decoder_config(num_hidden_layers=4), "cuda", seed=1)
    exact = copy.deepcopy(model).double()
    exact.config._attn_implementation = exact.model.config._attn_implementation = "eager"
    vocab, steps = model.config.vocab_size, 2
    kernels = generation(model, batch, length, (), steps)
    modules = generation(model, batch, length, ALL, steps)
    tokens = torch.tensor([[(7 * i + 31 * j + 3) % vocab for i in range(length)]
                           + [(5 + 13 * s + 7 * j) % vocab for s in range(steps)]
                           for j in range(batch)], device="cuda")
    with torch.inference_mode():
        want = exact(tokens, use_cache=False, logits_to_keep=steps + 1).logits
    for s in range(steps + 1):
        off = [float((x[s] - want[:, s]).norm() / want[:, s].norm()) for x in (kernels, modules)]
        assert off[0] <= 1.2 * off[1] and off[1] < 0.05, (s, off)
