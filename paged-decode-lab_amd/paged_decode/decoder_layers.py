"""The decoder's layers on this library's kernels.

``decoder_weights`` reads the model's modules and says whether every one of them is the
plain form the kernels compute; ``decoder_forward`` is then one forward of the model, with
the residual stream, the norms, the gated delta rule, rotary embedding, the K/V write and
the gates in HIP kernels between the matrix products.  Up to ``TOKEN_ROWS`` rows run the
products in them too.  A model that was changed (hooks, replaced or compiled modules,
biases, other dtypes or sizes, patched classes or functions of its file) keeps transformers'
modules: the weights are read from the modules on every forward, nothing is kept of them.
"""
import operator
import os
import types
from dataclasses import dataclass

import torch
import torch.nn.functional as F
import transformers
from torch import nn
from transformers.activations import SiLUActivation
from transformers.models.qwen3_5 import modeling_qwen3_5 as qwen
from transformers.models.qwen3_5.modeling_qwen3_5 import (
    Qwen3_5Attention, Qwen3_5DecoderLayer, Qwen3_5GatedDeltaNet, Qwen3_5MLP, Qwen3_5RMSNorm,
    Qwen3_5RMSNormGated, Qwen3_5TextRotaryEmbedding)

from . import _native
from .prefill import batched_prefill, device_cus

MAX_HIDDEN = 8192       # add_rms_norm keeps a row in the registers of one workgroup
TOKEN_ROWS = 16         # rows of one MFMA operand
MAX_BATCH, MAX_STEPS = 65535, 65535 * 16    # what the convolution's grid holds
# Tokens of a sequence from which the delta rule runs in chunks.  The recurrence and the
# chunks take 14 and 20 us at 64 tokens of one sequence, 19 and 23 at 96, 24 and 23 at 128 (16
# heads of 128 x 128); of two sequences 24 and 24 at 96, of four 28 and 33 at 96 and 35 and 34
# at 128, of eight 42 and 37 at 64 and 60 and 51 at 96.  The lines of one and of eight
# sequences are as far from 96; neither costs 6 us.
CHUNK_STEPS = 96

KINDS = (nn.Embedding, nn.Linear, nn.Conv1d, SiLUActivation, Qwen3_5Attention, Qwen3_5DecoderLayer,
         Qwen3_5GatedDeltaNet, Qwen3_5MLP, Qwen3_5RMSNorm, Qwen3_5RMSNormGated,
         Qwen3_5TextRotaryEmbedding)


def _definitions():
    """(getter, owner, names, values) of what runs in a plain layer: the functions and classes
    of the model's file, and the methods that a call of each kind goes through, found on the
    class as a call finds them."""
    space = vars(qwen)
    names = [n for n, f in space.items()
             if isinstance(f, types.FunctionType) and f.__module__ == qwen.__name__]
    names += [k.__name__ for k in KINDS if k.__module__ == qwen.__name__]
    found = [(operator.itemgetter(*names), space, names)]
    for kind in KINDS:
        own = {n for c in kind.__mro__ if c not in (nn.Module, object) for n, f in vars(c).items()
               if isinstance(f, types.FunctionType)}
        names = sorted(own - {"__init__", "__setstate__", "extra_repr", "reset_parameters"}
                       | {"forward", "__call__", "_call_impl", "_wrapped_call_impl", "__getattr__"})
        found.append((operator.attrgetter(*names), kind, names))
    return [(get, owner, names, get(owner)) for get, owner, names in found]


def _installed(value):
    """A function of the installed packages, or no function."""
    code = getattr(value, "__code__", None)
    return code is None or code.co_filename.startswith(
        tuple(os.path.dirname(p.__file__) + os.sep for p in (torch, transformers)))


# Compared on every forward: a patch made after this import shows as another value, one made
# before it as a function or class of another file.
_DEFINITIONS = _definitions()
_INSTALLED = (all(_installed(value) for *_, values in _DEFINITIONS for value in values)
              and all(k.__module__.split(".")[0] in ("torch", "transformers") for k in KINDS))


def _as_installed():
    for get, owner, _, values in _DEFINITIONS:
        if get(owner) != values:
            return False
    return _INSTALLED


def _plain_module(module, kind):
    """`module` runs the forward its class defines and nothing else."""
    return (type(module) is kind and not module._forward_hooks and not module._forward_pre_hooks
            and "forward" not in module.__dict__ and module._compiled_call_impl is None
            and not module.training)


def _tensor(module, name, device, shape):
    t = module._parameters.get(name)
    if (t is None or type(t) not in (nn.Parameter, torch.Tensor) or t.dtype != torch.bfloat16
            or t.device != device or t.shape != shape or not t.is_contiguous()
            or t.data_ptr() % 16):
        return None
    return t


class _Reader:
    """Collects the weights of plain modules; ``ok`` turns false at the first other one."""

    def __init__(self, device):
        self.device, self.ok = device, True

    def module(self, parent, name, kind):
        module = parent._modules.get(name)
        self.ok = self.ok and module is not None and _plain_module(module, kind)
        return module

    def weight(self, module, shape, name="weight"):
        t = _tensor(module, name, self.device, shape) if self.ok else None
        self.ok = self.ok and t is not None
        return t

    def linear(self, parent, name, rows, cols):
        module = self.module(parent, name, nn.Linear)
        if self.ok and module._parameters.get("bias") is not None:
            self.ok = False
        return self.weight(module, (rows, cols))

    def norm(self, parent, name, dim, kind=Qwen3_5RMSNorm):
        module = self.module(parent, name, kind)
        if not self.ok:
            return None, 0.0
        if kind is Qwen3_5RMSNorm:
            self.ok = "_norm" not in module.__dict__
            return self.weight(module, (dim,)), float(module.eps)
        self.ok = module.__dict__.get("activation", "silu") == "silu"
        return self.weight(module, (dim,)), float(module.variance_epsilon)


@dataclass
class LayerWeights:
    index: int
    module: object          # the attention module of a full-attention layer, else None
    mixer: tuple
    in_norm: tuple
    post_norm: tuple
    gate: torch.Tensor
    up: torch.Tensor
    down: torch.Tensor


@dataclass
class DecoderWeights:
    layers: list
    norm: tuple
    head: torch.Tensor
    inv_freq: torch.Tensor
    half: int               # rotated pairs per head
    linear: tuple           # (key heads, value heads, key dim, value dim)


def _linear_mixer(read, layer, cfg):
    hk, hv = cfg.linear_num_key_heads, cfg.linear_num_value_heads
    dk, dv, hid = cfg.linear_key_head_dim, cfg.linear_value_head_dim, cfg.hidden_size
    m = read.module(layer, "linear_attn", Qwen3_5GatedDeltaNet)
    if (not read.ok or (m.num_k_heads, m.num_v_heads, m.head_k_dim, m.head_v_dim) != (hk, hv, dk, dv)
            or m.conv_kernel_size != 4 or m.activation != "silu"):
        read.ok = False
        return None
    channels = 2 * hk * dk + hv * dv
    conv = read.module(m, "conv1d", nn.Conv1d)
    if read.ok and (conv._parameters.get("bias") is not None or conv.groups != channels
                    or conv.kernel_size != (4,) or conv.stride != (1,) or conv.dilation != (1,)
                    or conv.padding != (3,) or conv.padding_mode != "zeros"):
        read.ok = False
    return (read.linear(m, "in_proj_qkv", channels, hid), read.linear(m, "in_proj_z", hv * dv, hid),
            read.linear(m, "in_proj_b", hv, hid), read.linear(m, "in_proj_a", hv, hid),
            read.weight(conv, (channels, 1, 4)), read.weight(m, (hv,), "A_log"),
            read.weight(m, (hv,), "dt_bias"), read.norm(m, "norm", dv, Qwen3_5RMSNormGated),
            read.linear(m, "out_proj", hid, hv * dv))


def _full_mixer(read, layer, cfg):
    hq, hkv, d, hid = (cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim,
                       cfg.hidden_size)
    m = read.module(layer, "self_attn", Qwen3_5Attention)
    if not read.ok or m.head_dim != d:
        read.ok = False
        return None
    mixer = (read.linear(m, "q_proj", 2 * hq * d, hid), read.linear(m, "k_proj", hkv * d, hid),
             read.linear(m, "v_proj", hkv * d, hid), read.norm(m, "q_norm", d),
             read.norm(m, "k_norm", d), read.linear(m, "o_proj", hid, hq * d))
    if read.ok and mixer[3][1] != mixer[4][1]:
        read.ok = False
    return mixer


def decoder_weights(model, device):
    """The model's weights, or None when the kernels do not cover it as it is."""
    text, cfg = model.model, model.model.config
    hooks = nn.modules.module
    read = _Reader(device)
    if hooks._global_forward_hooks or hooks._global_forward_pre_hooks or not _as_installed():
        return None
    hk, hv = cfg.linear_num_key_heads, cfg.linear_num_value_heads
    dk, dv, hid, mid = (cfg.linear_key_head_dim, cfg.linear_value_head_dim, cfg.hidden_size,
                        cfg.intermediate_size)
    if (cfg._attn_implementation != "paged_decode_lab_hip" or hid % 64 or hid > MAX_HIDDEN or mid % 8
            or dk not in (64, 128) or dv not in (64, 128) or hk < 1 or hv % hk
            or cfg.head_dim not in (64, 128, 256)):
        return None
    embed = read.module(text, "embed_tokens", nn.Embedding)
    rope = read.module(text, "rotary_emb", Qwen3_5TextRotaryEmbedding)
    if not read.ok or read.weight(embed, (cfg.vocab_size, hid)) is None:
        return None
    inv = rope._buffers.get("inv_freq")
    if (rope.rope_type != "default" or rope.attention_scaling != 1.0 or inv is None
            or inv.dtype not in (torch.bfloat16, torch.float32) or inv.device != device
            or inv.dim() != 1 or not inv.is_contiguous() or not 0 < 2 * inv.shape[0] <= cfg.head_dim):
        return None
    layers = []
    for i, layer in enumerate(text.layers):
        full = cfg.layer_types[i] == "full_attention"
        if not _plain_module(layer, Qwen3_5DecoderLayer):
            return None
        mixer = _full_mixer(read, layer, cfg) if full else _linear_mixer(read, layer, cfg)
        mlp = read.module(layer, "mlp", Qwen3_5MLP)
        if not read.ok:
            return None
        read.module(mlp, "act_fn", SiLUActivation)
        layers.append(LayerWeights(
            i, layer._modules["self_attn"] if full else None, mixer,
            read.norm(layer, "input_layernorm", hid),
            read.norm(layer, "post_attention_layernorm", hid), read.linear(mlp, "gate_proj", mid, hid),
            read.linear(mlp, "up_proj", mid, hid), read.linear(mlp, "down_proj", hid, mid)))
        if not read.ok:
            return None
    weights = DecoderWeights(layers, read.norm(text, "norm", hid),
                             read.linear(model, "lm_head", cfg.vocab_size, hid), inv, inv.shape[0],
                             (hk, hv, dk, dv))
    return weights if read.ok else None


def _linear_states(cache, index, batch, weights, device):
    """(conv state, recurrent state, whether they hold earlier tokens) of one layer, made
    through the cache's own protocol on first use; None when they have another form."""
    hk, hv, dk, dv = weights.linear
    layer, channels = cache.linear[index], 2 * hk * dk + hv * dv
    held = cache.has_previous_state(index)
    if layer.conv_states.get(0) is None or layer.recurrent_states.get(0) is None:
        cache.update_conv_state(torch.zeros((batch, channels, 4), device=device,
                                            dtype=torch.bfloat16), index)
        cache.update_recurrent_state(torch.zeros((batch, hv, dk, dv), device=device,
                                                 dtype=torch.float32), index)
        held = False
    conv, state = layer.conv_states[0], layer.recurrent_states[0]
    if (conv.shape != (batch, channels, 4) or conv.dtype != torch.bfloat16
            or state.shape != (batch, hv, dk, dv) or state.dtype != torch.float32
            or not conv.is_contiguous() or not state.is_contiguous()
            or conv.data_ptr() % 16 or state.data_ptr() % 16):
        return None
    return conv, state, held


def decoder_states(runner, weights, tokens):
    """The linear-attention states of every layer, or None where the kernels cannot run:
    another batch than the runner's, more tokens than a grid holds, several steps on top of
    earlier tokens, or states of another form."""
    cache, found = runner.cache, {}
    if (tokens.dim() != 2 or tokens.shape[0] != runner.batch or tokens.shape[0] > MAX_BATCH
            or not 1 <= tokens.shape[1] <= MAX_STEPS):
        return None
    steps = tokens.shape[1]
    for index in cache.linear:
        states = _linear_states(cache, index, runner.batch, weights, runner.device)
        if states is None or (states[2] and steps > 1):
            return None
        found[index] = states
    return found


def _products(h, *matrices):
    """h times each matrix: one launch while its tiles are one round of the CUs
    (pd_linears), else the library's products."""
    rows, dim = h.shape
    features = [m.shape[0] for m in matrices]
    tile = _one_round_tile(rows, dim, features, h.device)
    if not tile:
        return [F.linear(h, m) for m in matrices]
    outs = [torch.empty((rows, f), device=h.device, dtype=h.dtype) for f in features]
    _native.linears(h, matrices, outs, tile=tile)
    return outs


def _gate_up(h, gate, up):
    """silu(h gate^T) (h up^T), on the same rule; half a tile's features are the gate's."""
    rows, dim = h.shape
    tile = gate.shape[0] % 4 == 0 and _one_round_tile(rows, dim, [2 * gate.shape[0]], h.device)
    if not tile:
        a, b = F.linear(h, gate), F.linear(h, up)
        _native.silu_mul(a, b, a)
        return a
    out = torch.empty((rows, gate.shape[0]), device=h.device, dtype=h.dtype)
    _native.linears(h, (gate, up), (out,), _native.LINEAR_SILU_MUL, tile)
    return out


def _one_round_tile(rows, dim, features, device):
    """The features of a tile whose 128-row tiles are one round of the CUs, 0 if none's are.
    The smaller tile is the faster one where both would do (24 and 36 us, 8192 features of
    2048 at 512 rows)."""
    if dim % 64 or any(f % 4 for f in features):
        return 0
    for tile in (128, 256):
        if sum(-(-f // tile) for f in features) * -(-rows // 128) <= device_cus(device):
            return tile
    return 0


def _delta_attention(h, mixed, gate, w, weights, states, batch, steps):
    """The layer's output before its projection, of the normed rows and their products."""
    hk, hv, dk, dv = weights.linear
    _, _, b, a, taps, a_log, dt_bias, (norm, eps), _ = w.mixer
    conv, state, held = states
    rows = batch * steps
    act = torch.empty((rows, mixed.shape[1]), device=h.device, dtype=torch.float32)
    gates = torch.empty((rows, hv, 2), device=h.device, dtype=torch.float32)
    _native.conv(mixed, taps, conv, act, batch, steps, hk, hv, dk, dv, held)
    _native.gates(h, a, b, a_log, dt_bias, gates)
    out = torch.empty((rows, hv * dv), device=h.device, dtype=torch.float32)
    if steps >= CHUNK_STEPS:
        work = torch.empty(_native.delta_workspace(batch, steps, hv, dk, dv), device=h.device,
                           dtype=torch.float32)
        _native.delta_chunks(act, gates, state, out, work, batch, steps, hk, hv, dk, dv, held)
    else:
        _native.delta_rule(act, gates, state, out, batch, steps, hk, hv, dk, dv, held)
    y = torch.empty((rows, hv * dv), device=h.device, dtype=torch.bfloat16)
    _native.gated_norm(out, gate, norm, y, rows * hv, dv, eps)
    return y


def _full_attention(h, w, weights, rope, runner, batch, steps, attend):
    spec, pool = runner.spec, runner.cache.pool
    hq, hkv, d = spec.num_heads, spec.num_kv_heads, spec.head_dim
    q_proj, k_proj, v_proj, (q_norm, eps), (k_norm, _), o_proj = w.mixer
    q, k, v = _products(h, q_proj, k_proj, v_proj)
    fill = runner.cache.phase == "prefill"
    query = torch.empty((batch, steps, hq, d), device=h.device, dtype=torch.bfloat16)
    keys = torch.empty((batch, steps, hkv, d), device=h.device, dtype=torch.bfloat16) if fill else None
    k_pages, v_pages = pool.pages(w.index)
    _native.qk_rope(q, k, v, q_norm, k_norm, rope, query, keys, k_pages, v_pages, pool.tables,
                    pool.positions, batch, steps, hq, hkv, d, weights.half, eps)
    if fill:
        out = batched_prefill(query.transpose(1, 2), keys.transpose(1, 2),
                              v.view(batch, steps, hkv, d).transpose(1, 2), w.module.scaling)
    else:
        out = attend(runner, w.module, query.view(batch, hq, d), k_pages, v_pages)
    y = torch.empty((batch * steps, hq * d), device=h.device, dtype=torch.bfloat16)
    _native.sigmoid_gate(out, q.view(-1, 2 * d)[:, d:], y, batch * steps * hq, d)
    return F.linear(y, o_proj)


def _token_form(weights, rows):
    """Few rows: products that read each weight once, with the norms, gates and residuals
    folded in.  The normed rows must fit a workgroup's LDS."""
    hid = weights.head.shape[1]
    mid = weights.layers[0].down.shape[1] if weights.layers else 64
    hk, hv, dk, dv = weights.linear
    full = [w.mixer[5].shape[1] for w in weights.layers if w.module is not None]
    return (rows <= TOKEN_ROWS and hid % 64 == 0 and mid % 64 == 0 and hv * dv % 64 == 0
            and all(k % 64 == 0 for k in full) and rows * (hid + 8) * 2 + 16384 <= 160 * 1024)


def _token_linear(x, w, weights, states, batch):
    """One token of each sequence: the convolution in the projection, the delta rule's
    single step with its gated norm."""
    hk, hv, dk, dv = weights.linear
    qkv, z, b, a, taps, a_log, dt_bias, (norm, eps), out_proj = w.mixer
    conv, state, held = states
    act = torch.empty((batch, qkv.shape[0]), device=x.device, dtype=torch.float32)
    rest = torch.empty((2 * batch * (hv * dv + 8 * hv)), device=x.device, dtype=torch.bfloat16)
    gate = rest[:batch * hv * dv]
    beta, decay = rest[gate.numel():], rest[gate.numel() + 8 * batch * hv:]
    out = rest[gate.numel() + 16 * batch * hv:]
    _native.norm_linears(x, w.in_norm[0], w.in_norm[1], (qkv, z, b, a), (act, gate, beta, decay), taps,
                         conv, held)
    _native.delta_step(act, decay, beta, a_log, dt_bias, gate, norm, eps, state, out, batch, hk, hv,
                       dk, dv, held)
    _native.linear_add(out, out_proj, x)


def _few_linear(x, w, weights, states, batch, steps):
    """Several tokens of each sequence, in few rows."""
    qkv, z, _, _, _, _, _, _, out_proj = w.mixer
    rows = lambda m: torch.empty((x.shape[0], m.shape[0]), device=x.device, dtype=x.dtype)  # noqa: E731
    mixed, gate, h = rows(qkv), rows(z), torch.empty_like(x)
    _native.norm_linears(x, w.in_norm[0], w.in_norm[1], (qkv, z), (mixed, gate))
    _native.add_rms_norm(x, None, w.in_norm[0], h, w.in_norm[1])
    _native.linear_add(_delta_attention(h, mixed, gate, w, weights, states, batch, steps), out_proj, x)


def _token_full(x, w, weights, rope, runner, batch, steps, attend):
    spec, pool = runner.spec, runner.cache.pool
    hq, hkv, d = spec.num_heads, spec.num_kv_heads, spec.head_dim
    q_proj, k_proj, v_proj, (q_norm, eps), (k_norm, _), o_proj = w.mixer
    rows = lambda *shape: torch.empty((batch, steps, *shape), device=x.device, dtype=x.dtype)  # noqa: E731
    q, k, v, query = rows(hq, 2 * d), rows(hkv, d), rows(hkv, d), rows(hq, d)
    _native.norm_linears(x, w.in_norm[0], w.in_norm[1], (q_proj, k_proj, v_proj), (q, k, v))
    k_pages, v_pages = pool.pages(w.index)
    fill = runner.cache.phase == "prefill"
    keys = torch.empty_like(k) if fill else None
    _native.qk_rope(q, k, v, q_norm, k_norm, rope, query, keys, k_pages, v_pages, pool.tables,
                    pool.positions, batch, steps, hq, hkv, d, weights.half, eps)
    if fill:
        out = batched_prefill(query.transpose(1, 2), keys.transpose(1, 2), v.transpose(1, 2),
                              w.module.scaling)
    else:
        out = attend(runner, w.module, query.view(batch, hq, d), k_pages, v_pages)
    _native.linear_add(out, o_proj, x, q[..., d:], d)


def _token_layers(x, runner, weights, states, rope, batch, steps, attend):
    """Up to TOKEN_ROWS rows, added to the residual stream x."""
    for w in weights.layers:
        if w.module is not None:
            _token_full(x, w, weights, rope, runner, batch, steps, attend)
        else:
            if steps == 1:
                _token_linear(x, w, weights, states[w.index], batch)
            else:
                _few_linear(x, w, weights, states[w.index], batch, steps)
            runner.cache.linear[w.index].has_previous_state[0] = True
        h = torch.empty((x.shape[0], w.gate.shape[0]), device=x.device, dtype=x.dtype)
        _native.norm_gate_up(x, w.post_norm[0], w.post_norm[1], w.gate, w.up, h)
        _native.linear_add(h, w.down, x)


def _row_layers(x, runner, weights, states, rope, batch, steps, attend):
    """Any number of rows: products with the kernels between them; returns the
    last layer's output, not yet added to the residual stream x."""
    y = None
    for w in weights.layers:
        h = torch.empty_like(x)
        _native.add_rms_norm(x, y, w.in_norm[0], h, w.in_norm[1])
        if w.module is None:
            mixed, gate = _products(h, w.mixer[0], w.mixer[1])
            y = F.linear(_delta_attention(h, mixed, gate, w, weights, states[w.index], batch, steps),
                         w.mixer[8])
            runner.cache.linear[w.index].has_previous_state[0] = True
        else:
            y = _full_attention(h, w, weights, rope, runner, batch, steps, attend)
        _native.add_rms_norm(x, y, w.post_norm[0], h, w.post_norm[1])
        y = F.linear(_gate_up(h, w.gate, w.up), w.down)
    return y


def decoder_forward(runner, weights, states, tokens, positions, attend):
    """Logits of the last token; as HybridRunner._forward, on the kernels.  ``attend`` is
    the decode attention of one layer over its pages."""
    text = runner.text
    batch, steps = tokens.shape
    runner.cache.pool.begin_step(positions)
    x = text.embed_tokens(tokens)
    hid = x.shape[-1]
    x = x.view(batch * steps, hid)
    rope = torch.empty((steps, weights.half, 2), device=x.device, dtype=torch.float32)
    _native.rope_table(positions, weights.inv_freq, rope)
    y = None
    if _token_form(weights, batch * steps):
        _token_layers(x, runner, weights, states, rope, batch, steps, attend)
    else:
        y = _row_layers(x, runner, weights, states, rope, batch, steps, attend)
    if steps > 1:
        x = x.view(batch, steps, hid)[:, -1].contiguous()
        y = y if y is None else y.view(batch, steps, hid)[:, -1].contiguous()
    norm, eps = weights.norm
    if _token_form(weights, batch):
        if y is not None:
            x = x + y
        logits = torch.empty((batch, weights.head.shape[0]), device=x.device, dtype=x.dtype)
        _native.norm_linears(x, norm, eps, (weights.head,), (logits,))
        return logits
    h = torch.empty_like(x)
    _native.add_rms_norm(x, y, norm, h, eps)
    return F.linear(h, weights.head)
