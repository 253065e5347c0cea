"""Timed cases: what programs built on this framework have it do.

Seven kinds of pass, each through a public entry point:

  matched     matched_decode: one decode step's attention, split-KV plan, fixed batch
  paged       paged_decode with hip_base or hip_splitk: the same on the engine's backends
  store       store_kvcache: new K/V rows into their cache slots
  layer_step  Attention.forward of the engine on a decode step (K/V write + attention)
  layer_fill  Attention.forward of the engine on a prefill of several sequences, with or
              without a cached prefix (K/V write + causal attention)
  model_step  HybridRunner.decode_step: the decoder's logits for one more token per sequence
  model_fill  HybridRunner.prefill: the decoder's logits after a prompt

``prepare`` builds what such a program keeps (caches, tables, plans, weights, a captured
step), ``run`` makes one pass, ``exact`` restates the result in 64 bits in plain torch.
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _path in (_ROOT, os.path.join(_ROOT, "paged-decode-lab_amd")):
    if _path not in sys.path:
        sys.path.insert(0, _path)

from paged_decode import hybrid  # noqa: E402
from paged_decode.engine_attention import Attention, reset_context, set_context  # noqa: E402
from paged_decode.kv_write import store_kvcache  # noqa: E402
from paged_decode.matched_splitkv import allocate_matched_resources, matched_decode  # noqa: E402
from paged_decode.runtime import allocate_resources, paged_decode  # noqa: E402
from paged_decode.spec import DecodeSpec  # noqa: E402

PAGE = 256
DEV = "cuda"
STEPS = 64                      # decode positions a model_step state cycles through

# (query heads, kv heads, head dim) of the benchmark, the engine tests and the edge batches
GEOMETRIES = [(16, 4, 256), (32, 8, 128), (32, 4, 256), (16, 16, 64), (16, 8, 128), (8, 2, 128)]

# Widths of the end-to-end decoder, and of the small one its tests use.
WIDTHS = {
    "full": dict(hidden_size=2048, intermediate_size=6144, vocab_size=151936,
                 linear_num_key_heads=16, linear_key_head_dim=128,
                 linear_num_value_heads=16, linear_value_head_dim=128),
    "small": dict(hidden_size=256, intermediate_size=512, vocab_size=512,
                  linear_num_key_heads=4, linear_key_head_dim=64,
                  linear_num_value_heads=4, linear_value_head_dim=64),
}
HQ, HKV, HEAD, CONV = 8, 2, 256, 4      # the decoder's full-attention heads, its conv taps


def listed():
    return [
        # the benchmark's headline: one sequence, a short context, latency-bound
        {"name": "matched_ctx2064", "kind": "matched", "batch": 1, "hq": 16, "hkv": 4, "dim": 256,
         "low": 2064, "high": 2064},
        # the same model at a long context: one sequence over the whole chip
        {"name": "matched_ctx32768", "kind": "matched", "batch": 1, "hq": 16, "hkv": 4,
         "dim": 256, "low": 32768, "high": 32768},
        # a serving batch of a multi-head model, lengths spread up to 4096 tokens
        {"name": "splitk_b128_mha64", "kind": "paged", "backend": "hip_splitk", "batch": 128,
         "hq": 16, "hkv": 16, "dim": 64, "low": 1, "high": 4096},
        # the bandwidth sweep: 64 long-context sequences of a grouped-query model
        {"name": "base_b64_gqa128", "kind": "paged", "backend": "hip_base", "batch": 64,
         "hq": 32, "hkv": 8, "dim": 128, "low": 1, "high": 32768},
        # one layer of a small serving batch's eager decode step
        {"name": "layer_step_b8", "kind": "layer_step", "backend": "hip_splitk", "batch": 8,
         "hq": 32, "hkv": 8, "dim": 128, "low": 1024, "high": 4096},
        # one layer of a prefill batch: ragged prompts packed into one call
        {"name": "layer_fill_ragged", "kind": "layer_fill", "batch": 4, "hq": 32, "hkv": 8,
         "dim": 128, "low": 17, "high": 2048, "prefix": 0},
        # one layer of a prompt's tail whose first 3072 tokens are in the prefix cache
        {"name": "layer_fill_prefix", "kind": "layer_fill", "batch": 1, "hq": 16, "hkv": 4,
         "dim": 256, "low": 1000, "high": 1000, "prefix": 3072},
        # the K/V write of a prompt's chunk
        {"name": "store_2048", "kind": "store", "rows": 2048, "hkv": 8, "dim": 128},
        # the decoder serving one user: one token through 24 layers and the head, captured
        {"name": "model_step_24l", "kind": "model_step", "width": "full", "layers": 24,
         "batch": 1, "prompt": 512, "backend": "hip_matched", "mode": "graph"},
        # four of its layers for a few users at once, run eagerly
        {"name": "model_step_4l_b4", "kind": "model_step", "width": "full", "layers": 4,
         "batch": 4, "prompt": 1500, "backend": "hip_splitk", "mode": "eager"},
        # the whole decoder's time to first token on a short prompt
        {"name": "model_fill_24l", "kind": "model_fill", "width": "full", "layers": 24,
         "batch": 1, "prompt": 512, "backend": "hip_matched"},
        # four layers on a long prompt of odd length
        {"name": "model_fill_4l_long", "kind": "model_fill", "width": "full", "layers": 4,
         "batch": 1, "prompt": 2049, "backend": "hip_matched"},
    ]


def _log(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["matched", "paged", "store", "layer_step", "layer_fill", "model_step",
                       "model_fill"])
    if kind == "store":
        hq, hkv, dim = rng.choice(GEOMETRIES)
        return {"kind": kind, "rows": _log(rng, 1, 16384), "hkv": hkv, "dim": dim}
    if kind in ("model_step", "model_fill"):
        case = {"kind": kind, "width": rng.choice(["full", "full", "small"]),
                "layers": rng.choice([4, 8]), "batch": rng.choice([1, 1, 2, 3, 4, 8]),
                "backend": rng.choice(["hip_matched", "hip_base", "hip_splitk"])}
        case["prompt"] = _log(rng, 1, 3072 // case["batch"])
        if kind == "model_step":
            case["mode"] = rng.choice(["graph", "eager"])
        return case
    hq, hkv, dim = rng.choice(GEOMETRIES)
    case = {"kind": kind, "hq": hq, "hkv": hkv, "dim": dim}
    if kind == "layer_fill":
        case["batch"] = _log(rng, 1, 8)
        case["prefix"] = rng.choice([0, 0, 256 * _log(rng, 1, 12)])
        case["high"] = _log(rng, 1, 4096 // case["batch"])
        case["low"] = rng.randint(1, case["high"])
        return case
    case["batch"] = _log(rng, 1, 128)
    most = min(131072, int(3e9) // (case["batch"] * hkv * dim * 4))
    case["high"] = _log(rng, 16, most)
    case["low"] = rng.choice([1, case["high"]])
    if kind != "matched":
        case["backend"] = rng.choice(["hip_base", "hip_splitk"])
    return case


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)


def _lengths(case):
    """Tokens per sequence in [low, high], one of them high itself; the same for every seed,
    so that outputs keep their shapes."""
    rng = np.random.default_rng([case["low"], case["high"], case["batch"]])
    lens = rng.integers(case["low"], case["high"] + 1, case["batch"])
    lens[rng.integers(case["batch"])] = case["high"]
    return [int(n) for n in lens]


def _tables(lens, seed):
    """Physical pages of each sequence, in a random order over the pool."""
    pages = [-(-n // PAGE) for n in lens]
    order = [int(p) for p in np.random.default_rng([seed, 2]).permutation(sum(pages))]
    return [[order.pop() for _ in range(n)] for n in pages], sum(pages)


def _table_tensor(tables, width=None):
    width = width or max(len(t) for t in tables)
    return torch.tensor([t + [-1] * (width - len(t)) for t in tables], dtype=torch.int32,
                        device=DEV)


def _slots(tables, starts, lens):
    """Cache slots of tokens [start, length) of every sequence, in order."""
    slots = np.concatenate([np.asarray(t, np.int64)[np.arange(a, n) // PAGE] * PAGE
                            + np.arange(a, n) % PAGE for t, a, n in zip(tables, starts, lens)])
    return torch.from_numpy(slots.astype(np.int32)).to(DEV)


def _attention_inputs(case, seed):
    """Host geometry and device tensors of one attention call, from the seed alone."""
    gen = _generator(seed)
    fill = case["kind"] == "layer_fill"
    new = _lengths(case)
    lens = [case["prefix"] + n for n in new] if fill else new
    starts = [case["prefix"]] * len(new) if fill else [n - 1 for n in lens]
    tables, pages = _tables(lens, seed)
    rows = sum(new) if fill else len(lens)
    hq, hkv, dim = case["hq"], case["hkv"], case["dim"]
    return dict(lens=lens, starts=starts, tables=tables,
                q=_normal(gen, rows, hq, dim), key=_normal(gen, rows, hkv, dim),
                value=_normal(gen, rows, hkv, dim), k=_normal(gen, pages, PAGE, hkv, dim),
                v=_normal(gen, pages, PAGE, hkv, dim))


def _store_inputs(case, seed):
    gen = _generator(seed)
    rows, shape = case["rows"], (case["hkv"], case["dim"])
    blocks = -(-rows // PAGE) + 8
    slots = np.random.default_rng([seed, 3]).permutation(blocks * PAGE)[:rows].astype(np.int32)
    return dict(key=_normal(gen, rows, *shape), value=_normal(gen, rows, *shape),
                k=_normal(gen, blocks, PAGE, *shape), v=_normal(gen, blocks, PAGE, *shape),
                slots=torch.from_numpy(slots).to(DEV))


def _kinds(layers):
    return ["full_attention" if (i + 1) % 4 == 0 else "linear_attention" for i in range(layers)]


def _parameter_shapes(case):
    w = WIDTHS[case["width"]]
    hid, mid = w["hidden_size"], w["intermediate_size"]
    hk, dk = w["linear_num_key_heads"], w["linear_key_head_dim"]
    hv, dv = w["linear_num_value_heads"], w["linear_value_head_dim"]
    conv = 2 * hk * dk + hv * dv
    shapes = {"model.embed_tokens.weight": (w["vocab_size"], hid)}
    for i, kind in enumerate(_kinds(case["layers"])):
        at = f"model.layers.{i}."
        shapes[at + "input_layernorm.weight"] = (hid,)
        if kind == "linear_attention":
            at += "linear_attn."
            shapes.update({at + "in_proj_qkv.weight": (conv, hid),
                           at + "in_proj_z.weight": (hv * dv, hid),
                           at + "in_proj_b.weight": (hv, hid), at + "in_proj_a.weight": (hv, hid),
                           at + "conv1d.weight": (conv, 1, CONV), at + "A_log": (hv,),
                           at + "dt_bias": (hv,), at + "norm.weight": (dv,),
                           at + "out_proj.weight": (hid, hv * dv)})
        else:
            at += "self_attn."
            shapes.update({at + "q_proj.weight": (2 * HQ * HEAD, hid),
                           at + "k_proj.weight": (HKV * HEAD, hid),
                           at + "v_proj.weight": (HKV * HEAD, hid),
                           at + "q_norm.weight": (HEAD,), at + "k_norm.weight": (HEAD,),
                           at + "o_proj.weight": (hid, HQ * HEAD)})
        at = f"model.layers.{i}."
        shapes.update({at + "post_attention_layernorm.weight": (hid,),
                       at + "mlp.gate_proj.weight": (mid, hid),
                       at + "mlp.up_proj.weight": (mid, hid),
                       at + "mlp.down_proj.weight": (hid, mid)})
    shapes["model.norm.weight"] = (hid,)
    shapes["lm_head.weight"] = (w["vocab_size"], hid)
    return shapes


def _draw_parameter(name, out, gen):
    """A trained decoder's spread: N(0, 0.02) matrices, smaller ones into the residual stream,
    which the embedding dominates at first, norms near their identity, and decay rates that
    remember a few tokens or hundreds."""
    if name.endswith("A_log"):
        return out.uniform_(0.0, 2.7, generator=gen)
    if name.endswith("dt_bias"):
        return out.normal_(-3.0, 1.0, generator=gen)
    if "norm" in name:
        return out.normal_(1.0 if "linear_attn.norm" in name else 0.0, 0.1, generator=gen)
    spread = {"embed_tokens": 1.0, "conv1d": 0.3, "o_proj": 0.003, "out_proj": 0.003,
              "down_proj": 0.003}
    return out.normal_(0.0, next((v for k, v in spread.items() if k in name), 0.02),
                       generator=gen)


def _model_tokens(case, seed):
    """The prompt [batch][prompt] and the tokens fed afterwards [STEPS][batch]."""
    rng = np.random.default_rng([seed, 4])
    vocab = WIDTHS[case["width"]]["vocab_size"]
    return (rng.integers(0, vocab, (case["batch"], case["prompt"])),
            rng.integers(0, vocab, (STEPS, case["batch"])))


def _model_runner(case, seed):
    config = hybrid.decoder_config(num_hidden_layers=case["layers"], **WIDTHS[case["width"]])
    model = hybrid.random_init_model(config, DEV, 0)
    gen = _generator(seed)
    for name in _parameter_shapes(case):
        _draw_parameter(name, model.get_parameter(name).data, gen)
    runner = hybrid.HybridRunner(model=model, backend=case["backend"], mode=case.get("mode", "eager"),
                                 batch=case["batch"], max_context=case["prompt"] + STEPS)
    runner.cache.pool.block.zero_()
    return runner


def prepare(case, seed):
    kind = case["kind"]
    if kind == "store":
        return dict(case=case, **_store_inputs(case, seed))
    if kind in ("model_step", "model_fill"):
        prompt, fed = _model_tokens(case, seed)
        state = dict(case=case, runner=_model_runner(case, seed), prompt=prompt.tolist())
        if kind == "model_step":
            state["fed"], state["step"] = torch.from_numpy(fed).to(DEV), 1
            state["runner"].prefill(state["prompt"])
            # the first step, which captures the graph in graph mode
            state["runner"].decode_step(state["fed"][0], case["prompt"])
        return state
    inputs = _attention_inputs(case, seed)
    lens, tables = inputs["lens"], inputs["tables"]
    state = dict(case=case, inputs=inputs,
                 lengths=torch.tensor(lens, dtype=torch.int32, device=DEV))
    hq, hkv, dim, batch = case["hq"], case["hkv"], case["dim"], case["batch"]
    if kind in ("matched", "paged", "layer_step"):
        spec = DecodeSpec(batch, hq, hkv, dim, case["high"])
        state["tables"] = _table_tensor(tables, spec.table_width)
        state["resources"] = (allocate_matched_resources(spec, DEV) if kind == "matched" else
                              allocate_resources(spec, DEV, case["backend"]))
    if kind.startswith("layer"):
        layer = Attention(hq, dim, dim ** -0.5, hkv)
        layer.k_cache, layer.v_cache = inputs["k"], inputs["v"]
        if kind == "layer_step":
            layer.decode_backend, layer.decode_resources = case["backend"], state["resources"]
        state["layer"] = layer
        state["slots"] = _slots(tables, inputs["starts"], lens)
    if kind == "layer_fill":
        new = [n - a for a, n in zip(inputs["starts"], lens)]
        cu = lambda ns: torch.tensor(np.cumsum([0] + ns), dtype=torch.int32, device=DEV)  # noqa: E731
        state.update(cu_q=cu(new), cu_k=cu(lens), max_q=max(new), max_k=max(lens),
                     tables=_table_tensor(tables) if case["prefix"] else None)
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "store":
        store_kvcache(state["key"], state["value"], state["k"], state["v"], state["slots"])
        return state["k"], state["v"]
    if kind in ("model_step", "model_fill"):
        runner = state["runner"]
        if kind == "model_fill":
            logits = runner.prefill(state["prompt"])
        else:
            step = state["step"]
            state["step"] = step % (STEPS - 1) + 1
            logits = runner.decode_step(state["fed"][step], case["prompt"] + step)
        return {"logits": logits, "states": runner.cache.state_tensors(),
                "pages": runner.cache.pool.block}
    x = state["inputs"]
    if kind == "matched":
        return matched_decode(x["q"], x["k"], x["v"], state["tables"], state["lengths"],
                              resources=state["resources"])
    if kind == "paged":
        return paged_decode(x["q"], x["k"], x["v"], state["tables"], state["lengths"],
                            resources=state["resources"], backend=case["backend"])
    if kind == "layer_step":
        set_context(False, slot_mapping=state["slots"], context_lens=state["lengths"],
                    block_tables=state["tables"])
    else:
        set_context(True, state["cu_q"], state["cu_k"], state["max_q"], state["max_k"],
                    state["slots"], block_tables=state["tables"])
    out = state["layer"](x["q"], x["key"], x["value"])
    reset_context()
    return {"out": out, "k": x["k"], "v": x["v"]}


def work(case):
    kind = case["kind"]
    if kind == "store":
        row = case["hkv"] * case["dim"] * 2
        return {"bytes": case["rows"] * (4 * row + 4), "flops": 0}
    if kind in ("model_step", "model_fill"):
        w, n, s = WIDTHS[case["width"]], case["batch"], case["prompt"]
        shapes = _parameter_shapes(case)
        embed = w["vocab_size"] * w["hidden_size"]
        total = sum(math.prod(v) for v in shapes.values())
        full = case["layers"] // 4
        linear = case["layers"] - full
        conv = 2 * w["linear_num_key_heads"] * w["linear_key_head_dim"] \
            + w["linear_num_value_heads"] * w["linear_value_head_dim"]
        cell = w["linear_num_value_heads"] * w["linear_key_head_dim"] * w["linear_value_head_dim"]
        kv = n * HKV * HEAD * 4
        new = s if kind == "model_fill" else 1
        rows = (n * new * w["hidden_size"] + n * w["vocab_size"]) * 2
        context = s + 1 + STEPS // 2                      # of an average decode step
        held = n * linear * (4 * cell + 2 * CONV * conv)
        moved = (total - embed) * 2 + rows + full * kv * new + held
        if kind == "model_step":
            moved += held + full * kv * (context - 1)
        scores = s * (s + 1) / 2 if kind == "model_fill" else context
        flops = 2 * n * (new * (total - 2 * embed) + embed) + full * n * 4 * HQ * HEAD * scores \
            + linear * n * new * 8 * cell
        return {"bytes": moved, "flops": flops}
    lens = _lengths(case)
    hq, hkv, dim = case["hq"], case["hkv"], case["dim"]
    if kind == "layer_fill":
        pre, new = case["prefix"], sum(lens)
        seen = case["batch"] * pre
        moved = new * (2 * hq + 4 * hkv) * dim * 2 + seen * hkv * dim * 4
        return {"bytes": moved + 4 * new,
                "flops": sum(4 * hq * dim * (n * pre + n * (n + 1) / 2) for n in lens)}
    moved = sum(lens) * hkv * dim * 4 + case["batch"] * hq * dim * 4 \
        + sum(-(-n // PAGE) * 4 + 4 for n in lens)
    if kind == "layer_step":
        moved += case["batch"] * (hkv * dim * 8 + 4)
    return {"bytes": moved, "flops": 4 * hq * dim * sum(lens)}


def tolerance(case):
    kind = case["kind"]
    if kind == "store":
        return "exact"
    if kind.startswith("model"):
        # bf16 activations: one rounding's change travels through every later layer
        return {"rel": 0.03, "max": 0.5}
    # bf16 outputs of float32 sums (matched also rounds its probabilities to bf16)
    return {"rel": 0.008, "max": 0.1}


def _exact_rows(q, keys, values, first, scale, block=256):
    """Causal attention of q [n, Hq, D] at positions first..first+n-1, 64 bits."""
    group = q.shape[1] // keys.shape[1]
    k = keys.double().repeat_interleave(group, 1).permute(1, 2, 0).contiguous()
    v = values.double().repeat_interleave(group, 1).transpose(0, 1).contiguous()
    out = torch.empty(q.shape, device=q.device, dtype=torch.float64)
    for a in range(0, q.shape[0], block):
        part = q[a:a + block].double().transpose(0, 1).contiguous()
        scores = torch.matmul(part, k) * scale
        at = first + a + torch.arange(part.shape[1], device=q.device)
        scores.masked_fill_(torch.arange(k.shape[2], device=q.device)[None, :] > at[:, None],
                            float("-inf"))
        out[a:a + block] = torch.matmul(scores.softmax(-1), v).transpose(0, 1)
    return out


def _rms(x, weight, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight


def _rope(x, positions):
    half = HEAD // 8                       # a quarter of the head rotates, in two halves
    inverse = (10000.0 ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half))
    angle = positions[:, None] * inverse.to(torch.bfloat16).double()
    a, b, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), rest],
                     -1)


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _exact_linear(x, weight, w):
    """Gated delta rule layer over x [B, S, hidden]: its output, conv and recurrent state."""
    n, s, _ = x.shape
    hk, dk = w["linear_num_key_heads"], w["linear_key_head_dim"]
    hv, dv = w["linear_num_value_heads"], w["linear_value_head_dim"]
    mixed = x @ weight("in_proj_qkv.weight").T
    gate = (x @ weight("in_proj_z.weight").T).view(n, s, hv, dv)
    beta = torch.sigmoid(x @ weight("in_proj_b.weight").T)[..., None]
    decay = torch.exp(-weight("A_log").exp() * F.softplus(
        x @ weight("in_proj_a.weight").T + weight("dt_bias")))[..., None, None]
    taps = weight("conv1d.weight")[:, 0]
    padded = F.pad(mixed, (0, 0, CONV - 1, 0))
    conv = F.silu(sum(padded[:, j:j + s] * taps[:, j] for j in range(CONV)))
    q, k, v = conv.split([hk * dk, hk * dk, hv * dv], -1)
    q = (_unit(q.reshape(n, s, hk, dk)) * dk ** -0.5).repeat_interleave(hv // hk, 2)
    k = _unit(k.reshape(n, s, hk, dk)).repeat_interleave(hv // hk, 2)
    v = v.reshape(n, s, hv, dv)
    state = torch.zeros((n, hv, dk, dv), device=x.device, dtype=torch.float64)
    out = torch.empty_like(v)
    for t in range(s):
        state = state * decay[:, t]
        change = (v[:, t] - torch.matmul(k[:, t].unsqueeze(-2), state).squeeze(-2)) * beta[:, t]
        state = state + k[:, t].unsqueeze(-1) * change.unsqueeze(-2)
        out[:, t] = torch.matmul(q[:, t].unsqueeze(-2), state).squeeze(-2)
    out = _rms(out, weight("norm.weight")) * F.silu(gate)
    held = F.pad(mixed, (0, 0, max(0, CONV - s), 0))[:, -CONV:].transpose(1, 2)
    return out.reshape(n, s, -1) @ weight("out_proj.weight").T, held, state


def _exact_full(x, weight):
    n, s, _ = x.shape
    both = (x @ weight("q_proj.weight").T).view(n, s, HQ, 2 * HEAD)
    q, gate = both[..., :HEAD], both[..., HEAD:]
    k = (x @ weight("k_proj.weight").T).view(n, s, HKV, HEAD)
    v = (x @ weight("v_proj.weight").T).view(n, s, HKV, HEAD)
    at = torch.arange(s, device=x.device, dtype=torch.float64)
    q = _rope(_rms(q, 1 + weight("q_norm.weight")).transpose(1, 2), at).transpose(1, 2)
    k = _rope(_rms(k, 1 + weight("k_norm.weight")).transpose(1, 2), at).transpose(1, 2)
    out = torch.stack([_exact_rows(q[b], k[b], v[b], 0, HEAD ** -0.5) for b in range(n)])
    return (out * torch.sigmoid(gate)).reshape(n, s, -1) @ weight("o_proj.weight").T


def _exact_model(case, seed):
    gen = _generator(seed)
    weights = {name: _draw_parameter(name, torch.empty(shape, device=DEV, dtype=torch.bfloat16),
                                     gen) for name, shape in _parameter_shapes(case).items()}
    prompt, fed = _model_tokens(case, seed)
    if case["kind"] == "model_step":
        prompt = np.concatenate([prompt, fed[:2].T], 1)
    x = weights["model.embed_tokens.weight"][torch.from_numpy(prompt).to(DEV)].double()
    states = []
    for i, kind in enumerate(_kinds(case["layers"])):
        weight = lambda name: weights[f"model.layers.{i}.{name}"].double()  # noqa: E731,B023
        h = _rms(x, 1 + weight("input_layernorm.weight"))
        if kind == "linear_attention":
            out, held, state = _exact_linear(h, lambda name: weight("linear_attn." + name),
                                             WIDTHS[case["width"]])
            states += [held, state]
        else:
            out = _exact_full(h, lambda name: weight("self_attn." + name))
        x = x + out
        h = _rms(x, 1 + weight("post_attention_layernorm.weight"))
        h = F.silu(h @ weight("mlp.gate_proj.weight").T) * (h @ weight("mlp.up_proj.weight").T)
        x = x + h @ weight("mlp.down_proj.weight").T
    last = _rms(x[:, -1], 1 + weights["model.norm.weight"].double())
    return {"logits": last @ weights["lm_head.weight"].double().T, "states": states, "pages": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "store":
        x = _store_inputs(case, seed)
        k, v = (x[n].double().view(-1, case["hkv"], case["dim"]) for n in ("k", "v"))
        k[x["slots"].long()], v[x["slots"].long()] = x["key"].double(), x["value"].double()
        return k.view(x["k"].shape), v.view(x["v"].shape)
    if kind.startswith("model"):
        return _exact_model(case, seed)
    x = _attention_inputs(case, seed)
    flat = {}
    for name, new in (("k", "key"), ("v", "value")):
        flat[name] = x[name].view(-1, case["hkv"], case["dim"])
        if kind.startswith("layer"):
            flat[name][_slots(x["tables"], x["starts"], x["lens"]).long()] = x[new]
    out, row = [], 0
    for table, start, n in zip(x["tables"], x["starts"], x["lens"]):
        at = _slots([table], [0], [n]).long()
        out.append(_exact_rows(x["q"][row:row + n - start], flat["k"][at], flat["v"][at], start,
                               case["dim"] ** -0.5))
        row += n - start
    out = torch.cat(out)
    if kind in ("matched", "paged"):
        return out
    return {"out": out.unsqueeze(1) if kind == "layer_step" else out, "k": x["k"].double(),
            "v": x["v"].double()}
