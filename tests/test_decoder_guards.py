"""Which models the decoder's kernels serve: plain ones, and none that was changed (CPU only)."""
import os
import subprocess
import sys
from types import SimpleNamespace

import pytest
import torch
from torch import nn
from transformers.activations import SiLUActivation
from transformers.models.qwen3_5 import modeling_qwen3_5 as qwen

from paged_decode import decoder_layers as DL
from paged_decode import hybrid as H

CPU = torch.device("cpu")


def build():
    cfg = H.decoder_config(num_hidden_layers=4, hidden_size=128, intermediate_size=128,
                           vocab_size=64, num_attention_heads=2, num_key_value_heads=1, head_dim=64,
                           linear_num_key_heads=1, linear_key_head_dim=64,
                           linear_num_value_heads=1, linear_value_head_dim=64)
    model = H.random_init_model(cfg, "cpu")
    model.config._attn_implementation = "paged_decode_lab_hip"
    model.model.config._attn_implementation = "paged_decode_lab_hip"
    return model


@pytest.fixture(scope="module")
def model():
    return build()


def served(model):
    return DL.decoder_weights(model, CPU) is not None


def other(*args, **kwargs):
    raise AssertionError("not called here")


@pytest.mark.parametrize("owner,name", [
    (qwen.Qwen3_5MLP, "forward"), (qwen.Qwen3_5Attention, "forward"),
    (qwen.Qwen3_5DecoderLayer, "forward"), (qwen.Qwen3_5DecoderLayer, "__call__"),
    (qwen.Qwen3_5GatedDeltaNet, "forward"), (qwen.Qwen3_5RMSNorm, "forward"),
    (qwen.Qwen3_5RMSNorm, "_norm"), (qwen.Qwen3_5RMSNormGated, "forward"),
    (qwen.Qwen3_5TextRotaryEmbedding, "forward"), (SiLUActivation, "forward"),
    (nn.Linear, "forward"), (nn.Linear, "__call__"), (nn.Conv1d, "_conv_forward"),
    (nn.Module, "_call_impl"), (qwen, "apply_rotary_pos_emb"), (qwen, "l2norm"),
    (qwen, "torch_recurrent_gated_delta_rule"), (qwen, "Qwen3_5MLP")])
def test_patched_classes_and_functions_keep_the_modules(model, monkeypatch, owner, name):
    assert served(model)
    with monkeypatch.context() as patch:
        patch.setattr(owner, name, other, raising=False)
        assert not served(model)
    assert served(model)


def test_a_class_of_another_file_keeps_the_modules(monkeypatch):
    class Qwen3_5MLP(qwen.Qwen3_5MLP):
        def forward(self, x):
            return 2 * super().forward(x)

    with monkeypatch.context() as patch:
        patch.setattr(qwen, "Qwen3_5MLP", Qwen3_5MLP)
        changed = build()
        assert not served(changed)
    assert not served(changed)


BEFORE_IMPORT = """
from transformers.models.qwen3_5 import modeling_qwen3_5 as qwen
plain = qwen.{name}
def patched(*args):
    return plain(*args)
qwen.{name} = patched
from paged_decode import decoder_layers as DL
assert not DL._as_installed()
"""


@pytest.mark.parametrize("name", ["Qwen3_5MLP.forward", "apply_rotary_pos_emb"])
def test_patches_made_before_the_import_are_seen(name):
    assert DL._as_installed()
    env = dict(os.environ, PYTHONPATH=os.pathsep.join(sys.path))
    code = BEFORE_IMPORT.format(name=name)
    if "." not in name:   # a function of the file: only its code's file tells
        code = code.replace("qwen." + name + " = patched",
                            "patched.__module__ = qwen.__name__; qwen." + name + " = patched")
    subprocess.run([sys.executable, "-c", code], check=True, env=env, timeout=300)


@pytest.mark.parametrize("change", ["hook", "pre_hook", "forward", "_norm", "bias", "train", "dtype"])
def test_changed_instances_keep_the_modules(change):
    model = build()
    assert served(model)
    layer = model.model.layers[0]
    if change == "hook":
        layer.mlp.register_forward_hook(lambda *a: None)
    elif change == "pre_hook":
        layer.linear_attn.register_forward_pre_hook(lambda *a: None)
    elif change == "forward":
        layer.mlp.forward = other
    elif change == "_norm":
        layer.input_layernorm._norm = other
    elif change == "bias":
        layer.mlp.up_proj.bias = nn.Parameter(torch.zeros(128, dtype=torch.bfloat16))
    elif change == "train":
        layer.mlp.train()
    else:
        layer.mlp.float()
    assert not served(model)


@pytest.mark.parametrize("batch,steps,runs", [(1, 65535 * 16, True), (1, 65535 * 16 + 1, False),
                                              (65536, 1, False), (2, 0, False)])
def test_token_counts_past_the_grids_keep_the_modules(batch, steps, runs):
    runner = SimpleNamespace(batch=batch, device=CPU, cache=SimpleNamespace(linear={}))
    tokens = torch.zeros(1, 1, dtype=torch.long).expand(batch, steps)
    assert (DL.decoder_states(runner, None, tokens) is not None) == runs
    other_batch = SimpleNamespace(**{**vars(runner), "batch": batch + 1})
    assert DL.decoder_states(other_batch, None, tokens) is None
