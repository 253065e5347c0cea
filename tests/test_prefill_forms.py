"""The PyTorch forms of the prefill attention, on the CPU."""
import numpy as np
import pytest
import torch

from paged_decode import prefill as PF
from paged_decode.engine_attention import Attention, reset_context, set_context


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,hq,hkv,s", [(1, 4, 2, 5), (2, 4, 4, 1), (3, 6, 2, 7)])
def test_batched_rows_are_contiguous(b, hq, hkv, s, dtype):
    """Callers read the result [B, S, Hq, D] by its address."""
    gen = torch.Generator().manual_seed(s)
    rows = lambda h: torch.randn((b, s, h, 64), generator=gen).to(dtype).transpose(1, 2)  # noqa: E731
    out = PF.batched_prefill(rows(hq), rows(hkv), rows(hkv), 0.125)
    assert out.shape == (b, s, hq, 64) and out.dtype == dtype and out.is_contiguous()


@pytest.mark.parametrize("hint", [None, 0, -1, 3000.0, torch.tensor(3000)])
def test_an_unknown_longest_sequence_is_one_span(monkeypatch, hint):
    monkeypatch.setattr(PF, "device_cus", lambda device: 256)
    assert PF._splits(1, hint, 128, "cuda") == 1
    assert PF._splits(1, np.int64(3000), 128, "cuda") == PF._splits(1, 3000, 128, "cuda") > 1


@pytest.mark.parametrize("heads,q_heads,k_heads", [((8, 2), 16, 2), ((8, 2), 8, 4), ((8, 2), 4, 2),
                                                   ((4, 4), 8, 2), ((8, 2), 2, 1)])
def test_other_head_counts_than_the_layers_fail(heads, q_heads, k_heads):
    layer = Attention(heads[0], 64, 0.125, heads[1])
    cu = torch.tensor([0, 5], dtype=torch.int32)
    set_context(True, cu, cu, 5, 5)
    try:
        with pytest.raises(RuntimeError):
            layer(torch.zeros(5, q_heads, 64), torch.zeros(5, k_heads, 64), torch.zeros(5, k_heads, 64))
        out = layer(torch.zeros(5, heads[0], 64), *[torch.zeros(5, heads[1], 64)] * 2)
        assert out.shape == (5, heads[0], 64)
    finally:
        reset_context()
