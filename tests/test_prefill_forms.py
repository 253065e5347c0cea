"""The PyTorch forms of the prefill attention, on the CPU."""
import numpy as np
import pytest
import torch

from paged_decode import prefill as PF


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
