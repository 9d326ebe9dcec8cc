"""Which layers of a captured step run through the fused kernels: fc1's row limit follows the model's width."""
from types import SimpleNamespace

import pytest
import torch

from src.model import graph_decode
from src.model.transformer import TinyTransformerLM


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d_model,rows,fused", [
    (256, 1024, True), (512, 1024, True), (1024, 1024, False), (1024, 800, False), (1024, 512, True)])
@torch.no_grad()
def test_fc1_of_wide_models_over_many_rows_runs_through_torch(monkeypatch, dtype, d_model, rows, fused):
    model = TinyTransformerLM(16, d_model, 4, 1, 128, 64).to(dtype).eval()
    gelu_calls = []

    def linear(x, layer, *, gelu=False, **kw):
        gelu_calls.append(gelu)
        return torch.zeros(x.shape[0], layer.out_features, dtype=dtype)

    monkeypatch.setattr(graph_decode.hip_linear, "linear_rows_hip", linear)
    monkeypatch.setattr(graph_decode.hip_linear, "qkv_append_hip", lambda x, *a: torch.zeros_like(x))
    for name in ("paged_attention_prefill_hip", "prefill_in_workspace"):
        if hasattr(graph_decode, name):
            monkeypatch.setattr(graph_decode, name, lambda *a, **kw: torch.zeros(4, 4, rows // 4, d_model // 4, dtype=dtype))
    monkeypatch.setattr(graph_decode, "_pool_tensors", lambda pool: (None, None))
    step = graph_decode.GraphedStep(model)
    cap = SimpleNamespace(B=4, Tb=rows // 4, folded=False, cur=None, split_blocks=0, ws=None)
    step._fused_layers(cap, [None], torch.zeros(rows, d_model, dtype=dtype), None, None, None)
    assert (True in gelu_calls) == fused
