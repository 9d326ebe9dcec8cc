"""The balanced prefill launch over requests far shorter than their page table is wide: its grid follows
the table, its shares the lengths, so there are fewer KV steps than workgroup gangs."""
import pytest
import torch

from src.kernels.hip_paged_attention import paged_attention_prefill_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Hd", [64, 128])
@pytest.mark.parametrize("lens", [[1], [40], [240], [5, 1200], [0, 700, 33]], ids=str)
def test_fewer_steps_than_gangs(device, monkeypatch, dtype, Hd, lens):
    B, H, T = len(lens), 8, 40
    g = torch.Generator().manual_seed(sum(lens) + Hd)
    blocks = B * 1024
    k, v = (torch.randn(128 * B, H, 16, Hd, generator=g).to(dtype).to(device) for _ in range(2))
    table = (torch.arange(blocks).view(B, 1024) % (128 * B)).to(torch.int32).to(device)
    seq = torch.tensor(lens, dtype=torch.int32, device=device)
    cur = torch.tensor([min(n, T) for n in lens], dtype=torch.int32, device=device)
    print(f"balanced launch, short requests {lens} {dtype} head_dim {Hd}", flush=True)
    monkeypatch.setenv("PAGED_HIP_PREFILL_KERNEL", "wide")
    for _ in range(3):  # (other inputs each time: a call that leaves its arrival counters behind spoils the next)
        q = torch.randn(B, H, T, Hd, generator=g).to(device)
        monkeypatch.setenv("PAGED_HIP_PREFILL_BALANCE", "off")
        want = paged_attention_prefill_hip(q, k, v, table, seq, cur)
        monkeypatch.setenv("PAGED_HIP_PREFILL_BALANCE", "force")
        got = paged_attention_prefill_hip(q, k, v, table, seq, cur, out=torch.full_like(q, 7.0))
        # the same products in another order of the steps; bf16 KV rounds the softmax weights to bf16
        # at another running maximum
        assert float((got - want).abs().max()) < (2e-6 if dtype == torch.float32 else 3e-2)
