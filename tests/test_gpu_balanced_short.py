"""The balanced prefill launch over requests far shorter than their page table is wide: its grid follows
the table, its shares the lengths, so there are fewer KV steps than workgroup gangs."""
import pytest
import torch

from src.kernels.hip_paged_attention import PREFILL_BALANCED, paged_attention_prefill_hip, prefill_workspace_size

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
        assert prefill_workspace_size(B, H, T, Hd, 1024, PREFILL_BALANCED, dtype) > 0  # (it is the one that runs)
        got = paged_attention_prefill_hip(q, k, v, table, seq, cur, out=torch.full_like(q, 7.0))
        # the same products in another order of the steps; bf16 KV rounds the softmax weights to bf16
        # at another running maximum
        assert float((got - want).abs().max()) < (2e-6 if dtype == torch.float32 else 3e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Hd", [64, 128])
def test_infinite_values_through_a_merge(device, monkeypatch, dtype, Hd):
    """An infinity in V's last keys: what the finishing workgroup holds of a cut tile is merged once, as its
    record, so rows that see the key come out infinite as in the uncut launch."""
    T, n = 130, 4000
    g = torch.Generator().manual_seed(Hd)
    k, v = (torch.randn(250, 8, 16, Hd, generator=g).to(dtype) for _ in range(2))
    table = torch.randperm(250, generator=g).view(1, 250).to(torch.int32)
    at = [3, 1000, 2500, 3860]  # (keys that every row of the chunk sees)
    for h, key in enumerate(at):
        v[table[0, key // 16], h, key % 16, h] = float("inf") if h % 2 else float("-inf")
    q = torch.randn(1, 8, T, Hd, generator=g).to(device)
    args = (q, k.to(device), v.to(device), table.to(device), torch.tensor([n], dtype=torch.int32, device=device),
            torch.tensor([T], dtype=torch.int32, device=device))
    monkeypatch.setenv("PAGED_HIP_PREFILL_KERNEL", "wide")
    monkeypatch.setenv("PAGED_HIP_PREFILL_BALANCE", "force")
    assert prefill_workspace_size(1, 8, T, Hd, 250, PREFILL_BALANCED, dtype) > 0
    for _ in range(4):  # (any workgroup may be the last)
        got = paged_attention_prefill_hip(*args)
        for h in range(4):
            assert bool((got[0, h, :, h] == (float("inf") if h % 2 else float("-inf"))).all()), h
            got[0, h, :, h] = 0
        assert bool(got.isfinite().all())
