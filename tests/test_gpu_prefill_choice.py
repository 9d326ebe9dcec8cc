"""The kernel that a prefill call takes by its sizes: on every side of the lines between the kernels, the
default call against the 16-row kernel, which serves all of them."""
import pytest
import torch

from src.kernels.hip_paged_attention import PREFILL_BALANCED, paged_attention_prefill_hip, prefill_workspace_size

pytestmark = pytest.mark.gpu

def test_balanced_calls_on_two_streams_and_in_graphs(device, monkeypatch):
    """Calls on other streams and captured calls have workspaces of their own."""
    monkeypatch.setenv("PAGED_HIP_PREFILL_BALANCE", "force")
    cases = []
    for seed, lens in ((1, [3000, 200]), (2, [1500, 2500, 900])):
        g = torch.Generator(device=device).manual_seed(seed)
        k, v = (torch.randn(600, 8, 16, 64, generator=g, device=device) for _ in range(2))
        q = torch.randn(len(lens), 8, 200, 64, generator=g, device=device)
        table = torch.randint(0, 600, (len(lens), 188), generator=g, device=device, dtype=torch.int32)
        cases.append((q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=device),
                      torch.full((len(lens),), 200, dtype=torch.int32, device=device)))
    for q, k, _, table, _, _ in cases:  # (the balanced launch is the one that runs)
        assert prefill_workspace_size(*q.shape, table.shape[1], PREFILL_BALANCED, k.dtype) > 0
    want = [paged_attention_prefill_hip(*c).clone() for c in cases]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(8):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(paged_attention_prefill_hip(*cases[i]))
    torch.cuda.synchronize()
    assert all(torch.equal(x, want[i]) for i in range(2) for x in got[i])
    out = torch.empty_like(want[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        paged_attention_prefill_hip(*cases[0], out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        other = paged_attention_prefill_hip(*cases[1])
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]) and torch.equal(other, want[1])


SHAPES = [  # requests, heads, head_dim, chunk, longest context
    (8, 32, 128, 16, 400), (8, 32, 128, 100, 1500), (2, 32, 128, 257, 1500), (1, 32, 128, 512, 8192),
    (16, 32, 128, 128, 200), (3, 12, 128, 129, 900), (64, 8, 64, 16, 400), (64, 8, 64, 1, 300), (8, 8, 64, 512, 2000),
    (4, 8, 64, 61, 5000), (1, 8, 64, 128, 9000), (32, 8, 64, 64, 1500), (16, 8, 64, 100, 6000), (5, 3, 64, 33, 70),
    (300, 8, 64, 17, 40), (2, 8, 64, 128, 0)]


@pytest.mark.parametrize("io,kv", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                   (torch.bfloat16, torch.bfloat16)], ids=["fp32", "bf16kv", "bf16"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_default_call_against_the_16_row_kernel(device, monkeypatch, shape, io, kv):
    B, H, Hd, T, hi = shape
    print(f"prefill choice {shape} {io} {kv}", flush=True)
    g = torch.Generator(device=device).manual_seed(T + hi)
    ctx = [hi * (b + 1) // B // (1 if b % 2 else 3) for b in range(B)]
    cur = [T if b % 3 else max(1, T - 7) for b in range(B)]
    lens = [c + n for c, n in zip(ctx, cur)]
    pages = -(-max(lens) // 16)
    N = min(B * pages, 4096)
    k, v = (torch.randn(N, H, 16, Hd, generator=g, device=device).to(kv) for _ in range(2))
    q = torch.randn(B, T, H, Hd, generator=g, device=device).to(io).transpose(1, 2)
    table = torch.randint(0, N, (B, pages), generator=g, device=device, dtype=torch.int32)
    args = (q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=device),
            torch.tensor(cur, dtype=torch.int32, device=device))
    for name in ("KERNEL", "BALANCE"):
        monkeypatch.delenv("PAGED_HIP_PREFILL_" + name, raising=False)
    got = paged_attention_prefill_hip(*args).float()
    monkeypatch.setenv("PAGED_HIP_PREFILL_KERNEL", "tile")
    want = paged_attention_prefill_hip(*args, split_blocks=0).float()
    # fp32: sums of up to 9128 keys in another order. bf16 KV: the softmax weights are rounded to bf16 at
    # another running maximum, 2^-9 each, and bf16 outputs once more
    assert float((got - want).abs().max()) < (2e-5 if kv == torch.float32 else 3e-2)
