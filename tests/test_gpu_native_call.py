"""The native front of the entry points against the Python wrappers behind it: the same outputs bit for bit,
and None (so that the wrapper runs, and raises what it always raised) for every form it does not take."""
import pytest
import torch
import torch.nn as nn

from src.kernels import hip_linear, hip_paged_attention as hpa


def _attention(device, T, dtype=torch.float32, B=3, H=8, Hd=64):
    g = torch.Generator().manual_seed(T)
    q = torch.randn(B, T, H, Hd, generator=g).to(dtype).to(device).transpose(1, 2)
    k, v = (torch.randn(64, H, 16, Hd, generator=g).to(dtype).to(device) for _ in range(2))
    table = torch.randperm(64, generator=g)[: B * 20].view(B, 20).to(torch.int32).to(device)
    lens = torch.tensor([300, 90, 17], dtype=torch.int32, device=device)
    return q, k, v, table, lens, torch.full((B,), T, dtype=torch.int32, device=device)


def test_leaves_cpu_tensors_and_odd_arguments_to_the_wrapper():
    if hpa._call is None:
        pytest.skip("not built")
    c = hpa._call
    d, p = _attention("cpu", 1), _attention("cpu", 16)
    assert c.decode(*d, None, None, None) is None and c.prefill(*p, -1, None) is None
    assert c.decode() is None and c.decode(*[None] * 9) is None and c.prefill(*[1] * 8) is None
    assert c.kv_append(d[0], d[0], d[1], d[2], d[4]) is None
    x, w = torch.zeros(4, 128), torch.zeros(8, 128)
    assert c.linear_rows(x, w, None, None, None, 0.0, False, None, None, None) is None
    assert c.qkv_append(x, None, None, 0.0, *[w] * 6, d[1], d[2], d[4], None) is None
    with pytest.raises(ValueError):
        hpa.paged_attention_decode_hip(*d)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_same_results_as_the_wrappers(device, monkeypatch, dtype):
    D = 512
    g = torch.Generator().manual_seed(1)
    x = torch.randn(20, D, generator=g).to(dtype).to(device)
    lin = [nn.Linear(D, D).to(dtype).to(device) for _ in range(3)]
    ln = nn.LayerNorm(D).to(dtype).to(device)
    attn = type("A", (), dict(zip(("q_proj", "k_proj", "v_proj"), lin)))()
    dec, pre = _attention(device, 1, dtype), _attention(device, 16, dtype)
    slots = torch.arange(48, dtype=torch.int32, device=device)

    def everything():
        pools = [torch.zeros_like(pre[1]) for _ in range(4)]
        hpa.kv_append_hip(pre[0], pre[0], pools[0], pools[1], slots)
        order = torch.tensor([2, 0, 1], dtype=torch.int32, device=device)
        out = torch.empty_like(dec[0])
        with torch.no_grad():
            return [*pools[:2], hpa.paged_attention_decode_hip(*dec),
                    hpa.paged_attention_decode_hip(*dec, order=order, split_blocks=4, out=out), out,
                    hpa.paged_attention_decode_hip(dec[0].contiguous(), *dec[1:], split_blocks=0),
                    hpa.paged_attention_prefill_hip(*pre), hpa.paged_attention_prefill_hip(*pre, split_blocks=0),
                    hip_linear.linear_rows_hip(x, lin[0], ln=ln, gelu=True, residual=x),
                    hip_linear.qkv_append_hip(x, ln, attn, pools[2], pools[3], slots), *pools[2:]]

    served = []
    real = hpa.native_call()
    assert real is not None

    class Spy:
        def __getattr__(self, name):
            def call(*args):
                r = getattr(real, name)(*args)
                served.append((name, r is not None))
                return r
            return call

    everything()  # (workspaces exist from here on)
    monkeypatch.setattr(hpa, "_call", Spy())
    got = everything()
    assert len(served) == 8 and all(ok for _, ok in served), served
    monkeypatch.setattr(hpa, "_call", None)
    monkeypatch.setattr(hpa, "_call_bound", False)
    want = everything()
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.gpu
def test_forms_left_to_the_wrapper(device):
    q, k, v, table, lens, cur = _attention(device, 1)
    c = hpa.native_call()
    none = (None, None, None)
    assert c.decode(q, k, v, table, lens, cur, None, 0, None) is not None
    for args in ((q.double(), k, v, table, lens, cur), (q, k.half(), v.half(), table, lens, cur),
                 (q, k[:, :4], v[:, :4], table, lens, cur), (q, k, v, table.long(), lens, cur),
                 (q, k, v, table.t(), lens, cur), (q, k, v, table, lens.cpu(), cur), (q[:0], k, v, table[:0], lens, cur),
                 (q.transpose(1, 3).contiguous().transpose(1, 3), k, v, table, lens, cur),
                 (q, k.transpose(0, 1), v.transpose(0, 1), table, lens, cur)):
        assert c.decode(*args, *none) is None
    assert c.decode(q, k, v, table, lens, cur, None, 0, q.bfloat16()) is None
    with pytest.raises(ValueError):
        hpa.paged_attention_decode_hip(q, k, v, table.long(), lens, cur)
    with pytest.raises(RuntimeError):  # no data pointer under vmap: refused as by the wrapper
        torch.vmap(lambda y: hpa.paged_attention_decode_hip(y, k, v, table, lens, cur))(q[None])


def _refused(call, *args, **kw):
    with pytest.raises(ValueError):
        call(*args, **kw)


@pytest.mark.gpu
def test_attention_operands_that_a_kernel_cannot_read(device):
    """Host memory and arrays shorter than the batch are refused before any launch, by either front."""
    for T, call in ((1, hpa.paged_attention_decode_hip), (16, hpa.paged_attention_prefill_hip)):
        q, k, v, table, lens, cur = _attention(device, T)
        want = call(q, k, v, table, lens, cur)
        for bad in ((table[:2], lens, cur), (table, lens[:2], cur), (table, lens, cur[:2]), (table, lens, cur.cpu())):
            _refused(call, q, k, v, *bad)
        assert torch.equal(call(q, k, v, torch.cat([table, table]), torch.cat([lens, lens]), torch.cat([cur, cur])), want)
    q, k, v, table, lens, cur = _attention(device, 1)
    want = hpa.paged_attention_decode_hip(q, k, v, table, lens, cur)
    order = torch.tensor([2, 0, 1], dtype=torch.int32)
    for bad in (order, order[:2].to(device), order.long().to(device)):
        _refused(hpa.paged_attention_decode_hip, q, k, v, table, lens, cur, order=bad)
    for good in (order.to(device), order.pin_memory()):  # (kernels read pinned host memory in place)
        assert torch.equal(hpa.paged_attention_decode_hip(q, k, v, table, lens, cur, order=good), want)
    _refused(hpa.kv_append_hip, q, q, k, v, order)


@pytest.mark.gpu
@torch.no_grad()
def test_layer_operands_that_a_kernel_cannot_reach(device):
    M, K, N = 5, 128, 64
    x = torch.randn(M, K, device=device)
    lin, ln = nn.Linear(K, N).to(device), nn.LayerNorm(K).to(device)
    rows = lambda m, n: torch.zeros(m, n, device=device)  # noqa: E731
    call = hip_linear.linear_rows_hip
    want = call(x, lin, ln=ln)
    for name in ("out", "residual", "copy_to"):
        for bad in (rows(M - 1, N), rows(M, N - 1), torch.zeros(M, N)):
            _refused(call, x, lin, ln=ln, **{name: bad})
    assert torch.equal(call(x, lin, ln=ln, out=rows(M + 1, N + 4))[:M, :N], want)
    _refused(call, x, nn.Linear(K, N))
    _refused(call, x, lin, ln=nn.LayerNorm(K))
    _refused(call, x, lin, ln=nn.LayerNorm(K // 2).to(device))
    strided = nn.Linear(K, N).to(device)
    strided.weight = nn.Parameter(torch.randn(K, N, device=device).t())
    _refused(call, x, strided)
    short = nn.Linear(K, N).to(device)
    short.bias = nn.Parameter(torch.zeros(N - 1, device=device))
    _refused(call, x, short)
    index = torch.zeros(1, dtype=torch.int32, device=device)
    _refused(hip_linear.linear_select_rows_hip, x, M, index, nn.Linear(K, N))

    layers = {n: nn.Linear(K, K).to(device) for n in ("q_proj", "k_proj", "v_proj")}
    attn = lambda **kw: type("A", (), {**layers, **kw})()  # noqa: E731
    pools = [torch.zeros(4, 2, 16, 64, device=device) for _ in range(2)]
    slots = torch.arange(M, dtype=torch.int32)
    qkv = hip_linear.qkv_append_hip
    qkv(x, ln, attn(), *pools, slots.to(device))
    _refused(qkv, x, ln, attn(), *pools, slots)
    _refused(qkv, x, ln, attn(), *pools, slots[: M - 1].to(device))
    _refused(qkv, x, ln, attn(), *pools, slots.to(device), out=rows(M - 1, K))
    _refused(qkv, x, ln, attn(k_proj=nn.Linear(K, K)), *pools, slots.to(device))
    _refused(qkv, x, ln, attn(v_proj=nn.Linear(K, K // 2).to(device)), *pools, slots.to(device))
    _refused(qkv, x, ln, attn(), *(p.cpu() for p in pools), slots.to(device))

    fc1, fc2 = nn.Linear(K, N).to(device), nn.Linear(N, K).to(device)
    _refused(hip_linear.mlp_rows_hip, x, ln, fc1, nn.Linear(N, K), rows(M, K))
    _refused(hip_linear.mlp_rows_hip, x, ln, fc1, fc2, rows(M, K), residual=rows(M - 1, K))
    ids, pos = torch.zeros(2, 3, dtype=torch.int64), torch.zeros(2, dtype=torch.int64)
    table = nn.Embedding(8, K).to(device)
    _refused(hip_linear.embed_rows_hip, ids.to(device), pos, table, table)
    _refused(hip_linear.embed_rows_hip, ids.to(device), pos.to(device), nn.Embedding(8, K), table)
    _refused(hip_linear.embed_rows_hip, ids.to(device), pos.to(device), table, table, out=rows(5, K))
