"""Which workspace a split call takes: one per stream and per capture, so that calls that may run at the same
time never share arrival counters or records."""
import pytest
import torch

from src.kernels import hip_paged_attention as hpa


@pytest.fixture
def streams(monkeypatch):
    """The wrapper's view of the current stream and capture, set by the test; empty workspace tables."""
    now = {"stream": 0, "capture": 0}
    monkeypatch.setattr(hpa, "_stream_ptr", lambda device: now["stream"])
    monkeypatch.setattr(hpa, "_capture_id", lambda stream: now["capture"])
    monkeypatch.setattr(hpa, "_workspaces", {})
    monkeypatch.setattr(hpa, "_stream_workspaces", {})

    def take(stream, capture=0, nbytes=1000, kind="decode"):
        now.update(stream=stream, capture=capture)
        return hpa._call_workspace(torch.device("cpu", 0), nbytes, kind)

    return take


def test_one_workspace_per_stream_and_capture(streams):
    default, a, b = streams(0), streams(7), streams(8)
    assert len({t.data_ptr() for t in (default, a, b)}) == 3
    assert streams(0) is default and streams(7) is a and streams(8) is b
    first = streams(7, capture=1)
    assert first is not a and streams(7, capture=1) is first  # the calls of one capture follow each other
    assert streams(7, capture=2) is not first
    assert streams(7) is not first


def test_larger_calls_and_the_bound(streams):
    a = streams(7)
    assert a.numel() >= 1 << 20 and streams(7, nbytes=a.numel()) is a
    b = streams(7, nbytes=a.numel() + 1)
    assert b.numel() == a.numel() + 1 and streams(7) is b
    for s in range(100, 100 + hpa.MAX_STREAM_WORKSPACES - 1):
        streams(s)
    assert streams(7) is b  # (used last from here on)
    streams(200)
    assert len(hpa._stream_workspaces) == hpa.MAX_STREAM_WORKSPACES
    assert (0, 100, "decode") not in hpa._stream_workspaces and streams(7) is b


@pytest.mark.parametrize("kind", ["decode", "prefill"])
def test_counters_start_at_zero(streams, kind):
    junk = torch.full((1 << 20,), 7, dtype=torch.uint8)  # (whatever memory the allocator hands out next)
    del junk
    for stream in (0, 7):
        assert int(torch.count_nonzero(streams(stream, kind=kind)[:hpa.COUNTER_BYTES[kind]])) == 0


def _batch(device, seed, lens, H=8, Hd=64):
    g = torch.Generator(device=device).manual_seed(seed)
    pages = -(-max(lens) // 16)
    k, v = (torch.randn(len(lens) * pages, H, 16, Hd, generator=g, device=device) for _ in range(2))
    q = torch.randn(len(lens), H, 1, Hd, generator=g, device=device)
    table = torch.randperm(len(lens) * pages, generator=g, device=device).view(-1, pages).to(torch.int32)
    return (q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=device),
            torch.ones(len(lens), dtype=torch.int32, device=device))


@pytest.mark.gpu
@pytest.mark.parametrize("split", [16, 4], ids=["merged in the launch", "merged by a second launch"])
def test_split_decode_on_two_streams_and_in_two_graphs(device, split):
    """Split calls on two streams at once, and two graphs replayed on two streams with eager calls beside
    them, give what they give alone."""
    cases = [_batch(device, 1, [900, 30, 700, 1000]), _batch(device, 2, [64, 1020, 500])]
    call = lambda c, **kw: hpa.paged_attention_decode_hip(*c, split_blocks=split, **kw)  # noqa: E731
    want = [call(c).clone() for c in cases]
    for w, c in zip(want, cases):
        plain = hpa.paged_attention_decode_hip(*c, split_blocks=0)
        assert float((w - plain).abs().max()) < 4e-6  # (fp32 sums in another order, values of N(0, 1) averaged)
    side = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for i, st in enumerate(side):
            with torch.cuda.stream(st):
                got[i].append(call(cases[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(x, want[i]) for x in got[i])
    outs, graphs = [[torch.empty_like(w) for _ in range(3)] for w in want], []
    for c, o in zip(cases, outs):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for x in o:
                call(c, out=x)
        graphs.append(graph)
    for _ in range(4):
        for o in outs:
            for x in o:
                x.fill_(float("nan"))
        torch.cuda.synchronize()
        for st, graph in zip(side, graphs):
            with torch.cuda.stream(st):
                graph.replay()
        eager = [call(c) for c in cases]
        torch.cuda.synchronize()
        for i in range(2):
            assert torch.equal(eager[i], want[i]) and all(torch.equal(x, want[i]) for x in outs[i])


@pytest.mark.gpu
def test_captures_are_told_apart(device):
    """The capture identifier: 0 outside, one per capture, the same for every stream of it."""
    seen, x = [], torch.zeros(4, device=device)
    st, other = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(2):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(st):
            assert hpa._capture_id(st.cuda_stream) == 0
            graph.capture_begin()
            here = hpa._capture_id(st.cuda_stream)
            other.wait_stream(st)
            there = hpa._capture_id(other.cuda_stream)
            x.add_(1)
            st.wait_stream(other)
            graph.capture_end()
        assert here == there != 0
        seen.append(here)
    assert seen[0] != seen[1] and hpa._capture_id(st.cuda_stream) == 0


@pytest.mark.gpu
def test_captured_steps_have_their_own_workspaces(device, monkeypatch):
    """One per graph, zeroed before the capture: no step takes the stream's or clears counters as it runs."""
    import numpy as np

    from src.cache.paged_kv import BatchedPagedKVCache
    from src.model.transformer import TinyTransformerLM

    def taken(*args):
        raise AssertionError("a captured step took a stream's workspace")

    torch.manual_seed(0)
    model = TinyTransformerLM(64, 512, 8, 2, 512, 1024).to(device).eval()
    B = 2
    requests = model.create_request_kv_caches(B)
    caches = [BatchedPagedKVCache([requests[r][layer] for r in range(B)], model.layer_block_pools[layer])
              for layer in range(2)]
    ids = np.arange(B * 40).reshape(B, 40) % 64
    step = lambda n, at: model.greedy_step(ids[:, :n].copy(), caches, position_offset=[at] * B,  # noqa: E731
                                           current_lengths=[n] * B, return_logits=True)
    step(40, 0)  # (eager: the pools are allocated)
    monkeypatch.setattr(hpa, "_call_workspace", taken)
    monkeypatch.setenv("PAGED_HIP_PREFILL_BALANCE", "force")
    step(40, 40)
    for t in range(3):
        step(1, 80 + t)
    torch.cuda.synchronize()
    caps = list(model._graph_step.captured.values())
    assert sorted(c.Tb for c in caps) == [1, 64]
    for c in caps:
        kind = "decode" if c.Tb == 1 else "prefill"
        assert int(torch.count_nonzero(c.ws[:hpa.COUNTER_BYTES[kind]])) == 0
    assert len({c.ws.data_ptr() for c in caps}) == 2


@pytest.mark.gpu
def test_prefill_workspace_by_kv_dtype(device):
    """Where a call over fp32 KV would be balanced and one over bf16 KV is not, the latter takes none."""
    from src.kernels import _lib

    lib = _lib.load()
    found = 0
    for B, H, T, Hd, pages in ((4, 8, 128, 64, 512), (1, 8, 128, 64, 2048), (8, 32, 128, 128, 400), (4, 8, 64, 64, 64)):
        sizes = [hpa.prefill_workspace_size(B, H, T, Hd, pages, hpa.PREFILL_BALANCED, dt)
                 for dt in (torch.float32, torch.bfloat16)]
        assert lib.pa_prefill_workspace_size(B, H, T, Hd, pages, hpa.PREFILL_BALANCED) == max(sizes)
        if sizes[0] == 0 or sizes[1] > 0:
            continue
        found += 1
        g = torch.Generator(device=device).manual_seed(T)
        k, v = (torch.randn(64, H, 16, Hd, generator=g, device=device).bfloat16() for _ in range(2))
        q = torch.randn(B, H, T, Hd, generator=g, device=device)
        table = torch.randint(0, 64, (B, pages), generator=g, device=device, dtype=torch.int32)
        lens = torch.full((B,), 300, dtype=torch.int32, device=device)
        cur = torch.full((B,), T, dtype=torch.int32, device=device)
        want = hpa.paged_attention_prefill_hip(q, k, v, table, lens, cur, split_blocks=0)
        st = torch.cuda.Stream()
        hpa._stream_workspaces.clear()
        torch.cuda.synchronize()
        with torch.cuda.stream(st):
            got = hpa.paged_attention_prefill_hip(q, k, v, table, lens, cur)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and not hpa._stream_workspaces
    assert found
