"""The balanced decode launch (split_blocks = DECODE_BALANCED): workgroup gangs share all requests' KV
blocks evenly, cutting requests anywhere. Against the unsplit launch and the oracle."""
import math

import pytest
import torch

import oracle
from src.kernels import _lib
from src.kernels.hip_paged_attention import DECODE_BALANCED, default_split_blocks, paged_attention_decode_hip

pytestmark = pytest.mark.gpu


def _batch(device, lens, H, Hd, io, kv, seed=0, extra_pages=3):
    g = torch.Generator().manual_seed(seed)
    counts = [-(-n // 16) for n in lens]
    N = sum(counts) + 5
    perm = torch.randperm(N, generator=g).to(torch.int32)
    table = torch.full((len(lens), max(counts) + extra_pages), -1, dtype=torch.int32)
    lists, at = [], 0
    for b, c in enumerate(counts):
        lists.append(perm[at:at + c].tolist())
        table[b, :c] = perm[at:at + c]
        at += c
    q = torch.randn(len(lens), 1, H, Hd, generator=g).to(io).transpose(1, 2)
    k, v = (torch.randn(N, H, 16, Hd, generator=g).to(kv) for _ in range(2))
    seq = torch.tensor(lens, dtype=torch.int32)
    return (q, k, v, table, seq, torch.ones_like(seq)), lists


LENS = [[512] * 40, [513] + [512] * 39, [300, 5] * 100, [1], [4000], [0, 0, 0], [0, 5, 0, 300, 16, 17], [16] * 70, [2000, 1, 1, 1, 900], list(range(1, 513)),
        [333] * 31 + [7000]]


@pytest.mark.parametrize("io,kv", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                   (torch.bfloat16, torch.bfloat16)], ids=["fp32", "bf16kv", "bf16"])
@pytest.mark.parametrize("H,Hd", [(8, 64), (32, 128), (3, 64)])
@pytest.mark.parametrize("lens", LENS, ids=lambda x: f"{len(x)}x{max(x)}")
def test_same_as_unsplit(device, lens, H, Hd, io, kv):
    print(f"balanced decode {lens[:6]} H {H} Hd {Hd} {io} {kv}", flush=True)
    args, lists = _batch(device, lens, H, Hd, io, kv)
    dev = [t.to(device) for t in args]
    # (the balanced launch is the one that runs)
    assert _lib.load().pa_decode_workspace_size(len(lens), H, Hd, dev[3].shape[1], DECODE_BALANCED) > 0
    want = paged_attention_decode_hip(*dev, split_blocks=0).float()
    out = torch.full_like(dev[0], 9.0)
    got = paged_attention_decode_hip(*dev, split_blocks=DECODE_BALANCED, out=out).float()
    # fp32 sums in another order (values of N(0, 1) averaged: at most a few ulp of 1); bf16 outputs may
    # round to the neighbour, 2^-8 of their size
    bound = 4e-6 if io == torch.float32 else 2.0**-8 * float(want.abs().max()) + 4e-6
    assert float((got - want).abs().max()) <= bound
    if len(lens) < 40 and max(lens) <= 4000:
        ref = oracle.paged_attention(*(x.float() for x in args[:3]), lists, lens, [1] * len(lens))
        assert float((got.cpu() - torch.as_tensor(ref)).abs().max()) <= (1e-4 if io == torch.float32 else 2e-2)


def test_two_streams_and_graph_replays(device):
    """Each call takes its own records: calls on two streams at once, and a captured call replayed between
    eager ones, give what they give alone."""
    cases = [_batch(device, lens, 32, 128, torch.float32, torch.bfloat16, seed)[0]
             for seed, lens in ((1, [9000, 30, 700, 2500]), (2, [64, 12000, 5000]))]
    cases = [[t.to(device) for t in c] for c in cases]
    call = lambda c, **kw: paged_attention_decode_hip(*c, split_blocks=DECODE_BALANCED, **kw)  # noqa: E731
    want = [call(c).clone() for c in cases]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(10):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(call(cases[i]))
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(g, want[i]) for g in got[i])
    out = torch.empty_like(want[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(cases[0], out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        other = call(cases[1])
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]) and torch.equal(other, want[1])


def test_limits(device):
    """More requests than one workgroup lists, another block size, or no workspace: the call runs unsplit."""
    lib = _lib.load()
    assert lib.pa_decode_workspace_size(513, 8, 64, 600, DECODE_BALANCED) == 0
    assert lib.pa_decode_workspace_size(8, 8, 96, 600, DECODE_BALANCED) == 0
    assert lib.pa_decode_workspace_size(8, 1 << 20, 64, 600, DECODE_BALANCED) == 0
    assert default_split_blocks(513, 8, 600, device) == 0 and default_split_blocks(64, 8, 600, device) == DECODE_BALANCED
    assert default_split_blocks(64, 32, 600, device, True) == 0
    args, _ = _batch(device, [5] * 600, 2, 64, torch.float32, torch.float32)
    dev = [t.to(device) for t in args]
    assert torch.equal(paged_attention_decode_hip(*dev, split_blocks=DECODE_BALANCED),
                       paged_attention_decode_hip(*dev, split_blocks=0))
    q, k, v, table, seq, cur = dev = [t.to(device) for t in _batch(device, [300, 9], 8, 64, torch.float32, torch.float32)[0]]
    want, out = paged_attention_decode_hip(*dev, split_blocks=0), torch.empty_like(q)
    for fn, tail in ((lib.pa_decode, (None, 0)), (lib.pa_decode_noalloc, ())):
        out.fill_(9.0)
        st = fn(q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), out.stride(0), out.stride(1), 0, k.data_ptr(),
                v.data_ptr(), 0, k.shape[0], table.data_ptr(), table.stride(0), table.shape[1], seq.data_ptr(),
                cur.data_ptr(), None, 2, 8, 64, 16, 1 / math.sqrt(64), DECODE_BALANCED, *tail,
                torch.cuda.current_stream().cuda_stream)
        assert st == 0 and torch.equal(out, want)


def _entry(lib, dev, out, split, ws, nbytes):
    """pa_decode itself, on a workspace of the caller's."""
    q, k, v, table, seq, cur = dev
    B, H, _, Hd = q.shape
    return lib.pa_decode(q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), out.stride(0), out.stride(1),
                         _lib.dtype_code(q.dtype), k.data_ptr(), v.data_ptr(), _lib.dtype_code(k.dtype), k.shape[0],
                         table.data_ptr(), table.stride(0), table.shape[1], seq.data_ptr(), cur.data_ptr(), None,
                         B, H, Hd, 16, 1 / math.sqrt(Hd), split, ws.data_ptr(), nbytes,
                         torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("io,kv", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)],
                         ids=["fp32", "bf16"])
def test_one_workspace_for_balanced_and_split_calls(device, io, kv):
    """A workspace zeroed once serves balanced and split calls in any order: the balanced launch's records
    stay clear of the arrival counters, which are zero after every call."""
    lib = _lib.load()
    dev = [t.to(device) for t in _batch(device, [900, 40, 1000], 8, 64, io, kv)[0]]
    sizes = [lib.pa_decode_workspace_size(3, 8, 64, dev[3].shape[1], s) for s in (DECODE_BALANCED, 16)]
    assert min(sizes) > 0
    ws = torch.zeros(max(sizes), dtype=torch.uint8, device=device)
    want = paged_attention_decode_hip(*dev, split_blocks=0).float()
    bound = 4e-6 if io == torch.float32 else 2.0**-8 * float(want.abs().max()) + 4e-6  # (as above)
    for split in (DECODE_BALANCED, 16, 16, DECODE_BALANCED, 16):
        out = torch.full_like(dev[0], 9.0)
        assert _entry(lib, dev, out, split, ws, ws.numel()) == 0
        assert float((out.float() - want).abs().max()) <= bound, split
        assert int(torch.count_nonzero(ws[:256 << 10])) == 0, split


def test_a_workspace_too_small_for_the_records_runs_unsplit(device):
    """As without a workspace: the balanced launch is a wish, whatever memory comes with the call."""
    lib = _lib.load()
    dev = [t.to(device) for t in _batch(device, [900, 40, 1000], 8, 64, torch.float32, torch.float32)[0]]
    need = lib.pa_decode_workspace_size(3, 8, 64, dev[3].shape[1], DECODE_BALANCED)
    assert need > 0
    ws = torch.zeros(need, dtype=torch.uint8, device=device)
    want = paged_attention_decode_hip(*dev, split_blocks=0)
    for nbytes in (0, 4096, 256 << 10):
        out = torch.full_like(dev[0], 9.0)
        assert _entry(lib, dev, out, DECODE_BALANCED, ws, nbytes) == 0, lib.pa_last_error_message()
        assert torch.equal(out, want) and int(torch.count_nonzero(ws)) == 0


@pytest.mark.parametrize("fill", ["random", "ones", "earlier call"])
def test_any_state_of_the_workspace(device, fill):
    """The tickets and records need no initial state: noise, all ones, or what a call of another shape left."""
    lib = _lib.load()
    cases = [[t.to(device) for t in _batch(device, lens, H, Hd, torch.float32, kv, 5)[0]]
             for lens, H, Hd, kv in (([3000, 1, 700, 2500], 8, 64, torch.float32),
                                     ([900] * 30 + [6000], 32, 128, torch.bfloat16), ([1500, 700], 3, 64, torch.float32))]
    size = max(lib.pa_decode_workspace_size(c[0].shape[0], c[0].shape[1], c[0].shape[3], c[3].shape[1], DECODE_BALANCED)
               for c in cases)
    ws = torch.zeros(size, dtype=torch.uint8, device=device)
    want = [paged_attention_decode_hip(*c, split_blocks=0) for c in cases]
    first = [None] * 3
    for rep in range(3):
        for i, c in enumerate(cases):
            if fill == "random":
                ws.random_(0, 256)
            elif fill == "ones":
                ws.fill_(255)
            out = torch.full_like(c[0], 9.0)
            assert _entry(lib, c, out, DECODE_BALANCED, ws, size) == 0
            assert float((out - want[i]).abs().max()) <= 4e-6, (rep, i)  # (as test_same_as_unsplit)
            assert rep == 0 or torch.equal(out, first[i])  # whichever gang arrives last
            first[i] = out


@pytest.mark.parametrize("lens", [[40] * 16, [9000, 30, 700, 2500] * 4], ids=["short", "long"])
def test_one_launch(device, lens):
    """A balanced call is one kernel, whatever it has to merge: a server that hands one wide table for short
    contexts pays for no second one."""
    import ctypes
    from pathlib import Path

    hip = ctypes.CDLL(str(Path(torch.__file__).parent / "lib" / "libamdhip64.so"))
    dev = [t.to(device) for t in _batch(device, lens, 32, 128, torch.bfloat16, torch.bfloat16, extra_pages=600)[0]]
    out = torch.empty_like(dev[0])
    want = paged_attention_decode_hip(*dev, out=torch.empty_like(out)).clone()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        assert default_split_blocks(len(lens), 32, dev[3].shape[1], device) == DECODE_BALANCED
        paged_attention_decode_hip(*dev, out=out)
    nodes = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    assert nodes.value == 1
    graph.instantiate()
    for _ in range(2):
        out.fill_(9.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
