"""The fp32 wide prefill kernel forms fp32 products from three bf16 parts per operand: against float64 at
ordinary values, and against the 16-row kernel (fp32 matrix instructions) where a part would overflow."""
import pytest
import torch

from src.kernels.hip_paged_attention import PREFILL_BALANCED, paged_attention_prefill_hip, prefill_workspace_size

pytestmark = pytest.mark.gpu


def _case(Hd, lens, T, seed, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    B, H = len(lens), 8
    pages = max(-(-n // 16) for n in lens) + 1
    k, v = (torch.randn(B * pages, H, 16, Hd, generator=g) * scale for _ in range(2))
    table = torch.randperm(B * pages, generator=g).view(B, pages).to(torch.int32)
    q = torch.randn(B, H, T, Hd, generator=g).to(dtype)
    cur = [min(n, T) for n in lens]
    return q, k, v, table, lens, cur


def _run(case, device, monkeypatch, kernel, balance="off"):
    q, k, v, table, lens, cur = case
    monkeypatch.setenv("PAGED_HIP_PREFILL_KERNEL", kernel)
    monkeypatch.setenv("PAGED_HIP_PREFILL_BALANCE", balance)
    B, H, T, Hd = q.shape  # (the launch under test is the one that runs)
    assert (prefill_workspace_size(B, H, T, Hd, table.shape[1], PREFILL_BALANCED, k.dtype) > 0) == (balance == "force")
    return paged_attention_prefill_hip(q.to(device), k.to(device), v.to(device), table.to(device),
                                       torch.tensor(lens, dtype=torch.int32, device=device),
                                       torch.tensor(cur, dtype=torch.int32, device=device)).cpu()


def _f64(case):
    q, k, v, table, lens, cur = case
    out = torch.zeros(q.shape, dtype=torch.float64)
    for b, (n, c) in enumerate(zip(lens, cur)):
        kk, vv = (p[table[b].long()].transpose(0, 1).reshape(q.shape[1], -1, q.shape[3])[:, :n].double() for p in (k, v))
        s = q[b].double() @ kk.transpose(1, 2).contiguous() / q.shape[3] ** 0.5
        limit = torch.clamp(n - c + 1 + torch.arange(q.shape[2]), max=n)
        s.masked_fill_(torch.arange(n)[None, :] >= limit[:, None], float("-inf"))
        out[b] = torch.softmax(s, -1) @ vv
    return out


@pytest.mark.parametrize("balance", ["off", "force"])
@pytest.mark.parametrize("Hd", [64, 128])
@pytest.mark.parametrize("lens,T", [([1], 1), ([33, 31, 32], 33), ([130, 700, 257], 129), ([1500], 300)], ids=str)
def test_error_of_fp32_sums(device, monkeypatch, Hd, lens, T, balance):
    case = _case(Hd, lens, T, Hd + T)
    want = _f64(case)
    got = _run(case, device, monkeypatch, "wide", balance)
    err = float((got.double() - want).norm() / want.norm())
    # at most 12 rounded additions per 32 keys and output, each half an ulp of the running sum at most and
    # of either sign; 4 more for the scores, the weights and the division
    assert err <= 2.0**-24 * (4 + (12 * max(lens) / 32) ** 0.5), err


@pytest.mark.parametrize("balance", ["off", "force"])
@pytest.mark.parametrize("Hd", [64, 128])
@pytest.mark.parametrize("where", ["k", "v", "q"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), -3.4028234663852886e38, 3e38, 2.0**61])
def test_values_without_a_finite_split(device, monkeypatch, where, value, Hd, balance):
    lens, T = [150, 70], 140
    case = _case(Hd, lens, T, 3)
    q, k, v, table, _, _ = case
    if where == "q":
        q[0, 1, 137, 5] = value
        q[1, 2, 3, Hd - 1] = value
    else:
        pool = k if where == "k" else v
        pool[table[0, 2], 1, 3, 7] = value        # key 35 of request 0
        pool[table[1, 4], 3, 5, Hd - 2] = value   # its last keys
    got = _run(case, device, monkeypatch, "wide", balance)
    ref = _run(case, device, monkeypatch, "tile")
    # to 1e-5 (float32 sums of up to 150 keys in another order) of the row's largest value
    bound = 1e-5 * ref.nan_to_num(0, 0, 0).abs().amax(-1, keepdim=True).clamp(min=1.0).expand_as(ref)
    same = (got - ref).abs() <= bound
    reached = torch.zeros_like(ref, dtype=torch.bool)  # outputs that a planted value reaches
    if where == "q":
        reached[0, 1, 137] = reached[1, 2, 3] = True
    elif where == "k":
        reached[0, 1, 25:] = reached[1, 3] = True  # (row 25 of request 0 sees keys 0-35)
    else:  # (its own column)
        reached[0, 1, :, 7] = reached[1, 3, :, Hd - 2] = True
    assert bool(ref[~reached].isfinite().all()) and bool(same[~reached].all())
    if abs(value) < 1e30:
        assert bool(ref.isfinite().all()) and bool(same.all())
    elif where == "v":
        sees = reached.clone()  # rows that see the key; to the others its weight is 0, and 0 * inf is NaN
        sees[0, 1, :25] = sees[1, 3, :69] = False
        if abs(value) < float("inf"):  # (the value times a weight of up to 2^8 may overflow on the way)
            both = got.isfinite() & ref.isfinite()
            assert bool(same[reached & both].all()) and bool(both[reached & ~sees].all())
            one = sees & (got.isfinite() != ref.isfinite())
            assert bool((torch.where(got.isfinite(), got, ref).abs() > 1e35)[one].all())
        else:
            assert torch.equal(got[sees].isnan(), ref[sees].isnan())
            assert torch.equal(got[sees].nan_to_num(0, 1, -1), ref[sees].nan_to_num(0, 1, -1))
            assert bool((same | got.isnan())[reached & ~sees & ref.isfinite()].all())
    else:  # scores without a number: a NaN row, or 0 (no positive weight sum)
        number = ref.isfinite() & (ref != 0)
        assert bool(same[reached & number].all())
        assert bool((~got.isfinite() | (got == 0))[reached & ~number].all())


@pytest.mark.parametrize("balance", ["off", "force"])
@pytest.mark.parametrize("Hd", [64, 128])
@pytest.mark.parametrize("where", ["k", "v", "q"])
@pytest.mark.parametrize("value", [3.4028234663852886e38, -3.4028234663852886e38, 3e38])
def test_values_that_only_fp32_products_hold(device, monkeypatch, where, value, Hd, balance):
    """Finite results from values whose parts are not finite: the products are formed again in fp32, or the
    outputs would be NaN. The other operand is small enough for every product to be finite."""
    assert torch.tensor(value * 2.0**24, dtype=torch.float64).bfloat16().isinf()  # (V's leading part)
    lens, T, d = [150, 70], 140, 7
    q, k, v, table, _, _ = case = _case(Hd, lens, T, 11)
    at = table[0, 2], 1, 3      # key 35 of request 0, head 1
    last = table[1, 4], 3, 5    # the last key of request 1, head 3
    if where == "v":  # that key's score is far below the others', its weight about 1e-9
        q.abs_()
        k.abs_()
        for x in (at, last):
            k[x] *= -1
            v[x][d] = value
    else:  # scores of size 1: value * 1e-37 among the products
        big, small = (k, q) if where == "k" else (q, k)
        small[..., d] = 1e-37
        for x in (at, last) if where == "k" else ((0, 1, 137), (1, 2, 3)):
            big[x][d] = value
        if where == "k":
            assert torch.tensor(value).bfloat16().isinf() or abs(value) < 3.39e38
    want = _f64(case)
    assert bool(want.isfinite().all())
    got = _run(case, device, monkeypatch, "wide", balance).double()
    assert bool(got.isfinite().all())
    # fp32 sums of values of N(0, 1), and the planted one's weight, whose exponent of about 30 is rounded to fp32
    assert bool(((got - want).abs() <= 1e-5 + 1e-4 * want.abs()).all())


@pytest.mark.parametrize("scale", [1e-30, 1e-12, 1e12])
def test_scales_far_from_one(device, monkeypatch, scale):
    q, k, v, table, lens, cur = _case(128, [300, 90], 140, 9)
    case = (q / scale, k * scale, v * scale, table, lens, cur)
    got, ref = _run(case, device, monkeypatch, "wide"), _run(case, device, monkeypatch, "tile")
    assert float((got - ref).abs().max()) < 1e-5 * scale


@pytest.mark.parametrize("balance", ["off", "force"])
@pytest.mark.parametrize("Hd", [64, 128])
@pytest.mark.parametrize("exponent", [-100, -112, -120, -126, -136, -147])
def test_small_values_keep_their_bits(device, monkeypatch, exponent, Hd, balance):
    """V down to fp32's denormals, whose bf16 parts would be no normal numbers."""
    q, k, v, table, lens, cur = _case(Hd, [150, 700], 140, Hd - exponent)
    case = (q, k, v * 2.0**exponent, table, lens, cur)
    want = _f64(case)
    got = _run(case, device, monkeypatch, "wide", balance).double()
    # as test_error_of_fp32_sums, and two roundings to the denormals' spacing
    bound = 2.0**-24 * (4 + (12 * max(lens) / 32) ** 0.5) * float(want.norm()) + 2.0**-149 * want.numel() ** 0.5
    assert float((got - want).norm()) <= bound
