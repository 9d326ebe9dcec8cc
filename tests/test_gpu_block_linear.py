"""The block kernel of LayerNorm layers over many rows (128 x 64 output tiles; fp32 products from three bf16
parts): tile edges and every epilogue against float64, and values without a finite split against torch."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from src.kernels.hip_linear import linear_rows_hip, qkv_append_hip

pytestmark = pytest.mark.gpu
K = 512


def _layer(N, dtype, device, seed, bias=True):
    torch.manual_seed(seed)
    lin, ln = nn.Linear(K, N, bias=bias), nn.LayerNorm(K)
    nn.init.normal_(ln.weight, 1, 0.2)
    nn.init.normal_(ln.bias, 0, 0.2)
    return lin.to(dtype).to(device), ln.to(dtype).to(device)


def _want(x, lin, ln):
    h = F.layer_norm(x.double(), (K,), ln.weight.double(), ln.bias.double(), ln.eps)
    if x.dtype == torch.bfloat16:
        h = h.bfloat16().double()  # (the normalised rows are bf16 operands)
    y = h @ lin.weight.double().t().contiguous()
    return y + lin.bias.double() if lin.bias is not None else y


# fp32: sums of 512 products and a LayerNorm; bf16: one rounding of the output, and of operands that fall
# on the other side of a rounding boundary
def _bound(dtype):
    return 1e-6 if dtype == torch.float32 else 4e-3


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N", [(1, 64), (127, 65), (128, 2048), (129, 16), (300, 200), (2048, 63)])
@torch.no_grad()
def test_tile_edges_and_epilogues(device, monkeypatch, dtype, M, N):
    monkeypatch.setenv("PAGED_HIP_LINEAR_KERNEL", "block")
    lin, ln = _layer(N, dtype, device, M + N, bias=N != 16)
    wide = torch.randn(M, K + 8, device=device).mul_(3).add_(1.5).to(dtype)
    x = wide[:, :K]  # (a row stride of its own)
    res = torch.randn(M, N, device=device).to(dtype)
    want = _want(x, lin, ln)
    for gelu, r in ((False, None), (True, None), (False, res)):
        copy = torch.empty(M, N, device=device, dtype=dtype) if r is not None else None
        got = linear_rows_hip(x, lin, ln=ln, gelu=gelu, residual=r, copy_to=copy)
        ref = (F.gelu(want) if gelu else want) + (r.double() if r is not None else 0)
        assert float((got.double() - ref).norm() / ref.norm()) < _bound(dtype)
        assert copy is None or torch.equal(copy, got)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pool", [torch.float32, torch.bfloat16])
@torch.no_grad()
def test_qkv_scatter(device, monkeypatch, dtype, pool):
    M, H, Hd = 200, 8, 64
    layers = [_layer(K, dtype, device, i) for i in range(3)]
    attn = type("A", (), {n: l[0] for n, l in zip(("q_proj", "k_proj", "v_proj"), layers)})()
    ln = layers[0][1]
    x = torch.randn(M, K, device=device).to(dtype)
    slots = torch.randperm(20 * 16, device=device)[:M].to(torch.int32)
    slots[::9] = -1
    slots[5::31] = 20 * 16 + 3
    out = {}
    for kernel in ("block", "tiled"):
        monkeypatch.setenv("PAGED_HIP_LINEAR_KERNEL", kernel)
        pools = [torch.full((20, H, 16, Hd), 7.0, device=device, dtype=pool) for _ in range(2)]
        out[kernel] = [qkv_append_hip(x, ln, attn, *pools, slots), *pools]
    for a, b in zip(out["block"], out["tiled"]):
        assert torch.equal(a == 7, b == 7)
        low = dtype == torch.bfloat16 or pool == torch.bfloat16
        assert float((a.float() - b.float()).norm() / b.float().norm()) < (4e-3 if low else 1e-6)


def _same(got, want, rel):
    """Numbers to a relative error, infinities and NaNs by themselves."""
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    ok = want.isfinite()
    assert float((got - want)[ok].norm()) <= rel * float(want[ok].norm())


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3e38, -2.0**61])
@torch.no_grad()
def test_values_without_a_finite_split(device, monkeypatch, value):
    """In the weights (one output column) and in the rows (one row): only what they reach differs."""
    monkeypatch.setenv("PAGED_HIP_LINEAR_KERNEL", "block")
    M, N = 150, 130
    lin, ln = _layer(N, torch.float32, device, 3)
    x = torch.randn(M, K, device=device)
    lin.weight[7, 11] = value
    got, want = linear_rows_hip(x, lin, ln=ln), _want(x, lin, ln).float()
    keep = torch.arange(N, device=device) != 7
    _same(got[:, keep], want[:, keep], 1e-6)
    _same(got[:, 7], want[:, 7], 1e-6)
    lin.weight[7, 11] = 0.1
    x[140, 3] = value
    got, want = linear_rows_hip(x, lin, ln=ln), _want(x, lin, ln).float()
    keep = torch.arange(M, device=device) != 140
    _same(got[keep], want[keep], 1e-6)
    if abs(value) < 1e19:  # (the row's variance is an fp32 number)
        _same(got[140], want[140], 1e-6)
    elif not abs(value) < float("inf"):
        assert bool(got[140].isnan().all())


@pytest.mark.parametrize("where", ["weight", "norm"])
@pytest.mark.parametrize("value", [3.4028234663852886e38, -3.4028234663852886e38, 3e37])
@torch.no_grad()
def test_values_that_only_fp32_products_hold(device, monkeypatch, where, value):
    """Finite results from values whose parts are not finite: the products are formed again in fp32, or the
    outputs would be NaN. The other operand is small enough for every product to be finite."""
    assert torch.tensor(value * 2.0**24, dtype=torch.float64).bfloat16().isinf()  # (the leading part)
    monkeypatch.setenv("PAGED_HIP_LINEAR_KERNEL", "block")
    M, N = 150, 130
    lin, ln = _layer(N, torch.float32, device, 3)
    x = torch.randn(M, K, device=device)
    if where == "weight":
        ln.weight[11], ln.bias[11] = 1e-3, 0.0
        lin.weight[7, 11] = value
    else:
        ln.weight[11], ln.bias[11] = value / 8, 0.0  # (rows of up to 5 standard deviations)
        lin.weight[:, 11] *= 1e-3
    want = _want(x, lin, ln)
    assert bool(want.isfinite().all())
    got = linear_rows_hip(x, lin, ln=ln).double()
    assert bool(got.isfinite().all())
    cols = torch.arange(N, device=device) == 7 if where == "weight" else torch.ones(N, dtype=torch.bool, device=device)
    assert float(((got - want)[:, cols]).abs().max()) <= 1e-6 * float(want[:, cols].abs().max())
    if where == "weight":
        assert float((got - want)[:, ~cols].norm()) < 1e-6 * float(want[:, ~cols].norm())


@pytest.mark.parametrize("side", [-1, 0, 1, 256])
@torch.no_grad()
def test_default_choice_near_its_line(device, monkeypatch, side):
    """fc1-shaped layers on both sides of the line (four and a half tiled workgroups per compute unit; 544 and
    545 rows on 256): the default call gives the bits of the kernel that the line says."""
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    line = 32 * (-(-9 * cus // 128) - 1)  # the most rows that stay with the tiled kernel: 64 column tiles
    rows = line + side
    lin, ln = _layer(2048, torch.float32, device, rows)
    x = torch.randn(rows, K, device=device)
    want = F.gelu(_want(x, lin, ln))
    out = {}
    for kernel in ("block", "tiled", ""):
        if kernel:
            monkeypatch.setenv("PAGED_HIP_LINEAR_KERNEL", kernel)
        else:
            monkeypatch.delenv("PAGED_HIP_LINEAR_KERNEL", raising=False)
        out[kernel] = linear_rows_hip(x, lin, ln=ln, gelu=True)
        assert float((out[kernel].double() - want).norm() / want.norm()) < 1e-6
    assert not torch.equal(out["block"], out["tiled"])
    assert torch.equal(out[""], out["block" if side > 0 else "tiled"])


@pytest.mark.parametrize("where", ["weight", "norm"])
@pytest.mark.parametrize("exponent", [-20, -90, -112, -120, -126, -136])
@torch.no_grad()
def test_small_values_keep_their_bits(device, monkeypatch, where, exponent):
    """Weights, or normalised rows, down to fp32's denormals, whose bf16 parts would be no normal numbers."""
    monkeypatch.setenv("PAGED_HIP_LINEAR_KERNEL", "block")
    lin, ln = _layer(130, torch.float32, device, -exponent, bias=False)
    x = torch.randn(150, K, device=device)
    if where == "weight":
        lin.weight.mul_(2.0**exponent)
    else:
        ln.weight.mul_(2.0**exponent)
        ln.bias.mul_(2.0**exponent)
    want = _want(x, lin, ln)
    # (the normalised rows are rounded to fp32, at denormal scales to their spacing, and so is the result)
    small = 2.0**-149 * (want.numel() ** 0.5) * (1 if where == "weight" else (1 + float(lin.weight.norm(dim=1).max())))
    assert float((linear_rows_hip(x, lin, ln=ln).double() - want).norm()) < 1e-6 * float(want.norm()) + small
