"""The append's vector kernel and its element-wise fallback (head_dims that are no whole number of
vectors, strides and bases off the 16-byte grid): every dtype pair, bit-exact against torch."""
import pytest
import torch

from src.kernels.hip_paged_attention import kv_append_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dst", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 1, 1, 8), (3, 2, 5, 12), (2, 8, 37, 64), (5, 3, 130, 128), (2, 3, 9, 10)],
                         ids=str)
@pytest.mark.parametrize("layout", ["rows", "heads", "offset", "odd_stride"])
def test_append_layouts_bit_exact(device, src, dst, shape, layout):
    B, H, T, Hd = shape
    g = torch.Generator().manual_seed(B * T + Hd)
    pad = {"offset": 1, "odd_stride": 3}.get(layout, 0)

    def rows():
        if layout == "heads":
            return torch.randn(B, H, T, Hd, generator=g).to(src).to(device)
        x = torch.randn(B * T * H * (Hd + pad) + 8, generator=g)
        x[:: 97] = float("inf")
        x[5:: 89] = float("nan")
        x = x.to(src).to(device)
        if layout == "odd_stride":
            return x[: B * T * H * (Hd + pad)].view(B, T, H, Hd + pad)[..., :Hd].transpose(1, 2)
        off = 1 if layout == "offset" else 0
        return x[off:off + B * T * H * Hd].view(B, T, H, Hd).transpose(1, 2)

    k, v = rows(), rows()
    blocks = B * T // 16 + 3
    kp = torch.randn(blocks, H, 16, Hd, generator=g).to(dst).to(device)
    vp = torch.randn(blocks, H, 16, Hd, generator=g).to(dst).to(device)
    want_k, want_v = kp.clone(), vp.clone()
    slots = torch.randperm(blocks * 16, generator=g)[: B * T].to(torch.int32)
    slots[:: 7] = -1
    slots[1:: 11] = blocks * 16 + 5  # past the pool: skipped
    kv_append_hip(k, v, kp, vp, slots.to(device))
    keep = ((slots >= 0) & (slots < blocks * 16)).to(device)
    at = slots.to(device)[keep].long()
    for pool, new in ((want_k, k), (want_v, v)):
        pool[at // 16, :, at % 16] = new.transpose(1, 2).reshape(B * T, H, Hd)[keep].to(dst)
    bits = torch.int32 if dst == torch.float32 else torch.int16
    for got, want in ((kp, want_k), (vp, want_v)):
        same = (got.view(bits) == want.view(bits)) | (got.isnan() & want.isnan())
        assert bool(same.all())
