"""bfaintb_quantize and bfaintb_prepack on the device against the torch form of the quantiser and the oracle's packing: byte for byte."""
import numpy as np
import pytest
import torch

import awesome_fusion_amd as af
import awesome_fusion_amd.torch_op as top
import oracle

pytestmark = pytest.mark.gpu


def _torch_form(w, bits, group):
    """quantize_weight's chain of torch operations, on the same device (its division by qmax is a product there)."""
    was = top._quantizes_on_device
    top._quantizes_on_device = lambda *a: False
    try:
        return top.quantize_weight(w, bits, group)
    finally:
        top._quantizes_on_device = was


# one tile and a fraction of the next in both directions, groups within a tile (32, 64, 128), across tiles and over all of k
@pytest.mark.parametrize("n,k,bits,group", [(16, 32, 4, 32), (16, 8, 8, 0), (272, 192, 4, 64), (144, 384, 8, 128), (528, 1000, 4, 0),
                                            (1040, 1000, 8, 0), (256, 768, 4, 256), (128, 288, 8, 96), (64, 16384, 8, 0), (2048, 2048, 4, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_codes_and_scales_are_the_torch_forms(n, k, bits, group, dtype):
    g = torch.Generator(device="cuda").manual_seed(n + k)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.05).to(dtype)
    w[0, :] = 0                                             # a group of zeros: the smallest scale
    w[1, : k // 2] = torch.arange(k // 2, device="cuda") % 15 / 2 - 3.5   # quotients half-way between codes
    w[2, 0] = 3e4
    b, s = top.quantize_weight(w, bits, group)
    assert top._quantizes_on_device(w, bits, group)
    b0, s0 = _torch_form(w, bits, group)
    assert torch.equal(s.view(torch.int16), s0.view(torch.int16))
    assert torch.equal(b, b0)
    strided = torch.zeros((n, k + 24), dtype=dtype, device="cuda")
    strided[:, :k] = w
    b1, s1 = top.quantize_weight(strided[:, :k], bits, group)
    assert torch.equal(b, b1) and torch.equal(s.view(torch.int16), s1.view(torch.int16))


@pytest.mark.parametrize("n,k,bits,group", [(48, 384, 4, 128), (144, 192, 8, 64), (272, 1000, 8, 0), (64, 768, 4, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_groups_with_nans_and_infinities_are_code_0(n, k, bits, group, dtype):
    """A NaN or an infinity makes its group's scale one and all of the group's codes 0; the other groups do not notice.  The
    largest finite weights stay finite: their group's extreme code times its scale is within half a step of them."""
    g = torch.Generator(device="cuda").manual_seed(n * k)
    w = (torch.randn((n, k), generator=g, device="cuda") * 0.05).to(dtype)
    size, zero = group or k, 128 if bits == 8 else 8
    codes = lambda b: b if bits == 8 else torch.stack((b & 15, b >> 4), dim=2).reshape(k, n)
    b0, s0 = top.quantize_weight(w, bits, group)
    hit = torch.zeros((k // size, n), dtype=torch.bool, device="cuda")
    x = w.clone()
    for row, col, value in ((0, 0, float("nan")), (3, k - 1, float("inf")), (4, size - 1, float("-inf")), (n - 1, k // 2, float("nan")), (9, 5, float("nan"))):
        x[row, col] = value
        hit[col // size, row] = True
    x[9, 6] = float("inf")
    b, s = top.quantize_weight(x, bits, group)
    assert torch.equal(~s.isfinite(), hit) and bool(s[0, 0].isnan()) and bool(s[0, 9].isnan()) and float(s[(k - 1) // size, 3]) == float("inf") == float(s[0, 4])
    assert torch.equal(s.view(torch.int16)[~hit], s0.view(torch.int16)[~hit])
    wide = hit.repeat_interleave(size, dim=0)
    assert bool((codes(b)[wide] == zero).all()) and torch.equal(codes(b)[~wide], codes(b0)[~wide])
    top_value = torch.finfo(dtype).max
    x = w.clone()
    x[1, 1], x[2, 2] = top_value, -top_value
    b, s = top.quantize_weight(x, bits, group)
    assert bool(s.isfinite().all())
    for row, at in ((1, 1), (2, 2)):
        value = (int(codes(b)[at, row]) - zero) * float(s[0, row])
        assert abs(value - float(x[row, at])) <= 0.51 * float(s[0, row])


@pytest.mark.parametrize("n,k,bits", [(16, 64, 8), (16, 128, 4), (272, 192, 8), (528, 384, 4), (4112, 64, 8), (48, 2048, 4)])
def test_packing_is_the_oracles(n, k, bits):
    rng = np.random.default_rng(n + k)
    b = rng.integers(0, 256, (k, n * bits // 8), dtype=np.uint8)
    got = top.prepack_weight(torch.from_numpy(b).cuda(), bits)
    assert np.array_equal(got.cpu().numpy(), oracle.pack_mfma16(b, k, n, bits))
    back = torch.zeros((k, n * bits // 8), dtype=torch.uint8, device="cuda")
    af.unpack(back, got, n, k, weight_bits=bits)
    assert np.array_equal(back.cpu().numpy(), b)
