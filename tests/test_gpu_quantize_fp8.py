"""The fp8 quantisation kernel against the same steps as separate torch
operators: bytes and scales are equal, so no tolerance is involved."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _by_operators(x, per_token):
    amax = (x.abs().amax(dim=-1) if per_token else x.abs().amax()).clamp_min(1e-6).to(torch.float32)
    scale = amax / 448.0
    sc = scale.unsqueeze(-1) if per_token else scale
    return (x.to(torch.float32) / sc).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), scale


def _check(x, per_token):
    from late_interaction_kernels.fp8 import (_quantize_kernel, quantize_fp8_per_tensor, quantize_fp8_per_token)

    assert _quantize_kernel(x, torch.float8_e4m3fn, per_token) is not None  # the kernel takes this call
    got, scale = (quantize_fp8_per_token if per_token else quantize_fp8_per_tensor)(x)
    want, wscale = _by_operators(x, per_token)
    assert got.shape == x.shape and scale.shape == wscale.shape and scale.dtype == torch.float32
    assert torch.equal(scale, wscale) or torch.equal(scale.isnan(), wscale.isnan()) and torch.equal(
        scale.nan_to_num(), wscale.nan_to_num())
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))


# rows around the 64 / 32 / 16 of a workgroup, widths around the 16 chunks a
# lane group holds per register
@pytest.mark.parametrize("per_token", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 8), (63, 128), (65, 128), (3, 31, 96), (17, 136), (33, 256), (5, 264),
                                   (2, 512), (1030, 64), (5, 1030, 128)])
def test_quantize_equals_operators(shape, dtype, per_token):
    g = torch.Generator(device="cuda").manual_seed(shape[-1])
    x = torch.randn(*shape, generator=g, device="cuda") * torch.rand(*shape[:-1], 1, generator=g, device="cuda").exp2()
    _check(x.to(dtype), per_token)


@pytest.mark.parametrize("per_token", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_quantize_extremes(dtype, per_token):
    """Every 16-bit pattern (finite ones, per row of 128), then rows of zeros,
    the type's smallest and largest values, infinities and NaN."""
    bits = torch.arange(1 << 16, device="cuda", dtype=torch.int32).to(torch.int16)
    x = bits.view(torch.bfloat16 if dtype == torch.float32 else dtype).to(dtype)
    x = x[x.isfinite()]
    x = x[: x.numel() // 128 * 128]
    g = torch.Generator(device="cuda").manual_seed(1)
    _check(x.view(-1, 128), per_token)
    _check(x[torch.randperm(x.numel(), generator=g, device="cuda")].view(-1, 128), per_token)
    fi = torch.finfo(dtype)
    rows = torch.randn(8, 128, generator=g, device="cuda").to(dtype)
    rows[0] = 0
    rows[1] = -0.0
    rows[2, ::2], rows[2, 1::2] = fi.tiny, -fi.smallest_normal / 2
    rows[3, :3] = torch.tensor([fi.max, -fi.max, 1.0])
    rows[4, 5] = float("inf")
    rows[5, 6] = float("-inf")
    rows[6, 7] = float("nan")
    if per_token:
        _check(rows, True)
    else:
        for r in range(8):
            _check(rows[r : r + 1].clone(), False)


def test_quantize_other_calls_keep_the_operators():
    """Calls the kernel does not take: the operator chain's results."""
    from late_interaction_kernels.fp8 import _quantize_kernel, quantize_fp8_per_token

    x = torch.randn(4, 6, 128, device="cuda")
    for y in (x[..., ::2], x.transpose(0, 1), x[..., 1:127], x.cpu(), x.double(), x[:0]):
        assert _quantize_kernel(y, torch.float8_e4m3fn, True) is None
        q, s = quantize_fp8_per_token(y)
        want, ws = _by_operators(y, True)
        assert torch.equal(q.view(torch.uint8), want.contiguous().view(torch.uint8)) and torch.equal(s, ws)
    assert _quantize_kernel(x.requires_grad_(), torch.float8_e4m3fn, True) is None
    assert _quantize_kernel(x.detach(), torch.float8_e5m2, True) is None
    assert _quantize_kernel(x.detach().to(torch.bfloat16), torch.float8_e4m3fn, False) is not None
