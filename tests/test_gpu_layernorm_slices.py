"""LayerNorm over the fp32 slices of a product (rt_slices_residual_layernorm) against torch in fp64, for every number of slices
that has a kernel of its own and for more, at row counts that leave a workgroup partly empty."""
import ctypes

import pytest
import torch

import __graft_entry__ as graft

pytestmark = pytest.mark.gpu

BITS = {torch.float16: 10, torch.bfloat16: 7}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,hidden", [(1, 256), (5, 512), (67, 768), (130, 1024)])
@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 8])
def test_slices_residual_layernorm(parts, rows, hidden, dtype):
    capi = graft.load_package().capi
    g = torch.Generator(device="cuda").manual_seed(parts * rows)
    r = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    slices, residual, bias, beta = r(parts, rows, hidden), r(rows, hidden).to(dtype), r(hidden).to(dtype), r(hidden).to(dtype)
    gamma = (1 + 0.1 * r(hidden)).to(dtype)
    out = torch.empty(rows, hidden, dtype=dtype, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    capi.check(capi.lib().rt_slices_residual_layernorm(ptr(out), ptr(slices), parts, ptr(residual), ptr(bias), ptr(gamma), ptr(beta),
                                                       rows, hidden, 1e-5, capi._dtype_code(out), capi._stream()))
    x = slices.double().sum(0) + residual.double() + bias.double()
    y = (x - x.mean(1, keepdim=True)) * torch.rsqrt(x.var(1, unbiased=False, keepdim=True) + 1e-5)
    want = y * gamma.double() + beta.double()
    # half a unit in the last place of the stored type, and of the fp32 terms a few units each: the row's sum, mean and scale
    ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -14))) - BITS[dtype])
    bound = 0.51 * ulp + 2.0 ** -20 * (1 + y.abs() * gamma.double().abs() + beta.double().abs())
    assert ((out.double() - want).abs() - bound).max().item() <= 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hidden", [256, 512, 768, 1024])
def test_slices_of_zeros_change_no_bit(hidden, dtype):
    """Four slices, and the same with one or four of zeros behind them: the kernels differ, the sums and the one rounding do not."""
    capi = graft.load_package().capi
    g = torch.Generator(device="cuda").manual_seed(hidden)
    r = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    rows = 2000
    slices = torch.cat([r(4, rows, hidden), torch.zeros(4, rows, hidden, device="cuda")])
    residual, bias, gamma, beta = r(rows, hidden).to(dtype), r(hidden).to(dtype), r(hidden).to(dtype), r(hidden).to(dtype)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    outs = []
    for parts in (4, 5, 8):
        out = torch.empty(rows, hidden, dtype=dtype, device="cuda")
        capi.check(capi.lib().rt_slices_residual_layernorm(ptr(out), ptr(slices), parts, ptr(residual), ptr(bias), ptr(gamma), ptr(beta),
                                                           rows, hidden, 1e-5, capi._dtype_code(out), capi._stream()))
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
