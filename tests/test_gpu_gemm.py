"""The library's own dense products (rt_gemm_bt in a 16-bit type, rt_qkv_project) against fp32 references, at the
sizes where tiles, columns and reduction steps end unevenly."""
import pytest
import torch

import __graft_entry__ as graft

pytestmark = pytest.mark.gpu

BITS = {torch.float16: 10, torch.bfloat16: 7}


@pytest.fixture(scope="module")
def capi():
    p = graft.load_package()
    p.capi.lib()
    assert torch.cuda.is_available()
    return p.capi


def operands(m, n, k, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    return r(m, k), r(n, k) * 0.05, r(n)


def check(got, a, b, bias, gelu, dtype):
    """Per element: half a unit in the last place of the stored type, plus the error an fp32 sum of k terms may have in
    any order (k * 2^-24 * sum |a| |b|, twice for the reference's own), carried through the GELU's slope (<= 1.13) and
    its fp32 exponential and reciprocal (a few 2^-23 of the argument)."""
    a, b = a.float(), b.float()
    x = a @ b.t()
    acc = 2.0 ** -23 * a.shape[1] * (a.abs() @ b.abs().t())
    if bias is not None:
        x = x + bias.float()
        acc = acc + 2.0 ** -23 * x.abs()
    want = torch.nn.functional.gelu(x, approximate="tanh") if gelu else x
    ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -14))) - BITS[dtype])
    bound = 0.51 * ulp + 1.13 * acc + 2.0 ** -20 * x.abs()
    over = ((got.float() - want).abs() - bound).max().item()
    assert over <= 0, over


@pytest.mark.parametrize("m,n,k,dtype", [
    (12288, 256, 128, torch.float16),       # the shortest reduction: a tile's first step is followed by its last
    (12295, 264, 192, torch.bfloat16),      # odd number of steps; 8 columns and 7 rows in tiles of their own
    (9409, 520, 768, torch.float16),        # tiles of 224 rows: one row in the last
    (16384 + 33, 1000, 256, torch.bfloat16),
])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_gemm_bt_edges(capi, m, n, k, dtype, epilogue):
    print("gemm_bt", m, n, k, dtype, epilogue, flush=True)
    a, b, bias = operands(m, n, k, dtype)
    c = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
    capi.Gemm().bt(a, b, c[:m], bias=bias if epilogue else None, epilogue=epilogue)
    check(c[:m], a, b, bias if epilogue else None, epilogue == 2, dtype)
    assert bool((c[m] == 7.0).all())                   # nothing past the last row


@pytest.mark.parametrize("heads,seq_lens,dtype", [
    (12, [832, 64, 3008, 1024], torch.float16),
    (5, [64] * 70 + [2048], torch.bfloat16),          # more sequences than one wave looks up at a time, K and V halves of a tile
    (16, [4096, 320], torch.float16),
])
def test_qkv_project_equals_gemm_and_split(capi, heads, seq_lens, dtype):
    print("qkv_project", heads, len(seq_lens), dtype, flush=True)
    t, d = sum(seq_lens), heads * 64
    x, w, bias = operands(t, 3 * d, d, dtype, seed=1)
    sb = torch.from_numpy(capi.seq_prefix_blocks(seq_lens)).cuda()
    rows, k, vt = torch.full((t, 3 * d), 7.0, dtype=dtype, device="cuda"), *(torch.zeros(t * d, dtype=dtype, device="cuda") for _ in "kv")
    capi.qkv_project(x, w, bias, rows, k, vt, sb, heads)
    rows2, k2, vt2 = torch.empty_like(rows), torch.empty_like(k), torch.empty_like(vt)
    capi.Gemm().bt(x, w, rows2, bias=bias, epilogue=capi.RT_EPILOGUE_BIAS)
    check(rows2, x, w, bias, False, dtype)
    capi.qkv_bias_split(rows2, None, None, k2, vt2, sb, heads, 1.0)
    assert torch.equal(rows[:, :d], rows2[:, :d]) and torch.equal(k, k2) and torch.equal(vt, vt2)
    assert bool((rows[:, d:] == 7.0).all())            # only the queries' columns are written
