"""Block-sparse attention in fp32, whose products run on three bf16 parts of every operand: sizes at the edges of a tile's
halves and of the order in which rows are handed out, against the oracle to fp32's accuracy, and infinities, which the
parts cannot carry."""
import pytest
import torch

import __graft_entry__ as graft
from tests import layer_harness as lh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    p = graft.load_package()
    p.capi.lib()
    assert torch.cuda.is_available()
    return p.capi


@pytest.mark.parametrize("heads,lens,tokens,scale", [
    (1, [64], None, 1.0),                                       # one row: the first of its sequence and the last
    (3, [64, 128, 192, 64], None, 1.0),                         # sequences of one, two and three rows
    (3, [64, 128, 192, 64], [1, 96, 161, 32], 1.0),             # no key, some and all keys in the upper half of the last tile
    (2, [768, 64 * 40], [768 - 31, 64 * 40 - 63], 3.0),         # sparse rows and global rows of 40 tiles
    (7, [832, 1088], [65, 1088], 1.0),                          # whole blocks of padding; unit counts no multiple of 8
])
@pytest.mark.parametrize("n_wg", [0, 5])
def test_fp32_attention(capi, heads, lens, tokens, scale, n_wg):
    print("fp32 attention", heads, lens, tokens, n_wg, flush=True)
    g = torch.Generator().manual_seed(heads + len(lens))
    t = sum(lens)
    q, k, v = (torch.randn(t, heads, 64, generator=g).cuda() for _ in range(3))
    q = q * scale
    out, ref = lh.run_attention(capi, q, k, v, lens, heads, seed=3, n_wg=n_wg, seq_tokens=tokens)
    # sums of 64 products in fp32 on both sides: a score is off by up to 2 x 64 x 2^-24 x the largest product's size, a weight by
    # that share of itself, an output by that share of the largest value
    big = lambda x: x.abs().max().item()
    tol = 2 * 64 * 2.0 ** -24 * (1 + big(q) * big(k) / 8) * big(v)
    assert (out.cpu() - ref).abs().max().item() <= min(tol, 1e-4)


def test_fp32_attention_of_infinities(capi):
    heads, lens = 2, [1024, 256]
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(sum(lens), heads, 64, generator=g).cuda() for _ in range(3))
    k[100, 0, 3] = float("inf")            # a weight of zero, or no number at all, depending on the query's sign
    v[300, 1, 5] = -float("inf")
    v[1100, 0, 9] = float("nan")
    k[1200, 1, 0] = 3.4e38                 # finite, but not so when rounded to bf16
    out, ref = lh.run_attention(capi, q, k, v, lens, heads, seed=3)
    out = out.cpu()
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    assert 0 < int(out.isnan().sum()) < out.numel() // 2 and int(out.isinf().sum()) > 0
    assert torch.equal(out[out.isinf()], ref[out.isinf()])
    ok = out.isfinite()
    assert (out - ref)[ok].abs().max().item() <= 1e-4
