"""Block-sparse attention of batches with few units (rows shared by several waves): every number of rows to a
workgroup, the edges of the rule that picks it, padding, scores that outgrow the pipelined loop's reference, and
the caller's plan, against the oracle."""
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


@pytest.mark.parametrize("heads,lens,scale", [
    (1, [64], 1.0),                                   # one row, one tile: seven of its eight waves have none
    (12, [512], 1.0),                                 # 8 waves to a row
    (3, [704, 768, 64], 1.0),                         # sequences of 11 and 12 blocks: the last without and the first with global rows
    (12, [1024, 1088], 1.0),                          # 4 waves to a row
    (5, [2048, 832, 64], 40.0),                       # scores beyond the pipelined loop's range
    (12, [256, 1024, 640, 896], 1.0),                 # 2 waves to a row
    (12, [2048, 3008, 384], 1.0),                     # a wave to a row, global rows by 8 waves
    (2, [64] * 64, 1.0),                              # as many sequences as lanes
    (2, [64] * 64 + [128], 1.0),                      # one more: the persistent kernel
    (8, [4096 * 4], 1.0),                             # global rows of 256 tiles
    (11, [64 * 128, 64 * 128], 6.0),                  # 2816 units, the most the rule takes
])
@pytest.mark.parametrize("padded", [False, True])
def test_few_units(capi, heads, lens, scale, padded):
    print("few units", heads, lens[:4], scale, padded, flush=True)
    g = torch.Generator().manual_seed(heads + len(lens))
    t = sum(lens)
    q, k, v = (torch.randn(t, heads, 64, generator=g).half().cuda() for _ in range(3))
    q = q * scale
    tokens = [max(1, n - 17 - 3 * i) for i, n in enumerate(lens)] if padded else None
    max_pos = max(4096, max(lens))
    out, ref = lh.run_attention(capi, q, k, v, lens, heads, seed=3, seq_tokens=tokens, max_pos=max_pos)
    # weights and output rounded to half (2^-11 of values up to max |v| each), scores summed in float from the same halves
    tol = 4 * 2.0 ** -11 * v.float().abs().max().item()
    assert (out.float().cpu() - ref).abs().max().item() <= tol
    plan, _ = lh.run_attention(capi, q, k, v, lens, heads, seed=3, seq_tokens=tokens, max_pos=max_pos, n_wg=7)
    assert (plan.float().cpu() - ref).abs().max().item() <= tol
    if len(lens) <= 64:
        assert torch.equal(plan, out)                 # the caller's plan changes the order, not a unit's arithmetic
