"""How a launch cuts its rows: both sides of every line of the rule, more sequences than lanes, scores beyond the pipelined loop's
range in shared and unshared rows, padding that takes a row's first tile away; against the oracle, and a caller's plan against
the launch without one."""
import pytest
import torch

import __graft_entry__ as graft
from oracle import attention as oa
from tests import layer_harness as lh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    p = graft.load_package()
    p.capi.lib()
    assert torch.cuda.is_available()
    return p.capi


@pytest.mark.parametrize("cut,heads,blocks,scale,short", [
    ((4, 4, 4), 16, [16], 1.0, 0),                   # 256 units, the most whose every row four waves share
    ((4, 4, 4), 1, [3], 1.0, 63),                    # the shortest sequence whose rows are shared by four waves
    ((2, 4, 4), 1, [2], 1.0, 0),                     # by two waves
    ((2, 4, 4), 10, [26], 1.0, 9),                   # 260 units
    ((2, 4, 4), 10, [26], 40.0, 0),                  # the same beyond the pipelined loop's range
    ((2, 4, 4), 12, [34], 1.0, 0),                   # 216 workgroups so
    ((1, 4, 4), 12, [35], 1.0, 5),                   # 222 would be too many: a wave to a row
    ((4, 4, 4), 1, [75], 1.0, 0),                    # few units, on both sides of the line to workgroups of eight waves
    ((1, 8, 8), 1, [76], 1.0, 0),
    ((1, 4, 4), 12, [29] * 3, 1.0, 0),               # and where one round of those takes all
    ((1, 8, 8), 12, [30] * 3, 1.0, 7),
    ((1, 8, 8), 4, [250] + [2] * 9, 1.0, 7),         # one long sequence among short ones
    ((1, 8, 8), 6, [90], 1.0, 30),                   # a long sequence: eight waves to a global row
    ((1, 8, 8), 6, [90], 40.0, 30),
    ((1, 8, 8), 6, [100, 12, 90], 1.0, 1),
    ((1, 8, 8), 1, [600], 1.0, 0),                   # 75 tiles to a wave of a global row: the moving-maximum loop
    ((1, 4, 4), 1, [300] + [1] * 64, 1.0, 2),        # two shares of 38 tiles to each of four waves; more sequences than lanes
    ((1, 4, 4), 2, [300] + [10] * 30, 1.0, 0),       # the same with 31 sequences
    ((1, 4, 4), 2, [300] + [10] * 30, 40.0, 9),      # beyond the pipelined loop's range
    ((2, 4, 4), 1, [257] + [10] * 8, 1.0, 4),        # with two waves to the other rows, at the shortest sequence that takes them so
    ((2, 4, 4), 1, [256] + [10] * 8, 1.0, 4),        # 64 tiles to each of four waves
    ((1, 4, 4), 1, [600] + [1] * 64, 1.0, 1),        # 75 tiles to a share: the moving-maximum loop
    ((1, 4, 4), 2, [1 + i % 14 for i in range(65)], 1.0, 3),
    ((1, 4, 4), 1, [12 + i % 3 for i in range(130)], 40.0, 3),       # three chunks, every sequence with global rows
    ((1, 4, 4), 2, [1] * 80 + [13] + [1] * 15 + [2, 12, 1], 1.0, 0),  # sequences that begin and end a sixteen
    ((1, 4, 4), 1, [1] * 1023 + [14], 1.0, 1),       # the most sequences, the last of them with global rows
])
def test_rows(capi, cut, heads, blocks, scale, short):
    print("rows", cut, heads, blocks[:4], scale, short, flush=True)
    assert capi.bs_attention_cut(len(blocks), sum(blocks), heads) == cut
    lens = [64 * n for n in blocks]
    t, dtype = sum(lens), torch.float16
    gen = torch.Generator().manual_seed(t)
    q, k, v = (torch.randn(t, heads, 64, generator=gen).to(dtype) for _ in range(3))
    qs = (q.float() * (scale * lh.LOG2E / 8)).to(dtype)
    max_pos = max(4096, max(lens))
    sb, idx, pos, ph, sb_d, idx_d, pos_d = lh.device_plan(capi, lens, heads, max_pos=max_pos)
    tokens = [max(1, n - short) for n in lens] if short else None
    tok_d = None if tokens is None else torch.tensor(tokens, dtype=torch.int32).cuda()
    pack = lambda x, tr=False: lh.pack_heads(x, sb, transpose_v=tr).cuda()
    qp, kp, vp = pack(qs), pack(k), pack(v, True)

    def run(from_idx=None, from_pos=None):
        out = torch.full((t, heads * 64), float("nan"), dtype=dtype, device="cuda")
        capi.bs_attention_fwd(qp, kp, vp, out, sb_d, heads, idx_d, pos_d, ph, from_idx, from_pos, seq_tokens_dev=tok_d)
        return out
    out = run()
    fp, fi = capi.partition_lpt(sb, heads, 48)
    assert torch.equal(run(torch.from_numpy(fi).cuda(), torch.from_numpy(fp).cuda()), out)
    ref = oa.csr_attention(qs, k, v, sb.tolist(), idx, pos, ph, scale=1.0 / lh.LOG2E, seq_tokens=tokens)
    assert lh.excess(out.float().cpu(), ref, dtype) <= 0


def test_first_tile_is_padding(capi):
    """Rows that list the padded tile, or blocks that are padding as a whole, first: the loop starts from a tile that has keys."""
    heads, n, tokens = 3, 13, 64 * 9 + 5                    # block 9 ends in padding, blocks 10-12 are padding
    rows = [[9, 0, 12, 5], [12, 11, 3], [10, 9], [9, 9, 2], [12], [11, 9, 10, 4, 9], [0, 9]] + [[9 + i, i] for i in range(4)] + [[8], [9]]
    rows = [list(range(n))] + rows[:n - 2] + [list(range(n - 1, -1, -1))]
    assert len(rows) == n
    gen = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(64 * n, heads, 64, generator=gen).half() for _ in range(3))
    qs = (q.float() * (lh.LOG2E / 8)).half()
    sb = capi.seq_prefix_blocks([64 * n])
    idx = torch.tensor([b for r in rows for b in r], dtype=torch.int32)
    pos = torch.tensor([0] + [sum(len(r) for r in rows[:i + 1]) for i in range(n)], dtype=torch.int32)
    out = torch.full((64 * n, heads * 64), float("nan"), dtype=torch.float16, device="cuda")
    pack = lambda x, tr=False: lh.pack_heads(x, sb, transpose_v=tr).cuda()
    capi.bs_attention_fwd(pack(qs), pack(k), pack(v, True), out, torch.from_numpy(sb).cuda(), heads, idx.cuda(), pos.cuda(), 1,
                          seq_tokens_dev=torch.tensor([tokens], dtype=torch.int32).cuda())
    ref = oa.csr_attention(qs, k, v, sb.tolist(), idx.numpy(), pos.numpy(), 1, scale=1.0 / lh.LOG2E, seq_tokens=[tokens])
    empty = [i for i, r in enumerate(rows) if all(b > 9 for b in r)]          # no real key: zeros
    got = out.float().cpu()
    for i in range(n):
        sel = slice(64 * i, 64 * i + 64)
        if i in empty:
            assert (got[sel] == 0).all()
        else:
            assert lh.excess(got[sel], ref[sel], torch.float16) <= 0, i
