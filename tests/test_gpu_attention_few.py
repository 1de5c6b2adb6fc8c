"""Block-sparse attention of batches with few units, whose rows several waves share: every cut of a row, padding, scores that
outgrow the pipelined loop's reference, infinities, and the caller's plan, against the oracle.  Each case states the cut it is
meant for (shares of a row, of a global row, waves of a workgroup) and asks the library for it."""
import numpy as np
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


def cut_of(capi, heads, lens):
    return capi.bs_attention_cut(len(lens), sum(lens) // 64, heads)


@pytest.mark.parametrize("cut,heads,lens,scale", [
    ((1, 4, 4), 1, [64], 1.0),                        # one row, one tile: three of the workgroup's waves have no row
    ((4, 4, 4), 12, [512], 1.0),
    ((4, 4, 4), 3, [704, 768, 64], 1.0),              # sequences of 11 and 12 blocks: the last without and the first with global rows
    ((1, 4, 4), 12, [1024, 1088], 1.0),               # two workgroups too many for two waves to a row
    ((2, 4, 4), 12, [1024, 1024], 1.0),
    ((4, 4, 4), 5, [2048, 832, 64], 40.0),            # scores beyond the pipelined loop's range
    ((2, 4, 4), 10, [1664, 512], 40.0),
    ((1, 8, 8), 6, [5760], 40.0),
    ((1, 4, 4), 12, [256, 1024, 640, 896], 1.0),
    ((1, 4, 4), 12, [2048, 3008, 384], 1.0),
    ((1, 4, 4), 12, [2944, 3008, 2752], 1.0),
    ((1, 4, 4), 12, [4096, 2624, 1984], 40.0),
    ((1, 4, 4), 12, [4160, 2560, 1984], 1.0),
    ((1, 8, 8), 12, [1920] * 3, 1.0),                 # even sequences, one round of workgroups of eight waves
    ((1, 4, 4), 2, [64] * 64, 1.0),                   # as many sequences as lanes
    ((1, 4, 4), 2, [64] * 64 + [128], 1.0),           # one more
    ((1, 8, 8), 8, [4096 * 4], 1.0),                  # global rows of 256 tiles
    ((1, 8, 8), 11, [64 * 128, 64 * 128], 6.0),       # several rounds, and chains that outlast them
])
@pytest.mark.parametrize("padded", [False, True])
def test_few_units(capi, cut, heads, lens, scale, padded):
    print("few units", cut, heads, lens[:4], scale, padded, flush=True)
    assert cut_of(capi, heads, lens) == cut
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


@pytest.mark.parametrize("cut,heads,lens,scale", [
    ((4, 4, 4), 2, [512], 1.0),                       # a unit in 4 shares: one to each of the workgroup's four waves
    ((4, 4, 4), 2, [512], 40.0),                      # the same with scores beyond the pipelined loop's range
    ((2, 4, 4), 12, [1536, 512], 1.0),                # 2: two units side by side
    ((2, 4, 4), 10, [1664], 40.0),
    ((1, 4, 4), 12, [1024, 1088], 1.0),               # 1: four
    ((1, 4, 4), 12, [256, 1024, 640, 896], 1.0),
    ((1, 4, 4), 12, [2048, 3008, 384], 6.0),
    ((1, 8, 8), 6, [5760], 1.0),                      # global rows in 8 shares: two to each wave
    ((1, 8, 8), 6, [5760], 40.0),
    ((1, 8, 8), 12, [4096], 6.0),
    ((1, 4, 4), 12, [2944, 3008, 2752], 6.0),
    ((2, 4, 4), 1, [64 * 257] + [640] * 8, 40.0),     # a sequence whose global rows have 8 shares all the same
])
@pytest.mark.parametrize("padded", [False, True])
def test_few_units_walk_the_plan(capi, cut, heads, lens, scale, padded):
    """Every workgroup walks the slice that the partition gives it, whatever its neighbours have: one slice with all units,
    more slices than units, and slices whose ends do not meet (the first is empty, the second begins before its end)."""
    print("plan walk", cut, heads, lens, scale, padded, flush=True)
    assert cut_of(capi, heads, lens) == cut
    g = torch.Generator(device="cuda").manual_seed(3)
    t = sum(lens)
    sb, _, _, ph, sb_d, idx_d, pos_d = lh.device_plan(capi, lens, heads, 3, max_pos=max(4096, max(lens)))
    q, k, v = (torch.randn(t, heads, 64, generator=g, device="cuda").half() for _ in range(3))
    operands = lh.pack_heads(q * (scale * lh.LOG2E / 8), sb), lh.pack_heads(k, sb), lh.pack_heads(v, sb, transpose_v=True)
    tokens = torch.tensor([max(1, n - 81 - 3 * i) for i, n in enumerate(lens)], dtype=torch.int32).cuda() if padded else None
    units = t // 64 * heads

    def run(*plan):
        out = torch.full((t, heads * 64), float("nan"), dtype=torch.float16, device="cuda")
        capi.bs_attention_fwd(*operands, out, sb_d, heads, idx_d, pos_d, ph, *plan, seq_tokens_dev=tokens)
        torch.cuda.synchronize()
        return out

    want = run(None, None)
    assert not bool(want.isnan().any())
    for n_wg in (1, 5, units + 3):
        fp, fi = capi.partition_lpt(sb, heads, n_wg)
        assert torch.equal(run(torch.from_numpy(fi).cuda(), torch.from_numpy(fp).cuda()), want), n_wg
    ids = torch.arange(units, dtype=torch.int32).cuda()
    ends = torch.tensor([units // 2, 0, units], dtype=torch.int32).cuda()
    assert torch.equal(run(ids, ends), want)


@pytest.mark.parametrize("cut,heads,lens,n_wg", [
    ((4, 4, 4), 2, [512], 0),                         # two tiles to a wave
    ((4, 4, 4), 2, [512], 5),
    ((4, 4, 4), 12, [1024, 256], 0),
    ((2, 4, 4), 12, [1536, 512], 0),
    ((2, 4, 4), 12, [1536, 512], 31),
    ((1, 4, 4), 12, [512, 1024, 1280], 0),
    ((1, 4, 4), 12, [2048, 3008, 384], 0),
    ((1, 4, 4), 12, [2944, 3008, 2752], 0),
    ((1, 4, 4), 12, [2944, 3008, 2752], 300),
    ((1, 8, 8), 6, [5120, 512], 0),
    ((1, 8, 8), 6, [5120, 512], 40),                  # two shares to a wave
    ((1, 8, 8), 2, [5120], 0),
    ((1, 4, 4), 16, [2048] * 6, 0),                   # 3072 units
    ((1, 4, 4), 2, [512] + [64] * 60 + [1024] * 5, 0),               # more sequences than lanes
    ((1, 4, 4), 2, [512] + [64] * 60 + [1024] * 5, 20),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_infinite_and_very_low_scores(capi, cut, heads, lens, n_wg, dtype):
    """Key blocks that a query scores with minus infinity throughout (first, in the middle, last in a wave's share),
    queries with no other keys, infinite and undefined values and, where the type reaches so far, rows whose scores
    all lie below -1e30: weights as a softmax over the whole row gives them."""
    print("infinities", cut, heads, lens[:4], n_wg, dtype, flush=True)
    assert cut_of(capi, heads, lens) == cut
    g = torch.Generator().manual_seed(1)
    t = sum(lens)
    q, k, v = (torch.randn(t, heads, 64, generator=g).to(dtype) for _ in range(3))
    inf = float("inf")
    for block in (0, 2, lens[0] // 64 - 1):
        k[64 * block:64 * block + 64, 0, 3] = inf      # by the sign of a query's element: no weight, or no number
    k[320, 1, 5] = inf
    v[400, 1, 7] = inf
    v[410, 1, 9] = float("nan")
    if dtype == torch.bfloat16:
        q[:64, 1] = q[:64, 1].abs()
        k[:lens[0], 1] = -2e35 * k[:lens[0], 1].abs().clamp_min(.1)
        k[lens[0]:, 0, 9] = inf                        # the later sequences' head 0: every key, zeros or NaN
    out, ref = lh.run_attention(capi, q.cuda(), k.cuda(), v.cuda(), lens, heads, seed=3, n_wg=n_wg, max_pos=max(4096, max(lens)))
    out = out.float().cpu()
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    ok = out.isfinite()                                # of the two heads with infinite keys half the queries, about
    assert int(out.isnan().sum()) > 0 and int(ok.sum()) > out.numel() // 4
    # weights and output rounded to the type (half a unit in the last place of values up to max |v| each)
    tol = 4 * (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) * v[v.isfinite()].abs().max().item()
    assert (out - ref)[ok].abs().max().item() <= tol


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,lens,short", [
    (3, [1024, 768, 64], 17),                         # few units; 64 tokens: every entry is the padded tile
    (4, [1024, 1600, 320], 63),                       # a tail of one key
    (12, [1024] * 15, 40),                            # 2880 units
    (12, [1024, 768] * 8, 150),                       # whole blocks of padding dropped in front of it
])
def test_padded_tile_listed_several_times(capi, heads, lens, short, dtype):
    """Every third entry of the plan becomes the block the real tokens end in: rows that list it up to a dozen times,
    first, last and as their only tile."""
    print("padded tile listed several times", heads, lens[:3], short, dtype, flush=True)
    g = torch.Generator().manual_seed(heads)
    t = sum(lens)
    tokens = [max(1, n - short) for n in lens]
    q, k, v = (torch.randn(t, heads, 64, generator=g).to(dtype).cuda() for _ in range(3))
    sb, idx, pos, ph, sb_d, _, pos_d = lh.device_plan(capi, lens, heads, 5, None)
    idx = idx.copy()
    rng = np.random.default_rng(heads)
    row, seen = 0, 0
    for h in range(ph):                               # rows of the index: head by head, sequence by sequence
        for n, real in zip(lens, tokens):
            for _ in range(n // 64):
                a, b = int(pos[row]), int(pos[row + 1])
                last = (real - 1) // 64
                idx[a:b] = np.where(rng.random(b - a) < 1 / 3, last, idx[a:b])
                if not (idx[a:b] <= last).any():
                    idx[a] = last                     # a row of padding alone has no softmax
                seen = max(seen, int((idx[a:b] == last).sum()))
                row += 1
    assert row == len(pos) - 1 and seen > 4
    qs = (q.float() * (lh.LOG2E / 8.0)).to(dtype)
    out = torch.empty(t, heads * 64, dtype=dtype, device="cuda")
    capi.bs_attention_fwd(lh.pack_heads(qs, sb), lh.pack_heads(k, sb), lh.pack_heads(v, sb, transpose_v=True), out, sb_d,
                          heads, torch.from_numpy(idx).cuda(), pos_d, ph, None, None,
                          torch.tensor(tokens, dtype=torch.int32).cuda())
    torch.cuda.synchronize()
    ref = lh.oa.csr_attention(qs.cpu(), k.cpu(), v.cpu(), sb.tolist(), idx, pos, ph, scale=1.0 / lh.LOG2E, seq_tokens=tokens)
    # as above, with the type's own unit roundoff
    tol = 4 * 2.0 ** -(lh.MANTISSA_BITS[dtype] + 1) * v.float().abs().max().item()
    start = 0
    for n, real in zip(lens, tokens):                 # real query rows only
        err = (out[start:start + real].float().cpu() - ref[start:start + real]).abs().max().item()
        assert err <= tol, (n, real, err)
        start += n
