"""Block-sparse attention in fp32, whose products run on three bf16 parts of every operand: sizes at the edges of a tile's
halves and of the order in which rows are handed out, against the oracle to fp32's accuracy, and infinities, which the
parts cannot carry."""
import math

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
    (3, [64] * 70 + [192, 64, 448, 128], None, 1.0),            # more sequences than a wave looks up at a time, most of one row
    (1, [256, 64] * 64 + [320], [256 - i for i in range(128)] + [300], 1.0),
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


def attention64(qs, k, v, sb, idx, pos):
    """In float64 from the prepared queries (base-2 scores), heads' own plans: [T, H, 64]."""
    t, heads, _ = qs.shape
    nb, out = int(sb[-1]), torch.empty(t, heads, 64, dtype=torch.float64, device=qs.device)
    for s in range(len(sb) - 1):
        g0, n = int(sb[s]), int(sb[s + 1] - sb[s])
        rows = slice(g0 * 64, (g0 + n) * 64)
        for h in range(heads):
            times = torch.zeros(n, n, dtype=torch.float64)             # how often a row lists a block
            for i in range(n):
                for j in idx[pos[h * nb + g0 + i]:pos[h * nb + g0 + i + 1]]:
                    times[i, j] += 1
            w = times.to(qs.device).repeat_interleave(64, 0).repeat_interleave(64, 1)
            score = (qs[rows, h].double() @ k[rows, h].double().t()) * math.log(2.0)
            score = score.masked_fill(w == 0, -math.inf)
            p = torch.exp(score - score.amax(dim=1, keepdim=True)) * w
            out[rows, h] = (p @ v[rows, h].double()) / p.sum(dim=1, keepdim=True)
    return out


ONES = 1 + 2.0 ** -7 - 2.0 ** -19          # low bits all ones: what the products leave out is at its largest if parts are truncated
INPUTS = {
    "flat": lambda r, sign, power: (0.1 * r(), r(), r()),
    "normal": lambda r, sign, power: (r(), r(), r()),
    "peaked": lambda r, sign, power: (10 * r(), r(), r()),
    "positive": lambda r, sign, power: (r().abs(), r().abs(), r().abs()),
    "large mean": lambda r, sign, power: (r() + 4, r() + 4, r() + 4),
    "ones": lambda r, sign, power: (2 * sign() * ONES, sign() * ONES, sign() * ONES),
    "ones of many sizes": lambda r, sign, power: (sign() * power() * ONES, sign() * power() * ONES, sign() * power() * ONES),
    "tiny values": lambda r, sign, power: (r(), r(), r() * 2.0 ** -118),
    "tiny queries": lambda r, sign, power: (r() * 2.0 ** -120, r() * 2.0 ** 120, r()),
    "huge queries": lambda r, sign, power: (r() * 2.0 ** 120, r() * 2.0 ** -120, r()),
}


@pytest.mark.parametrize("kind", list(INPUTS))
@pytest.mark.parametrize("lens", [[64], [768, 2560]])
def test_fp32_attention_is_no_further_off_than_fp32_instructions(capi, kind, lens):
    """The products of parts against float64, beside the kernel on fp32 matrix instructions, which takes over the units
    that meet an infinity: here by one value in the last column, whose products touch no other column.  Sums of the same
    terms, in steps of 32 instead of 4, so no larger an error in the 2-norm (measured: 0.4 to 0.65 of it).  With any one of
    the six products left out, "normal" is 3.4e-6 off or more (worked out in float64), seven times what the bound allows."""
    print("fp32 attention error", kind, lens, flush=True)
    heads = 4
    g = torch.Generator(device="cuda").manual_seed(5)
    sb, idx, pos, ph, sb_d, idx_d, pos_d = lh.device_plan(capi, lens, heads, 3)
    r = lambda: torch.randn(sum(lens), heads, 64, generator=g, device="cuda")
    q, k, v = INPUTS[kind](r, lambda: torch.where(r() > 0, 1.0, -1.0), lambda: torch.exp2(torch.round(r())))
    # a power of two for the scale where the mantissas are to stay
    q = q * (0.125 if kind.startswith("ones") else lh.LOG2E / 8)
    want = attention64(q, k, v, sb, idx, pos)[..., :63]
    size = want.norm()

    def error(values):
        out = torch.full((sum(lens), heads * 64), float("nan"), device="cuda")
        capi.bs_attention_fwd(lh.pack_heads(q, sb), lh.pack_heads(k, sb), lh.pack_heads(values, sb, transpose_v=True), out, sb_d,
                              heads, idx_d, pos_d, ph)
        out = out.view(sum(lens), heads, 64)
        return out[..., 63], ((out[..., :63].double() - want).norm() / size).item()

    _, parts = error(v)
    first = [int(b) * 64 for b in sb[:-1]]                 # a key that every row of its sequence lists
    v[first, :, 63] = float("inf")
    last, plain = error(v)
    assert not bool(last.isfinite().any())
    print("  error %.2e, on fp32 instructions %.2e" % (parts, plain), flush=True)
    assert parts <= plain < 3e-6
