"""rt_bs_attention_fwd_no_alloc: the oracle's outputs, the bits of rt_bs_attention_fwd_masked (which is the same launch: what
differs is the limits that it states), no device memory taken by its launches, calls that overlap on two streams, and sizes
beyond the stated limits refused."""
import pytest
import torch

import __graft_entry__ as graft
from oracle import attention as oa
from tests import layer_harness as lh

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    pkg = graft.load_package()
    pkg.capi.lib()
    assert torch.cuda.is_available()
    return pkg.capi


def _case(capi, dtype, seq_lens, heads, seed, padded):
    t, dm = sum(seq_lens), heads * 64
    g = torch.Generator().manual_seed(seed)
    qkv = torch.randn(t, 3 * dm, generator=g).to(dtype).cuda()
    bias = (torch.randn(3 * dm, generator=g) * 0.5).to(dtype).cuda()
    sb, idx, pos, ph, sb_d, idx_d, pos_d = lh.device_plan(capi, seq_lens, heads, seed, None, max_pos=max(4096, max(seq_lens)))
    seq_tokens = [n - 9 for n in seq_lens] if padded else None
    tok_d = None if seq_tokens is None else torch.tensor(seq_tokens, dtype=torch.int32).cuda()
    q, k, vt = (torch.full((t * dm,), float("nan"), dtype=dtype, device="cuda") for _ in range(3))
    capi.qkv_bias_split(qkv, bias, q, k, vt, sb_d, heads, capi.Q_SCALE)
    x = qkv.float().cpu() + bias.float().cpu()
    qs = (x[:, :dm] * capi.Q_SCALE).to(dtype).view(t, heads, 64)
    kk, vv = (x[:, i * dm:(i + 1) * dm].to(dtype).view(t, heads, 64) for i in (1, 2))
    ref = oa.csr_attention(qs, kk, vv, sb.tolist(), idx, pos, ph, scale=1.0 / lh.LOG2E, seq_tokens=seq_tokens)
    return dict(t=t, dm=dm, q=q, k=k, vt=vt, sb_d=sb_d, idx_d=idx_d, pos_d=pos_d, ph=ph, tok_d=tok_d, heads=heads,
                ref=ref, dtype=dtype)


def _out(c):
    return torch.full((c["t"], c["dm"]), float("nan"), dtype=c["dtype"], device="cuda")


def _run(capi, c, no_alloc, out=None):
    out = _out(c) if out is None else out
    if no_alloc:
        capi.bs_attention_fwd_no_alloc(c["q"], c["k"], c["vt"], out, c["sb_d"], c["heads"], c["idx_d"], c["pos_d"],
                                       c["ph"], c["tok_d"])
    else:
        capi.bs_attention_fwd(c["q"], c["k"], c["vt"], out, c["sb_d"], c["heads"], c["idx_d"], c["pos_d"], c["ph"],
                              None, None, c["tok_d"])
    return out


# a batch for every cut of the rows, and more sequences than lanes
SHAPES = [([64 * 13, 64], 3), ([64 * 26], 10), ([64 * 21, 64 * 3, 64 * 40, 64, 64 * 12], 6), ([64 * 80, 128], 6), ([64 * 12] + [64] * 64, 2)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_no_alloc_entry_point_against_the_oracle(capi, dtype):
    """Launches take no device memory (behind the first of each kernel, for which the runtime takes some of its own)."""
    cases = [_case(capi, dtype, lens, heads, 11 + i, padded) for i, (lens, heads) in enumerate(SHAPES) for padded in (False, True)]
    outs = [_out(c) for c in cases]
    for c, out in zip(cases, outs):
        print("no_alloc", dtype, c["t"], c["heads"], c["tok_d"] is not None, flush=True)
        _run(capi, c, True, out)
    torch.cuda.synchronize()
    free, _ = torch.cuda.mem_get_info()
    for _ in range(20):
        for c, out in zip(cases, outs):
            _run(capi, c, True, out)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free
    for c, out in zip(cases, outs):
        assert torch.equal(_run(capi, c, False), out)
        assert (out.float().cpu() - c["ref"]).abs().max().item() <= 2e-2


def test_no_alloc_calls_overlap_on_two_streams(capi):
    """Nothing is shared between launches: two streams, a hundred calls each, every output with the bits of a call by itself."""
    print("no_alloc two streams", flush=True)
    cases = [_case(capi, torch.float16, lens, heads, 5, False) for lens, heads in (SHAPES[2], SHAPES[0])]
    want = [_run(capi, c, True) for c in cases]
    outs = [[_out(c) for _ in range(100)] for c in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in cases]
    for i in range(100):
        for c, st, out in zip(cases, streams, outs):
            with torch.cuda.stream(st):
                _run(capi, c, True, out[i])
    torch.cuda.synchronize()
    for w, out in zip(want, outs):
        assert all(torch.equal(o, w) for o in out)


def test_no_alloc_entry_point_refuses_sizes_beyond_its_limits(capi):
    print("no_alloc limits", flush=True)
    z = torch.zeros(64, 64, dtype=torch.float16, device="cuda")
    i32 = torch.zeros(8, dtype=torch.int32, device="cuda")
    L, vp = capi.lib(), capi._dp
    args = lambda batch, blocks: (vp(z), vp(z), vp(z), vp(z), vp(i32), None, batch, blocks, 1, vp(i32), vp(i32), 1,
                                  capi.RT_F16, None)
    assert L.rt_bs_attention_fwd_no_alloc(*args(1025, 1025)) == capi.RT_EINVAL
    assert b"at most" in L.rt_last_error_string()
    assert L.rt_bs_attention_fwd_no_alloc(*args(1, 4097)) == capi.RT_EINVAL
    assert L.rt_bs_attention_fwd_no_alloc(*args(0, 1)) == capi.RT_EINVAL
