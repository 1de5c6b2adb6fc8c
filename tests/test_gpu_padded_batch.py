"""Packing a padded batch and unpacking its rows on the GPU: the kernels against the same call on host tensors, which takes
the general way."""
import importlib

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import __graft_entry__ as graft

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ut():
    graft.load_package()
    return importlib.import_module("raptor_t_amd.util")


def mask_of(lens, width, dtype):
    return (torch.arange(width)[None, :] < torch.tensor(lens)[:, None]).to(dtype)


@pytest.mark.parametrize("lens,width", [([1], 1), ([64, 1, 63, 65], 65), ([130, 64, 1], 150), ([300, 256, 257, 1024], 1024),
                                        ([(7 * i) % 300 + 1 for i in range(300)], 301)])
@pytest.mark.parametrize("ids_dtype,mask_dtype,types_dtype", [(torch.int64, torch.int64, None), (torch.int32, torch.bool, torch.int64),
                                                              (torch.int64, torch.uint8, torch.int32), (torch.int32, torch.int32, torch.int32)])
@pytest.mark.parametrize("keep_width", [False, True])
def test_pack_equals_the_general_way(ut, lens, width, ids_dtype, mask_dtype, types_dtype, keep_width):
    gen = torch.Generator().manual_seed(width)
    wide = torch.randint(1, 50000, (len(lens), 2 * width), generator=gen).to(ids_dtype)
    ids = wide[:, width // 2:width // 2 + width]                     # rows further apart than they are long
    types = None if types_dtype is None else torch.randint(0, 2, (len(lens), width), generator=gen).to(types_dtype)
    mask = mask_of(lens, width, mask_dtype)
    want = ut.pack_padded_batch(ids, mask, types, keep_width=keep_width)
    got = ut.pack_padded_batch(wide.cuda()[:, width // 2:width // 2 + width], mask.cuda(), None if types is None else types.cuda(),
                               keep_width=keep_width)
    assert got["seq_lens"] == want["seq_lens"] and got["seq_tokens"] == want["seq_tokens"]
    for name in ("input_ids", "position_ids", "token_type_ids", "seq_tokens_tensor"):
        assert got[name].is_cuda and got[name].dtype == want[name].dtype and got[name].is_contiguous()
        assert torch.equal(got[name].cpu(), want[name]), name


@pytest.mark.parametrize("change", ["hole", "empty", "left", "values", "negative", "float", "transposed"])
def test_pack_odd_masks_as_the_general_way(ut, change):
    """What the general way refuses is refused, what it accepts gives the same batch."""
    ids = torch.arange(3 * 200).view(3, 200) + 1
    mask = mask_of([200, 100, 7], 200, torch.int64)
    if change == "hole":
        mask[1, 50] = 0
    elif change == "empty":
        mask[2] = 0
    elif change == "left":
        mask = mask.flip(1)
    elif change == "values":                        # the sum of the entries counts: 100 places hold a token, 2 more are claimed
        mask[1, :2] = 2
    elif change == "negative":                      # as many nonzero entries as their sum, the last of them there: accepted
        mask[1, :2] = torch.tensor([3, -1])
    elif change == "float":
        mask = mask.float()
    elif change == "transposed":
        ids = ids.t().contiguous().t()

    def call(i, m):
        try:
            return ut.pack_padded_batch(i, m)
        except ValueError as e:
            return str(e)
    want, got = call(ids, mask), call(ids.cuda() if change != "transposed" else ids.t().cuda().t(), mask.cuda())
    if isinstance(want, str):
        assert got == want
    else:
        assert got["seq_tokens"] == want["seq_tokens"] and torch.equal(got["input_ids"].cpu(), want["input_ids"])


@pytest.mark.parametrize("dtype", [torch.bool, torch.uint8, torch.int8, torch.int32, torch.int64])
def test_padded_tokens_counts_ones(dtype):
    """The entry point by itself: -1 for every row that holds other numbers than ones in front and zeros behind them."""
    capi = graft.load_package().capi
    rows = [[1] * 300, [0] * 300, [1] * 7 + [0] * 293, [0, 1] + [0] * 298, [1] * 256 + [0] + [1] * 43, [1] * 299 + [0]]
    want = [300, 0, 7, -1, -1, 299]
    if dtype != torch.bool:
        rows += [[2, 0] + [0] * 298, [1] * 100 + [0] * 199 + [2]]
        want += [-1, -1]
    if dtype in (torch.int8, torch.int32, torch.int64):
        rows += [[3, -1, 1, 0] + [0] * 296, [-1] * 300, [2, 0] + [1] * 298]
        want += [-1, -1, -1]
    if dtype == torch.int64:
        rows += [[1 << 32] + [0] * 299, [(1 << 32) + 1] + [0] * 299]
        want += [-1, -1]
    tokens = torch.full((len(rows),), -7, dtype=torch.int32, device="cuda")
    capi.padded_tokens(torch.tensor(rows).to(dtype).cuda(), tokens)
    assert tokens.tolist() == want


@pytest.mark.parametrize("lens,width", [([1], 1), ([64, 1, 63, 65], 65), ([130, 64, 1], 150), ([0, 5, 0], 9), ([700, 3], 1100),
                                        ([(7 * i) % 30 + 1 for i in range(300)], 31)])
@pytest.mark.parametrize("cols,dtype", [(8, torch.float16), (768, torch.bfloat16), (12, torch.float32), (3, torch.float32), (1024, torch.float32)])
def test_unpack_equals_the_general_way(ut, lens, width, cols, dtype):
    """Rows of one vector and of many, of whole vectors and not (3 columns: the general way), several launches (300 sequences),
    sequences without a row."""
    seq_lens = [-(-n // 64) * 64 for n in lens]
    packed = torch.randn(max(1, sum(seq_lens)), cols, generator=torch.Generator().manual_seed(cols)).to(dtype)
    want = ut.unpack_to_padded(packed, seq_lens, lens, width)
    torch.empty(want.shape, dtype=dtype, device="cuda").fill_(float("nan"))      # what the allocator hands out next is not zeros
    got = ut.unpack_to_padded(packed.cuda(), seq_lens, lens, width)
    assert got.dtype == dtype and torch.equal(got.cpu(), want)


@pytest.mark.parametrize("seq_lens,tokens,width", [([64, 64], [64, 65], 100), ([64, 64], [64, 64], 60), ([64], [64], 64.0)])
def test_unpack_refuses_what_the_general_way_refuses(ut, seq_lens, tokens, width):
    packed = torch.zeros(128 if len(seq_lens) > 1 else 64, 8, dtype=torch.float16, device="cuda")
    with pytest.raises((RuntimeError, TypeError)):
        ut.unpack_to_padded(packed, seq_lens, tokens, width)


class SeenByDispatch(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen += 1
        return func(*args, **(kwargs or {}))


class SeenByFunction(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = 0

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen += func is torch.Tensor.__setitem__
        return func(*args, **(kwargs or {}))


def test_unpack_traced_is_the_whole_computation(ut):
    """What a tracer records, run on other rows, gives their padded batch; the same for a compiled call in one graph."""
    seq_lens, tokens, width = [128, 64, 64], [70, 64, 1], 100
    rows = [torch.randn(256, 8, generator=torch.Generator().manual_seed(i)).half() for i in range(2)]
    call = lambda x: ut.unpack_to_padded(x, seq_lens, tokens, width)
    torch.empty(3, width, 8, dtype=torch.float16, device="cuda").fill_(float("nan"))
    graphs = [make_fx(call)(rows[0].cuda()), make_fx(call, pre_dispatch=True)(rows[0].cuda()), torch.jit.trace(call, rows[0].cuda()),
              torch.compile(call, backend="eager", fullgraph=True)]
    for graph in graphs:
        assert torch.equal(graph(rows[1].cuda()).cpu(), call(rows[1]))


@pytest.mark.parametrize("mode", [SeenByDispatch, SeenByFunction])
def test_modes_see_the_operators(ut, mode):
    packed = torch.randn(128, 8, device="cuda").half()
    ids, mask = torch.arange(120, device="cuda").view(2, 60), mask_of([60, 3], 60, torch.int64).cuda()
    with mode() as m:
        out = ut.unpack_to_padded(packed, [64, 64], [60, 3], 64)
        unpacked = m.seen
        batch = ut.pack_padded_batch(ids, mask)
    assert unpacked >= 2 and (mode is SeenByFunction or m.seen > unpacked + 2)
    assert torch.equal(out, ut.unpack_to_padded(packed, [64, 64], [60, 3], 64))
    assert torch.equal(batch["input_ids"], ut.pack_padded_batch(ids, mask)["input_ids"])


def test_default_device_is_no_mode(ut):
    with torch.device("cuda"):
        assert not ut._watched()


@pytest.mark.parametrize("lazy", ["conj", "neg", "zero"])
def test_unpack_of_lazy_tensors(ut, lazy):
    x = torch.randn(128, 8, dtype=torch.complex64 if lazy == "conj" else torch.float32)
    make = {"conj": lambda t: t.conj(), "neg": torch._neg_view, "zero": lambda t: torch._efficientzerotensor(t.shape, device=t.device)}[lazy]
    got = ut.unpack_to_padded(make(x.cuda()), [64, 64], [64, 5], 70)
    assert torch.equal(got.cpu().resolve_conj().resolve_neg(), ut.unpack_to_padded(make(x), [64, 64], [64, 5], 70).resolve_conj().resolve_neg())


def test_unpack_takes_any_iterable_of_counts(ut):
    packed = torch.randn(128, 8)
    want = ut.unpack_to_padded(packed, [64, 64], [64, 5], 70)
    for tokens in (iter([64, 5]), (n for n in (64, 5)), torch.tensor([64, 5]), [64, 5, 9]):
        assert torch.equal(ut.unpack_to_padded(packed.cuda(), [64, 64], tokens, 70).cpu(), want)
