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


# Tiles that rt_gemm_bt runs these on without and with GELU (None: the library)
EDGES = [
    (12288, 256, 128, torch.float16, "96x64 96x64"),        # whole tiles, the shortest reduction
    (12295, 264, 192, torch.bfloat16, "128x64 128x64"),     # odd number of steps; 8 columns and 7 rows in tiles of their own
    (9409, 520, 768, torch.float16, "128x192 128x192"),
    (16384 + 33, 1000, 256, torch.bfloat16, "192x128 192x128"),
    # More tiles than workgroups with the shortest reductions: a tile's first step is followed by its last (two steps, loads
    # reach into the tile after the next) or by one more (three); one row, 8 columns in the last tiles
    (8065, 2312, 128, torch.float16, "192x256 192x256"),
    (16353, 2304, 128, torch.bfloat16, "192x256 224x256"),
    (12289, 2312, 128, torch.float16, "192x256 192x256"),
    (8065, 2312, 192, torch.bfloat16, "192x256 192x256"),
    (12321, 3080, 192, torch.float16, "224x256 224x256"),
    (32641, 1288, 128, torch.float16, "192x256 256x256"),   # the last panel's lower half has one row
    (19969, 1288, 192, torch.bfloat16, "256x256 256x256"),
    (1, 8, 128, torch.float16, "96x64 96x64"),              # one row, one chunk of columns
    (64, 768, 3072, torch.bfloat16, "None None"),           # a long reduction with few outputs
    (333, 776, 768, torch.float16, "64x64 64x64"),
    (64, 5120, 1280, torch.bfloat16, "64x64 64x64"),
    (700, 2312, 192, torch.float16, "128x64 128x64"),
    (1500, 2304, 768, torch.bfloat16, "128x128 128x64"),
    (2049, 3080, 320, torch.float16, "128x256 128x256"),
    (5600, 768, 1024, torch.bfloat16, "192x128 192x128"),
]


def tile_name(capi, m, n, k, kind):
    tile = capi.gemm_bt_tile(m, n, k, kind)
    return "None" if tile is None else "%dx%d" % tile[:2]


@pytest.mark.parametrize("m,n,k,dtype,tiles", EDGES)
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_gemm_bt_edges(capi, m, n, k, dtype, tiles, epilogue):
    print("gemm_bt", m, n, k, dtype, epilogue, flush=True)
    assert tile_name(capi, m, n, k, epilogue) == tiles.split()[epilogue == 2]
    a, b, bias = operands(m, n, k, dtype)
    c = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
    capi.Gemm().bt(a, b, c[:m], bias=bias if epilogue else None, epilogue=epilogue)
    check(c[:m], a, b, bias if epilogue else None, epilogue == 2, dtype)
    assert bool((c[m] == 7.0).all())                   # nothing past the last row


# One row in the last panel and 8 columns in the last tile of every kernel (the model's choice for the shape), with as many
# steps as its stages hold, fewer, and more, in odd and even number.
TILES = {
    "64x64": [(2433, 776, 128), (2433, 776, 192), (65, 72, 256), (65, 72, 320), (513, 520, 704)],            # four stages
    "96x64": [(1, 8, 128), (97, 72, 128), (9217, 72, 192), (9217, 72, 256), (9217, 72, 320)],                # three
    "128x64": [(12289, 72, 128), (12289, 72, 192), (12289, 72, 256), (12289, 72, 448)],                      # three
    "128x128": [(1537, 1928, 768), (1537, 1928, 832)],                                                       # four
    "192x128": [(2305, 1672, 128), (2305, 1672, 192), (2305, 1672, 256), (2305, 1672, 320)],                 # three
    "128x192": [(7297, 520, 192), (7297, 520, 256), (7297, 520, 320)],                                       # three
    "128x256": [(2049, 3080, 128), (2049, 3080, 192), (2049, 3080, 256), (2049, 3080, 448)],                 # three
    "192x192": [(4609, 1736, 128), (4609, 1544, 192), (4609, 1544, 256), (4609, 1544, 320)],                 # three
    "192x256": [(8065, 2312, 128)],                                                                          # two rounds
    "224x256": [(3585, 3336, 128), (16577, 1288, 128)],                                                      # one round and two
    "256x256": [(8193, 1544, 128), (19969, 1288, 192)],                                                      # one round and two
}


@pytest.mark.parametrize("m,n,k,tile", [shape + (tile,) for tile, shapes in TILES.items() for shape in shapes])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gemm_bt_every_tile(capi, m, n, k, tile, dtype):
    print("gemm_bt tile", m, n, k, tile, dtype, flush=True)
    assert tile_name(capi, m, n, k, 2 if dtype == torch.float16 else 1) == tile
    a, b, bias = operands(m, n, k, dtype, seed=4)
    c = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
    gelu = dtype == torch.float16
    capi.Gemm().bt(a, b, c[:m], bias=bias, epilogue=2 if gelu else 1)
    check(c[:m], a, b, bias, gelu, dtype)
    assert bool((c[m] == 7.0).all())


@pytest.mark.parametrize("m,n,k,own", [
    (64, 768, 1536, True), (64, 768, 1600, False), (1, 256, 16384, False), (1, 4096, 4096, False), (1, 4104, 4096, True),
    (512, 512, 1536, True), (512, 512, 3072, False), (513, 512, 3072, True),
])
@pytest.mark.parametrize("epilogue", [0, 2])
def test_long_reductions_with_few_outputs_go_to_the_library(capi, m, n, k, own, epilogue):
    """They are slower as one chain of steps.  Which way a product went shows in the pair of events that the next launch
    of the own kernels takes and a product of the library leaves waiting."""
    print("gemm_bt route", m, n, k, epilogue, flush=True)
    a, b, bias = operands(m, n, k, torch.float16)
    c = torch.empty(m, n, dtype=torch.float16, device="cuda")
    gemm = capi.Gemm()
    gemm.set_tuning(1)
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for e in (start, stop):
        e.record()                                     # the handles exist from here on
    assert capi.time_next_launch(start.cuda_event, stop.cuda_event) == 0
    gemm.bt(a, b, c, bias=bias if epilogue else None, epilogue=epilogue)
    assert capi.time_next_launch(None, None) == (0 if own else 1)
    check(c, a, b, bias if epilogue else None, epilogue == 2, torch.float16)


QKV_CASES = [
    (12, [832, 64, 3008, 1024], torch.float16, "192x256"),
    (5, [64] * 70 + [2048], torch.bfloat16, "128x256"),     # more sequences than one wave looks up at a time, K and V halves of a tile
    (16, [4096, 320], torch.float16, "224x256"),
    (2, [64], torch.float16, "64x64"),
    (12, [192, 320], torch.bfloat16, "128x64"),
    (2, [192], torch.bfloat16, "64x64"),
    (3, [64, 256], torch.float16, "64x64"),
    (3, [2112], torch.bfloat16, "128x64"),                  # the last panel half full
    (9, [1216], torch.float16, "128x128"),                  # the same, and columns past the end
    (7, [3136], torch.bfloat16, "128x256"),                 # the same
    (7, [960, 576], torch.float16, "128x64"),               # 252 of 256 workgroups
    (7, [960, 640], torch.float16, "128x128"),
    (12, [2048, 1088], torch.bfloat16, "128x256"),
    # More tiles than workgroups, so that a tile is followed by another one, where some waves store nothing of it:
    (6, [14464], torch.float16, "192x256"),                 # columns past the end, and a last panel with its lower half past the end
    (10, [4096, 4096, 4160], torch.bfloat16, "224x256"),    # the same
    (6, [22976], torch.bfloat16, "256x256"),                # columns past the end
    (24, [3712], torch.float16, "192x256"),                 # rows past the end only
    (24, [4096, 2368], torch.bfloat16, "256x256"),          # the same
]


@pytest.mark.parametrize("heads,seq_lens,dtype,tile", QKV_CASES)
def test_qkv_project_equals_gemm_and_split(capi, heads, seq_lens, dtype, tile):
    print("qkv_project", heads, len(seq_lens), dtype, flush=True)
    t, d = sum(seq_lens), heads * 64
    assert tile_name(capi, t, 3 * d, d, capi.RT_PRODUCT_QKV) == tile
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


SLICED = [
    (1, 256, 768, torch.float16, (64, 64, 2)),
    (64, 768, 3072, torch.bfloat16, (64, 64, 8)),
    (515, 768, 3072, torch.float16, (64, 64, 2)),
    (1500, 1024, 4096, torch.bfloat16, (96, 64, 2)),
    (2816, 768, 3072, torch.float16, (192, 128, 2)),
    (1000, 512, 448, torch.float16, None),                  # seven steps: not cut
    (1, 256, 2048, torch.bfloat16, (64, 64, 5)),            # slices of six and seven steps
    (1441, 512, 3136, torch.float16, (96, 64, 2)),          # 24 and 25
    (1025, 512, 3136, torch.bfloat16, (128, 64, 3)),        # 16 and 17, one row in the last panel
    (1025, 1024, 3136, torch.float16, (128, 128, 3)),
    (2881, 768, 3136, torch.bfloat16, (192, 128, 2)),
    (64, 320, 1280, torch.float16, None),                   # a width the slices' LayerNorm does not have
    (9000, 768, 768, torch.float16, None),                  # enough rows: not cut
]


@pytest.mark.parametrize("m,n,k,dtype,tile", SLICED)
def test_gemm_bt_layernorm(capi, m, n, k, dtype, tile):
    """rt_gemm_bt_slices + rt_slices_residual_layernorm against fp32.  The LayerNorm's input x is a sum of the product
    (error of an fp32 sum as in check(); uncut, the product is also rounded to the stored type), bias and residual; an
    error e of an element moves the output by at most e * gamma / std plus the shift of mean and variance by the row's
    errors, less than as much again."""
    print("gemm_bt_layernorm", m, n, k, dtype, flush=True)
    a, b, bias = operands(m, n, k, dtype, seed=2)
    g = torch.Generator(device="cuda").manual_seed(3)
    res, gamma, beta = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((m, n), (n,), (n,)))
    out = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
    slices = capi.Gemm().bt_layernorm(a, b, bias, res, gamma, beta, out[:m], 1e-5)
    assert capi.gemm_bt_tile(m, n, k, capi.RT_PRODUCT_SLICES) == tile and slices == (tile[2] if tile else 0)
    prod = a.float() @ b.float().t()
    err = 2.0 ** -23 * k * (a.float().abs() @ b.float().abs().t())
    if slices == 0:
        err = err + 2.0 ** -(BITS[dtype] + 1) * prod.abs()
    x = prod + bias.float() + res.float()
    std = (x.var(dim=1, unbiased=False, keepdim=True) + 1e-5).sqrt()
    want = (x - x.mean(dim=1, keepdim=True)) / std * gamma.float() + beta.float()
    ulp = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -14))) - BITS[dtype])
    row = err.amax(dim=1, keepdim=True) / std
    bound = 0.51 * ulp + row * (2 * gamma.float().abs() + (want - beta.float()).abs()) + 2.0 ** -18 * (want.abs() + 1)
    over = ((out[:m].float() - want).abs() - bound).max().item()
    assert over <= 0, over
    assert bool((out[m] == 7.0).all())


def test_every_tile_of_the_selection_is_met(capi):
    """The shapes above reach every tile that a product of up to 40 000 rows can run on, in each of its forms."""
    rows = [64 * r for r in range(1, 64)] + [1024 * r for r in range(4, 40)]
    def chosen(kind, shapes):
        return {capi.gemm_bt_tile(m, n, k, kind)[:2] for n, k in shapes for m in rows if capi.gemm_bt_tile(m, n, k, kind)}
    def name(tiles):
        return {"%dx%d" % t for t in tiles}
    wide = [(n, k) for n in (8, 72, 264, 520, 776, 1288, 1672, 2056, 2304, 3072, 3336, 4096) for k in (128, 192, 768, 1024, 3072)]
    assert name(chosen(capi.RT_EPILOGUE_NONE, wide) | chosen(capi.RT_EPILOGUE_BIAS_GELU, wide)) == set(TILES)
    heads = [(192 * h, 64 * h) for h in range(2, 25)]
    assert name(chosen(capi.RT_PRODUCT_QKV, heads)) == {c[3] for c in QKV_CASES}
    ends = [(n, k) for n in (256, 512, 768, 1024) for k in (256, 768, 1024, 3072, 4096)]
    assert chosen(capi.RT_PRODUCT_SLICES, ends) == {c[4][:2] for c in SLICED if c[4]}


@pytest.mark.parametrize("m,n,k", [
    (256, 768, 768), (512, 768, 768), (649, 768, 768), (659, 1024, 1024), (2048, 256, 768),      # uncut
    (1024, 768, 3072), (1000, 1024, 3072), (5646, 256, 2048), (4096, 1024, 5120),
    (64, 768, 3072), (2816, 768, 3072),                                                          # in slices
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_sums_reach_the_layernorm_in_fp32(capi, m, n, k, dtype):
    """Cut or not, a product of few outputs is not rounded to 16 bits on its way to the LayerNorm: the output is as far from
    64 bits as its own rounding (fp32 sums and the LayerNorm add less than 1e-2 of that: k * 2^-24 against 2^-9 or 2^-12 of
    the root mean square); one more rounding on the way would make it 1.11 to 1.2 times as far."""
    print("sums in fp32", m, n, k, dtype, flush=True)
    a, b, bias = operands(m, n, k, dtype, seed=7)
    g = torch.Generator(device="cuda").manual_seed(8)
    res, gamma, beta = (torch.randn(*s, generator=g, device="cuda").to(dtype) for s in ((m, n), (n,), (n,)))
    out = torch.empty(m, n, dtype=dtype, device="cuda")
    assert capi.Gemm().bt_layernorm(a, b, bias, res, gamma, beta, out, 1e-5) >= 1
    x = a.double() @ b.double().t() + bias.double() + res.double()
    want = torch.nn.functional.layer_norm(x, (n,), gamma.double(), beta.double(), 1e-5)
    far = (out.double() - want).norm().item()
    rounding = (want.to(dtype).double() - want).norm().item()
    assert far <= 1.02 * rounding, far / rounding


def test_cut_product_as_first_call_in_a_capture(capi):
    """A context's first product that is cut may be met inside a capture, which allows no allocation."""
    m, n, k = 512, 768, 3072
    a, b, bias = operands(m, n, k, torch.float16)
    residual, out, want = (torch.randn(m, n, device="cuda").half() for _ in range(3))
    args = (a, b, bias, residual, 1 + 0 * bias, 0 * bias)
    assert capi.Gemm().bt_layernorm(*args, want, 1e-5) > 1
    fresh, graph = capi.Gemm(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        fresh.bt_layernorm(*args, out, 1e-5)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("call,dtype", [("bt", torch.float32), ("plain", torch.float16), ("bias_gelu", torch.bfloat16)])
def test_library_product_as_first_call_in_a_capture(capi, call, dtype):
    """The same for the products left to the library: fp32, and B[K, N]."""
    m, n, k = 128, 192, 256
    a, bt, bias = operands(m, n, k, dtype, seed=4)
    b, out, want = bt.t().contiguous(), *(torch.empty(m, n, dtype=dtype, device="cuda") for _ in range(2))

    def run(gemm, c):
        if call == "bt":
            gemm.bt(a, bt, c)
        elif call == "plain":
            gemm(a, b, c)
        else:
            gemm.bias_act(a, b, bias, c)

    eager = capi.Gemm()
    eager.set_tuning(1)                                # as in a capture, where no candidate can be timed
    run(eager, want)
    fresh, graph = capi.Gemm(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        run(fresh, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        run(eager, want)
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def on_own_kernel(capi, call):
    """Runs the call and asserts that it launched a kernel of the library's own, which takes a waiting pair of events."""
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for e in (start, stop):
        e.record()
    assert capi.time_next_launch(start.cuda_event, stop.cuda_event) == 0
    call()
    assert capi.time_next_launch(None, None) == 0


# Both sides of the line between the own kernel and the library at its best (tuned for the shape): own up to 7 % behind it
@pytest.mark.parametrize("m,n,k,own", [
    (1024, 768, 3072, True), (704, 2304, 768, True), (1024, 2304, 768, True), (2048, 768, 768, True), (1024, 1024, 1536, True), (4096, 768, 768, True),
    (640, 768, 3072, False), (512, 2304, 768, False), (1024, 768, 768, False), (384, 1024, 4096, False), (256, 3072, 768, False),
    (2113, 3076, 96, False), (2048, 2304, 256, False),                   # short reductions
])
def test_f32_products_run_on_the_faster_of_kernel_and_library(capi, m, n, k, own):
    a, b, _ = operands(m, n, k, torch.float32, seed=10)
    c, gemm = torch.empty(m, n, device="cuda"), capi.Gemm()
    gemm.set_tuning(1)
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for e in (start, stop):
        e.record()
    assert capi.time_next_launch(start.cuda_event, stop.cuda_event) == 0
    gemm.bt(a, b, c)
    assert capi.time_next_launch(None, None) == (0 if own else 1)        # an own kernel takes the pair, the library leaves it
    check_f32(c, a, b, None, False)


def check_f32(got, a, b, bias, gelu):
    """Per element against 64 bits: a sum of k terms in fp32 in any order (k * 2^-24 * sum |a| |b|) of products that miss at most a
    2^-24th, bias and rounding; the GELU's slope (<= 1.13) and its fp32 exponential and reciprocal, as in check()."""
    a, b = a.double(), b.double()
    x = a @ b.t()
    err = 2.0 ** -24 * (a.shape[1] + 2) * (a.abs() @ b.abs().t())
    if bias is not None:
        x = x + bias.double()
        err = err + 2.0 ** -23 * x.abs()
    want = torch.nn.functional.gelu(x, approximate="tanh") if gelu else x
    over = ((got.double() - want).abs() - 1.13 * err - 2.0 ** -20 * x.abs() * gelu - 2.0 ** -24 * want.abs()).max().item()
    assert over <= 0, over


# Sizes that the own kernel takes (gemm_f32_pays): one row and one chunk of columns in the last tiles, runs of 32 steps that the
# waves share unevenly, eight waves (up to 256 tiles) and four.
F32_SIZES = [(1025, 900, 3104), (961, 964, 2080), (1857, 1028, 1056), (4097, 3076, 480)]


@pytest.mark.parametrize("m,n,k", F32_SIZES + [(1024, 960, 1536), (2049, 772, 1056)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_f32_products(capi, m, n, k, epilogue):
    print("gemm f32", m, n, k, epilogue, flush=True)
    a, b, bias = operands(m, n, k, torch.float32, seed=5)
    c = torch.full((m + 1, n), 7.0, device="cuda")
    on_own_kernel(capi, lambda: capi.Gemm().bt(a, b, c[:m], bias=bias if epilogue else None, epilogue=epilogue))
    check_f32(c[:m], a, b, bias if epilogue else None, epilogue == 2)
    assert bool((c[m] == 7.0).all())


@pytest.mark.parametrize("m,n,k", [F32_SIZES[0], F32_SIZES[2]])
@pytest.mark.parametrize("scale_a,scale_b", [
    (0, 0), (50, 60),
    (-105, 0), (0, -115), (-118, 110),                               # parts below 2^-126
    (-42, -50), (-55, -60), (-60, -60), (-30, -90),                  # products of parts and their sums below it
])
def test_f32_products_of_single_terms(capi, m, n, k, scale_a, scale_b):
    """Sums of one term and zeros: nothing but the parts of two numbers.  What is left out is at most 2^-24 (1 + 2^-10) of the term; of
    the six sums of parts, which the instruction cuts off, the last costs up to 2^-23 and the others, at most 2^-7 of the
    term, 2^-28.  The mantissas leave out the most: a first part short by almost 2^-8, a second one by almost 2^-17."""
    print("gemm f32 single terms", m, n, k, scale_a, scale_b, flush=True)
    i, j = torch.arange(m, device="cuda"), torch.arange(n, device="cuda")
    x = (1 + 2.0 ** -8 + 2.0 ** -7 - (1 + i % 397) * 2.0 ** -23) * torch.exp2(i % 5 - 2.0) * 2.0 ** scale_a
    y = (1 + 2.0 ** -8 - (1 + j % 389) * 2.0 ** -23) * torch.exp2(j % 3 - 1.0) * (1 - 2 * (j % 2)) * 2.0 ** scale_b
    a, b = torch.zeros(m, k, device="cuda"), y.float()[:, None].repeat(1, k).contiguous()
    a[i, i * 37 % k] = x.float()
    c = torch.empty(m, n, device="cuda")
    on_own_kernel(capi, lambda: capi.Gemm().bt(a, b, c))
    want = a.double().sum(1)[:, None] * y.float().double()
    # (a sum below 2^-126 is cut off at 2^-149)
    over = (((c.double() - want).abs() - 6 * 2.0 ** -149).clamp_min(0) / want.abs()).max().item()
    assert over <= 1.5 * 2.0 ** -23 * (1 + 2.0 ** -5), over * 2.0 ** 23


RANGE_CASES = ["ones", "tiny", "both tiny", "tiny and huge", "largest", "infinite", "zeros", "zero column"]


# whole tiles on eight waves; on eight and on four waves one row and 4 columns in the last tiles, runs of 32 steps that the
# waves share unevenly, and the other epilogues behind the second pass
@pytest.mark.parametrize("m,n,k,epilogue", [(1024, 960, 1536, 0)] + [size + (e,) for size, e in zip(F32_SIZES, (1, 2, 1, 2))])
@pytest.mark.parametrize("case", RANGE_CASES)
def test_f32_products_at_the_ends_of_the_range(capi, case, m, n, k, epilogue):
    """Operands that bf16 parts hold badly or not at all: as accurate as the fp32 instruction all the same."""
    print("gemm f32 range", case, m, n, k, epilogue, flush=True)
    a, b, bias = operands(m, n, k, torch.float32, seed=6)
    if case == "ones":                                 # every bit of the mantissa set
        a = torch.exp2(torch.floor(torch.log2(a.abs().clamp_min(1e-3)))) * (2 - 2.0 ** -23)
        b = torch.exp2(torch.floor(torch.log2(b.abs().clamp_min(1e-3)))) * (2 - 2.0 ** -23)
    elif case == "tiny":                               # third parts below 2^-126, results above it
        a, b = a * 2.0 ** -112, b * 2.0 ** 4
    elif case == "both tiny":                          # all parts above 2^-126, products of parts below
        a, b = a * 2.0 ** -55, b * 2.0 ** -60
    elif case == "tiny and huge":
        a, b = a * 2.0 ** -118, b * 2.0 ** 110
    elif case == "largest":                            # a first part that rounds up to infinity
        a[5, 7], b[:, 7] = torch.finfo(torch.float32).max, b[:, 7] * 2.0 ** -30
    elif case == "infinite":
        a[3, 1], a[70, 2], b[9, 4] = float("inf"), float("nan"), float("-inf")
    elif case == "zeros":
        a[64:200] = 0
    else:
        b[70] = 0
    c = torch.full((m + 1, n), 7.0, device="cuda")
    bias = bias if epilogue else None
    on_own_kernel(capi, lambda: capi.Gemm().bt(a, b, c[:m], bias=bias, epilogue=epilogue))
    assert bool((c[m] == 7.0).all())
    c = c[:m]
    if case == "infinite":
        want = a.double() @ b.double().t() + (bias.double() if epilogue else 0)
        want = torch.nn.functional.gelu(want, approximate="tanh") if epilogue == 2 else want
        assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c == float("inf"), want == float("inf"))
        rows, cols = torch.ones(m, dtype=torch.bool), torch.ones(n, dtype=torch.bool)
        rows[[3, 70]], cols[9] = False, False
        c, a, b = c[rows.cuda()][:, cols.cuda()], a[rows.cuda()], b[cols.cuda()]
        bias = bias[cols.cuda()] if epilogue else None
    check_f32(c, a, b, bias, epilogue == 2)
    if epilogue == 0 and case in ("zeros", "zero column"):
        assert bool(((c[64:200] if case == "zeros" else c[:, 70]) == 0).all())


@pytest.mark.parametrize("m,n,k", [F32_SIZES[0], F32_SIZES[2]])
def test_f32_rows_and_columns_stand_alone(capi, m, n, k):
    """A row's or column's bits do not depend on what else lies in its tile, whichever of the two instructions that takes."""
    print("gemm f32 alone", m, n, k, flush=True)
    a, b, _ = operands(m, n, k, torch.float32, seed=9)
    want = torch.empty(m, n, device="cuda")
    capi.Gemm().bt(a, b, want)
    rows, cols = torch.ones(m, dtype=torch.bool, device="cuda"), torch.ones(n, dtype=torch.bool, device="cuda")
    rows[[2, 20, 70, 90, 130, m - 1]], cols[[5, 40, 75, n - 1]] = False, False
    a[2], a[20], a[70, 3], a[90] = 0, a[20] * 2.0 ** -120, float("inf"), a[90] * 2.0 ** 100
    a[130, 1:], a[m - 1, 7] = 0, float("nan")
    b[5], b[40, 1], b[75], b[n - 1] = 0, float("nan"), b[75] * 2.0 ** -100, b[n - 1] * 2.0 ** 90
    got = torch.empty(m, n, device="cuda")
    on_own_kernel(capi, lambda: capi.Gemm().bt(a, b, got))
    assert torch.equal(got[rows][:, cols], want[rows][:, cols])
