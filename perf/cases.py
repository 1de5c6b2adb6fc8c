"""Measured cases of the block-sparse encoder: what a user of the framework has it do, through its public entry
points, from one short document to the large long-sequence batch.

Kinds of a case:
  encoder     BertEncoder.__call__ on a packed batch whose metadata is at hand (the benchmark's step): the batch is
              published to the index pipeline and every layer runs
  model       BertModel.__call__ on a padded batch of token ids, the whole serving call: packing, batch metadata,
              embeddings, encoder, pooling head, unpacking
  attention   the isolated block-sparse attention operator, with true token counts where `short` says so
  layernorm   the isolated bias + residual + LayerNorm operator, in place
  gelu        the isolated bias + GELU operator, in place
"""
import importlib
import math
import random

import numpy as np
import torch

import __graft_entry__ as graft

pkg = graft.load_package()
capi = pkg.capi
mb = importlib.import_module("raptor_t_amd.modeling_bert")
ut = importlib.import_module("raptor_t_amd.util")

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SIZE = {"f16": 2, "bf16": 2, "f32": 4}
PAIR_FLOP = 4 * 64 * 64 * 64              # scores and values of one (from-block, to-block) pair of a head
BLOCK_LIMIT = 1024                        # workgroups of the batch's work plan (the benchmark's default)
VOCAB, POSITIONS = 50358, 4096            # BigBird's tables, as the benchmark's embedding sweep has them

BASE = {"hidden": 768, "heads": 12, "ffn": 3072, "layers": 12, "positions": 4096}
LARGE = {"hidden": 1024, "heads": 16, "ffn": 4096, "layers": 24, "positions": 16384}


def _encoder(dtype, batch, lo, hi, lengths, shape=BASE, **more):
    return dict(shape, kind="encoder", dtype=dtype, batch=batch, lo=lo, hi=hi, lengths=lengths, **more)


def _model(dtype, batch, lo, hi, lengths, pooling):
    return dict(BASE, kind="model", dtype=dtype, batch=batch, lo=lo, hi=hi, lengths=lengths, pooling=pooling)


def _attention(dtype, batch, lo, hi, lengths, short, heads=12):
    return {"kind": "attention", "dtype": dtype, "batch": batch, "lo": lo, "hi": hi, "lengths": lengths, "short": short,
            "heads": heads, "positions": 4096}


def _rowwise(kind, dtype, rows, width):
    return {"kind": kind, "dtype": dtype, "rows": rows, "width": width}


def listed():
    return [
        # one short document at a time: an interactive request, where launches and latency count
        dict(_encoder("f16", 1, 512, 512, 0), name="base f16 1 x 512"),
        # a small batch of paragraphs, dense and sparse sequences mixed, in bfloat16
        dict(_encoder("bf16", 4, 256, 1024, 0), name="base bf16 4 x 256-1024"),
        # one document of the model's full length
        dict(_encoder("f16", 1, 4096, 4096, 0), name="base f16 1 x 4096"),
        # the headline workload: a full batch of documents of any length
        dict(_encoder("f16", 16, 512, 4096, 0), name="base f16 16 x 512-4096"),
        # the long-sequence stress: large model, books and long reports, bfloat16
        dict(_encoder("bf16", 4, 2048, 16384, 0, LARGE), name="large bf16 4 x 2048-16384"),
        # the accuracy mode: one layer in fp32
        dict(_encoder("f32", 1, 1024, 1024, 0, dict(BASE, layers=1)), name="layer f32 1 x 1024"),
        # a serving call on a padded batch of odd token counts, text in and one vector per text out
        dict(_model("f16", 8, 150, 1700, 0, "First"), name="model f16 padded 8 x 150-1700"),
        # the attention operator by itself, fixed length
        dict(_attention("f16", 8, 4096, 4096, 0, False), name="attention f16 8 x 4096"),
        # the attention operator on a ragged batch with padded tails
        dict(_attention("bf16", 5, 320, 3000, 0, True), name="attention bf16 padded 5 x 320-3000"),
        # the memory-bound operators over the range that the benchmark sweeps
        dict(_rowwise("layernorm", "bf16", 32768, 768), name="layernorm bf16 32768 x 768"),
        dict(_rowwise("gelu", "f16", 8192, 3072), name="gelu f16 8192 x 3072"),
    ]


def _between(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["encoder"] * 5 + ["large", "fp32", "model", "model", "attention", "attention", "layernorm", "gelu"])
    lengths = rng.randrange(1 << 20)
    half = rng.choice(["f16", "bf16"])
    if kind in ("encoder", "large", "fp32"):
        hi = 64 * _between(rng, 2, {"encoder": 64, "large": 192, "fp32": 32}[kind])
        lo = 64 * rng.randint(1, hi // 64)
        batch = _between(rng, 1, {"encoder": 16, "large": 4, "fp32": 4}[kind])
        if kind == "large":
            return _encoder("bf16", batch, lo, hi, lengths, LARGE)
        if kind == "fp32":
            return _encoder("f32", batch, lo, hi, lengths, dict(BASE, layers=1))
        return _encoder(half, batch, lo, hi, lengths)
    if kind == "model":
        hi = _between(rng, 70, 4096)
        return _model(half, _between(rng, 1, 16), max(1, hi // rng.randint(2, 12)), hi, lengths, rng.choice(["First", "Mean", "Max"]))
    if kind == "attention":
        hi = 64 * _between(rng, 2, 64)
        return _attention(half, _between(rng, 1, 16), 64 * rng.randint(1, hi // 64), hi, lengths, rng.random() < 0.5,
                          rng.choice([12, 16]))
    rows = _between(rng, 512, 65536)
    if kind == "layernorm":
        return _rowwise("layernorm", half, rows, rng.choice([768, 1024]))
    return _rowwise("gelu", half, rows, rng.choice([3072, 4096]))


# ---- sizes of a case ----------------------------------------------------------------------------------------
def _tokens(case):
    """True token count of every sequence: any number for a padded batch, whole blocks otherwise."""
    rng = np.random.default_rng(case["lengths"])
    lo, hi, n = case["lo"], case["hi"], case["batch"]
    if case["kind"] == "model" or case.get("short"):
        return [int(v) for v in rng.integers(lo, hi + 1, size=n)]
    return [int(v) for v in ut.uniform_lengths(n, lo, hi, seed=case["lengths"])]


def _packed(tokens):
    return [-(-n // 64) * 64 for n in tokens]


def _pairs(lens, heads):
    blocks = [n // 64 for n in lens]
    return heads * sum(n * n if n < 12 else 10 * n - 18 for n in blocks)


def work(case):
    size = SIZE[case["dtype"]]
    if case["kind"] in ("layernorm", "gelu"):
        n = case["rows"] * case["width"]
        return {"bytes": (3 if case["kind"] == "layernorm" else 2) * n * size, "flops": (10 if case["kind"] == "layernorm" else 12) * n}
    lens = _packed(_tokens(case))
    t = sum(lens)
    if case["kind"] == "attention":
        return {"bytes": 4 * t * case["heads"] * 64 * size, "flops": _pairs(lens, case["heads"]) * PAIR_FLOP}
    d, f = case["hidden"], case["ffn"]
    weights = case["layers"] * (4 * d * d + 2 * d * f)
    flops = 2 * t * weights + case["layers"] * _pairs(lens, case["heads"]) * PAIR_FLOP
    count = weights * size + 2 * t * d * size                          # weights, hidden states in, hidden states out
    if case["kind"] == "model":
        count += t * d * 4 + case["batch"] * max(_tokens(case)) * 16   # embedding rows (fp32), ids and mask
    return {"bytes": count, "flops": flops}


# Largest error of a 16-bit case, about four times the distance from the same path run in fp32 on the same rounded
# weights and inputs (2-norm, largest): a stack of 12 layers in f16 1.3e-3, 9e-3, in bf16 1.0e-2, 6e-2, 24 layers in
# bf16 1.3e-2, 8e-2; attention f16 3.6e-4, 3.4e-3, bf16 2.9e-3, 2.4e-2; LayerNorm bf16 2.4e-3, 8e-3; GELU f16 2.1e-4,
# 5e-4.  A layer in fp32 is 2.1e-7, 1.6e-6 from the same layer with its LayerNorms and GELU as library operators; the sums
# of its matrix products (up to 3072 terms) in another order move it by several times that.
TOLERANCE = {
    "encoder": {"f16": {"rel": 5e-3, "max": 4e-2}, "bf16": {"rel": 3e-2, "max": 3e-1}, "f32": {"rel": 1e-5, "max": 1e-4}},
    "model": {"f16": {"rel": 5e-3, "max": 4e-2}, "bf16": {"rel": 3e-2, "max": 3e-1}},
    "attention": {"f16": {"rel": 1.5e-3, "max": 1.4e-2}, "bf16": {"rel": 1.2e-2, "max": 1e-1}},
    "layernorm": {"f16": {"rel": 1.2e-3, "max": 4e-3}, "bf16": {"rel": 1e-2, "max": 3e-2}},
    "gelu": {"f16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 6.4e-3, "max": 1.6e-2}},
}


def tolerance(case):
    return dict(TOLERANCE[case["kind"]][case["dtype"]])


# ---- inputs --------------------------------------------------------------------------------------------------
_built = [None]


def _configure(case):
    """A program runs one model: where the case before had another, the index pipeline's workers of that one end."""
    key = (case["hidden"], case["heads"], case["layers"], case["dtype"], case["positions"])
    if _built[0] != key:
        mb.cxx.MetaData().terminate_thread()
        mb.cxx.MetaData.set_plan(capi.RT_PLAN_HF, capi.RT_POLICY_REFERENCE_PATCHED, case["positions"])
        _built[0] = key


def _layer_weights(d, f, dt, gen):
    """N(0, 0.02) weights and biases, LayerNorm gains near 1 and shifts near 0, [in, out]."""
    n = lambda *shape: (torch.randn(*shape, generator=gen, device="cuda") * 0.02).to(dt)
    one = lambda: (1.0 + 0.02 * torch.randn(d, generator=gen, device="cuda")).to(dt)
    return {"qkv_weight": n(d, 3 * d), "qkv_bias": n(3 * d), "attn_out_weight": n(d, d), "attn_out_bias": n(d),
            "attn_ln_weight": one(), "attn_ln_bias": n(d), "inter_weight": n(d, f), "inter_bias": n(f),
            "out_weight": n(f, d), "out_bias": n(d), "out_ln_weight": one(), "out_ln_bias": n(d)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    randn = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(dt)
    if case["kind"] == "layernorm":
        w = case["width"]
        return {"case": case, "out": randn(case["rows"], w), "residual": randn(case["rows"], w), "bias": randn(w) * 0.02,
                "gamma": 1.0 + 0.02 * randn(w), "beta": 0.02 * randn(w)}
    if case["kind"] == "gelu":
        return {"case": case, "out": randn(case["rows"], case["width"]), "bias": randn(case["width"]) * 0.02}
    tokens = _tokens(case)
    lens = _packed(tokens)
    t = sum(lens)
    if case["kind"] == "attention":
        heads = case["heads"]
        sb = capi.seq_prefix_blocks(lens)
        idx, pos = capi.build_to_index(sb, heads, seed=seed % 97, max_pos=case["positions"])
        up = lambda a: torch.from_numpy(a).cuda()
        state = {"case": case, "seq_blocks": up(sb), "idx": up(idx), "pos": up(pos),
                 "out": torch.empty(t, heads * 64, dtype=dt, device="cuda"),
                 "tokens": up(np.asarray(tokens, dtype=np.int32)) if case["short"] else None}
        q, k, vt = (torch.empty(t * heads * 64, dtype=dt, device="cuda") for _ in range(3))
        capi.qkv_bias_split(randn(t, 3 * heads * 64), None, q, k, vt, state["seq_blocks"], heads, capi.Q_SCALE)
        return dict(state, q=q, k=k, vt=vt)

    _configure(case)
    d, f = case["hidden"], case["ffn"]
    encoder = mb.BertEncoder.from_weights([_layer_weights(d, f, dt, gen) for _ in range(case["layers"])], case["heads"], eps=1e-5)
    new = lambda w: torch.empty(t, w, dtype=dt, device="cuda")
    state = {"case": case, "encoder": encoder, "meta": mb.cxx.MetaData(), "tokens": t, "ffn": new(f), "temp": new(d), "attn": new(d)}
    if case["kind"] == "encoder":
        return dict(state, x=randn(t, d), hidden=new(d), info=ut.generate_data_metainfo(lens, 64, BLOCK_LIMIT, case["heads"]))
    table = lambda n: torch.randn(n, d, generator=gen, device="cuda") * 0.02
    emb = mb.BertEmbeddings(table(VOCAB), table(POSITIONS), table(2), torch.ones(d), torch.zeros(d), dtype=dt)
    pooler = mb.BertPooler((torch.randn(d, d, generator=gen, device="cuda") * 0.02).to(dt), torch.zeros(d, dtype=dt, device="cuda"))
    width = max(tokens)
    mask = (torch.arange(width, device="cuda")[None, :] < torch.tensor(tokens, device="cuda")[:, None]).to(torch.int64)
    ids = torch.randint(1, VOCAB, (len(tokens), width), generator=gen, device="cuda") * mask
    return dict(state, model=mb.BertModel(mb.BertModelNoPooler(emb, encoder), pooler), ids=ids, mask=mask, width=width,
                pooling=mb.PoolingType(case["pooling"]))


# ---- one pass ------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "layernorm":
        capi.bias_residual_layernorm(state["out"], state["residual"], state["bias"], state["gamma"], state["beta"], 1e-5)
        return state["out"]
    if case["kind"] == "gelu":
        capi.bias_gelu(state["out"], state["bias"])
        return state["out"]
    if case["kind"] == "attention":
        capi.bs_attention_fwd(state["q"], state["k"], state["vt"], state["out"], state["seq_blocks"], case["heads"],
                              state["idx"], state["pos"], case["heads"], seq_tokens_dev=state["tokens"])
        return state["out"]
    t = state["tokens"]
    if case["kind"] == "encoder":
        spi, spi_t, comp, ppi_t, pp_t = state["info"]
        state["hidden"].copy_(state["x"])
        state["meta"].update_meta_data(t, spi[-1] + 1, comp, spi)
        out, _ = state["encoder"](state["hidden"], t, BLOCK_LIMIT, spi, spi_t, ppi_t, pp_t, state["temp"], state["ffn"],
                                  state["attn"], test_info={})
        return out
    batch = ut.pack_padded_batch(state["ids"], state["mask"])
    spi, spi_t, comp, ppi_t, pp_t = ut.generate_data_metainfo(batch["seq_lens"], 64, BLOCK_LIMIT, case["heads"])
    state["meta"].update_meta_data(t, spi[-1] + 1, comp, spi)
    out, pooled, _ = state["model"](batch["input_ids"], t, BLOCK_LIMIT, spi, spi_t, ppi_t, pp_t, pooling_type=state["pooling"],
                                    attention_masks=batch["seq_tokens_tensor"], token_type_ids=batch["token_type_ids"],
                                    position_ids=batch["position_ids"], output_layer_temp=state["temp"],
                                    intermediate_temp=state["ffn"], attention_output=state["attn"])
    return ut.unpack_to_padded(out, batch["seq_lens"], batch["seq_tokens"], state["width"]), pooled
