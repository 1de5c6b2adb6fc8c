"""Host-side batch planning for the padding-free encoder.

Mirrors python/util.py of the reference: `generate_data_metainfo` (:36-50) and
`generate_parition_plan` (:11-34) keep their names, arguments and return order; the work
is done by the C-ABI library (`rt_meta_*`) instead of Python heapq loops, and the head
count is an argument instead of the literal 12.  `generate_array_with_avg` (:78-112) and
`generate_input_data` (:114-123) produce the synthetic variable-length batches of the
reference's benchmarks.
"""
import itertools
import random

import numpy as np
import torch
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import capi


def generate_parition_plan(block_num_array, seq_start_index, thread_block_num, head_num, device="cuda"):
    """LPT plan as (partition_part_index_tensor, partition_part_tensor).  `block_num_array` is
    accepted for signature compatibility; costs are derived from the geometry."""
    seq_blocks = [0]
    for start, count in seq_start_index:
        if start != seq_blocks[-1]:
            raise ValueError("seq_start_index must be contiguous")
        seq_blocks.append(start + count)
    pos, ids = capi.partition_lpt(seq_blocks, head_num, thread_block_num)
    return torch.from_numpy(pos).to(device), torch.from_numpy(ids).to(device)


def generate_data_metainfo(input_datas, block_size, thread_block_limit, head_num=12, device="cuda"):
    """(seq_position_info, seq_position_info_tensor, total_comp_block_num,
    partition_part_index_tensor, partition_part_tensor) for a list of token sequences (or
    of sequence lengths)."""
    if block_size != 64:
        raise ValueError("the kernels are built for 64-token blocks")
    lens = [int(x) if np.isscalar(x) else len(x) for x in input_datas]
    sb = capi.seq_prefix_blocks(lens)
    _, total = capi.block_costs(sb)
    pos, ids = capi.partition_lpt(sb, head_num, thread_block_limit)
    # pinned staging + asynchronous copies: a pageable copy is ordered behind everything already on the
    # stream and would make the host wait for the previous batch's layers
    up = lambda a: torch.from_numpy(a).pin_memory().to(device, non_blocking=True)
    if not str(device).startswith("cuda"):
        up = lambda a: torch.from_numpy(a).to(device)
    return sb.tolist(), up(sb), int(total), up(pos), up(ids)


def generate_array_with_avg(seq_len, batch_size, max_len, rng=None):
    """Variable lengths with a given average, floored at 768, rounded to 64, capped at
    `max_len` (python/util.py:78-112)."""
    rng = rng or random
    lens = [float(rng.randint(768, max_len + 1)) for _ in range(batch_size)]
    cur = sum(lens) / batch_size
    for i in range(batch_size):
        diff = seq_len - cur
        if lens[i] + diff > max_len:
            diff = lens[i] - max_len
        elif lens[i] + diff < 768:
            diff = lens[i] - 768
        lens[i] += diff
        cur = sum(lens) / batch_size
    diff_sum = (seq_len - cur) * batch_size
    lens.sort(reverse=diff_sum >= 0)
    for i in range(batch_size):
        diff = diff_sum / (batch_size - i)
        if lens[i] + diff > max_len:
            diff = max_len - lens[i]
        elif lens[i] + diff < 768:
            diff = 768 - lens[i]
        lens[i] += diff
        diff_sum -= diff
    return [min(max(int(round(v / 64)) * 64, 64), max_len) for v in lens]


def generate_input_data(batch_size, seq_lens, vocab=30000, rng=None):
    rng = rng or np.random
    return [rng.randint(0, vocab, (seq_lens[i],)).tolist() for i in range(batch_size)]


def uniform_lengths(batch, lo, hi, seed=0, block=64):
    """`batch` lengths uniform in [lo, hi], multiples of 64 (benchmark configs 3 and 5)."""
    rng = np.random.default_rng(seed)
    return (block * rng.integers(lo // block, hi // block + 1, size=batch)).tolist()


def pack_padded_batch(input_ids, attention_mask, token_type_ids=None, block_size=64, keep_width=False):
    """Padded HuggingFace-style batch -> the packed batch the encoder takes.

    input_ids, attention_mask: [B, L] (mask 1 on real tokens, which must be a prefix of each row).  Every
    sequence keeps its real tokens plus the padding needed to fill its own last 64-token block (the
    reference only takes lengths that are multiples of 64, python/util.py:36-46): the cheapest batch, in which
    every sequence gets the attention plan of its own length.  keep_width=True keeps every sequence at the
    batch's width L (rounded up to a block) instead, whole blocks of padding included: the plan of every
    sequence is then the one HuggingFace BigBird draws for the padded batch (python/modeling_big_bird.py:573-597
    chooses it by the padded length), so the real rows equal HuggingFace run on the padded batch itself, at the
    price of computing the padding.  Returns a dict:
      input_ids, position_ids, token_type_ids : int32 [T] packed, T = sum(seq_lens)
      seq_lens   : per-sequence packed length, a multiple of block_size
      seq_tokens : per-sequence true token count (list) and `seq_tokens_tensor` (int32, on the ids' device):
                   what the layers take as `attention_mask` so that the padded keys get no weight
    """
    if input_ids.dim() != 2 or attention_mask.shape != input_ids.shape:
        raise ValueError("input_ids and attention_mask must both be [batch, length]")
    packed = _pack_on_gpu(input_ids, attention_mask, token_type_ids, block_size, keep_width)
    if packed is not None:
        return packed
    mask = attention_mask.to(torch.int64)
    tokens = mask.sum(dim=1)
    b, length = input_ids.shape
    prefix = (torch.arange(length, device=mask.device)[None, :] < tokens[:, None]).to(torch.int64)
    if not torch.equal(prefix, (mask != 0).to(torch.int64)):
        raise ValueError("attention_mask must be 1 on a prefix of each row (right padding)")
    seq_tokens = [int(x) for x in tokens.tolist()]
    if min(seq_tokens) < 1:
        raise ValueError("every sequence needs at least one token")
    seq_lens = [(n + block_size - 1) // block_size * block_size for n in seq_tokens]
    if keep_width:
        seq_lens = [(length + block_size - 1) // block_size * block_size] * b
    pad_to = max(seq_lens)
    if pad_to > length:                                   # the padded width is not a block multiple itself
        extra = pad_to - length
        input_ids = torch.nn.functional.pad(input_ids, (0, extra))
        if token_type_ids is not None:
            token_type_ids = torch.nn.functional.pad(token_type_ids, (0, extra))
    ids, pos, typ = [], [], []
    for s, n in enumerate(seq_lens):
        ids.append(input_ids[s, :n])
        pos.append(torch.arange(n, device=input_ids.device))
        typ.append(token_type_ids[s, :n] if token_type_ids is not None else torch.zeros_like(ids[-1]))
    cat = lambda xs: torch.cat(xs).to(torch.int32).contiguous()
    return {"input_ids": cat(ids), "position_ids": cat(pos), "token_type_ids": cat(typ), "seq_lens": seq_lens,
            "seq_tokens": seq_tokens,
            "seq_tokens_tensor": torch.tensor(seq_tokens, dtype=torch.int32, device=input_ids.device)}


def _watched():
    """Whether something sees the operators that run now and would miss a kernel: a tracer or compiler, a transform, a dispatch or
    function mode (a default device is a function mode too, and not meant)."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing() or forward_ad._current_level >= 0 or
            torch._C._len_torch_dispatch_stack() > 0 or any(type(m) is not DeviceContext for m in _get_current_function_mode_stack()))


def _ordinary(t):
    """A tensor whose memory a kernel may read as it is: on the current GPU, no subclass, not batched or differentiated, no
    conjugation, sign or zeros that only its flags hold."""
    return (type(t) is torch.Tensor and t.is_cuda and t.device.index == torch.cuda.current_device() and not t.requires_grad and
            not torch._C._functorch.is_functorch_wrapped_tensor(t) and not (t.is_conj() or t.is_neg() or t._is_zerotensor()))


def _rows(t, dtypes):
    return _ordinary(t) and t.dtype in dtypes and t.stride(1) == 1 and t.stride(0) >= 0


def _pack_on_gpu(input_ids, attention_mask, token_type_ids, block_size, keep_width):
    """pack_padded_batch by two kernels; None where the batch has to take the general way: other types or strides, no entries,
    and every mask that is not plain ones and zeros with the ones in front, which the general way refuses or counts."""
    if _watched():
        return None
    ints = (torch.int32, torch.int64)
    if not (type(block_size) is int and block_size >= 1 and 1 <= input_ids.shape[0] <= 65535 and input_ids.shape[1] >= 1 and
            _rows(input_ids, ints) and _rows(attention_mask, ints + (torch.bool, torch.uint8))):
        return None
    if token_type_ids is not None and not (isinstance(token_type_ids, torch.Tensor) and token_type_ids.shape == input_ids.shape and
                                           _rows(token_type_ids, ints)):
        return None
    length = input_ids.shape[1]
    tokens = torch.empty(input_ids.shape[0], dtype=torch.int32, device=input_ids.device)
    seq_tokens = capi.padded_tokens(attention_mask, tokens).tolist()
    if min(seq_tokens) < 1:
        return None
    up = lambda n: (n + block_size - 1) // block_size * block_size
    fixed = up(length) if keep_width else 0
    seq_lens = [fixed] * len(seq_tokens) if keep_width else [up(n) for n in seq_tokens]
    total = sum(seq_lens)
    if total >= 1 << 31 or fixed >= 1 << 31:
        return None
    ids, pos, typ = (torch.empty(total, dtype=torch.int32, device=input_ids.device) for _ in range(3))
    capi.pack_tokens(input_ids, token_type_ids, tokens, block_size, fixed, max(seq_lens), ids, pos, typ)
    return {"input_ids": ids, "position_ids": pos, "token_type_ids": typ, "seq_lens": seq_lens, "seq_tokens": seq_tokens,
            "seq_tokens_tensor": tokens}


def _starts_on_gpu(packed, seq_lens, seq_tokens, length):
    """First rows of the sequences where the unpacking kernel takes them: ordinary rows of whole 16-byte vectors on the current
    GPU, every sequence inside of them and of the padded length; else None.  (The general way takes any iterable of counts, and has
    the words for what is wrong.)"""
    if _watched() or not (_ordinary(packed) and packed.dim() == 2 and packed.is_contiguous() and packed.data_ptr() % 16 == 0):
        return None
    if not (isinstance(seq_lens, (list, tuple)) and isinstance(seq_tokens, (list, tuple)) and len(seq_lens) == len(seq_tokens) >= 1 and
            all(type(n) is int for n in (*seq_lens, *seq_tokens))):
        return None
    row = packed.shape[1] * packed.element_size()
    if row == 0 or row % 16 or row >= 1 << 24 or type(length) is not int or not 1 <= length < 1 << 24 or length * row >= 1 << 37:
        return None
    starts = list(itertools.accumulate(seq_lens, initial=0))[:-1]
    inside = all(n >= 0 and 0 <= t <= length and s + t <= packed.shape[0] for s, n, t in zip(starts, seq_lens, seq_tokens))
    return starts if inside else None


def unpack_to_padded(packed, seq_lens, seq_tokens, length):
    """[T, D] packed encoder output -> [B, length, D] with zeros on the padded positions (the padded rows of
    the packed output are whatever the layers computed for padding tokens and are dropped here)."""
    starts = _starts_on_gpu(packed, seq_lens, seq_tokens, length)
    if starts is not None:
        out = torch.empty(len(seq_lens), length, packed.shape[1], dtype=packed.dtype, device=packed.device)
        return capi.unpack_rows(packed, starts, seq_tokens, out)
    out = packed.new_zeros(len(seq_lens), length, packed.shape[1])
    start = 0
    for s, (n, real) in enumerate(zip(seq_lens, seq_tokens)):
        out[s, :real] = packed[start:start + real]
        start += n
    return out
