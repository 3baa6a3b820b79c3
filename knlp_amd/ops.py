"""Drop-in replacements for the module functions of knlp's fused INT4 backend.

Same names, argument order, defaults and in-place / return conventions as
``fused-quant/fused_int4.v0.1.0.py`` (F): the write functions mutate the
caller's caches and return None; the decode functions return a new tensor
shaped like ``query`` (``torch.empty_like(query)``, F:932).  Every function
launches onto the current torch stream through the C ABI of
``libknlp_int4kv.so`` and performs no host synchronisation, so the calls can
be captured in a HIP graph.  There is no CPU fallback: a missing library
raises.

Extensions over the reference, all keyword-only and defaulting to the
reference's behaviour:
  * ``group_size`` / ``k_group_size`` / ``v_group_size`` -- the reference uses
    the module-wide GROUP_SIZE for K and V alike (F:1412-1418); per-plane
    sizes allow e.g. per-row INT8 K (group = head_size) with g32 INT4 V;
  * ``clip_ratio`` -- defaults to OUTLIER_CLIP_RATIO like F:470;
  * ``scale`` -- defaults to 1/sqrt(head_size) as F:924 fixes it;
  * ``split_tokens`` -- split-K length, default from the library's plan; 0 is
    the stream schedule (equal shares of all rows' tiles per CU);
  * ``total_context`` -- the batch's summed sequence lengths when the caller
    knows them on the host (0: unknown); with it the plan keeps split-K for
    uniform batches and picks the stream schedule for variable-length ones;
    unknown, it picks the stream schedule for any batch of several sequences
    the cooperative kernel takes.
``block_n`` is accepted for signature compatibility and ignored: the HIP
kernels pick their own token tiles.
"""
from __future__ import annotations

import ctypes

import torch

from . import config
from ._lib import (DT_BF16, DT_F16, KV_FP16, KV_INT4_ASYM, KV_INT4_SYM, KV_INT8_SYM, KvPlane,
                   check, host, lib)

GROUP_SIZE = config.GROUP_SIZE
OUTLIER_CLIP_RATIO = config.OUTLIER_CLIP_RATIO
ASYMMETRIC = config.ASYMMETRIC

_SRC_DTYPES = {torch.float16: DT_F16, torch.bfloat16: DT_BF16}


def _stream() -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _require_cuda(*ts: torch.Tensor) -> None:
    for t in ts:
        if t is not None and not t.is_cuda:
            raise ValueError("knlp_amd ops need device tensors (the HIP path has no CPU fallback)")


# a side without rows in an append, and a decode without an append
_NO_PLANE = (None, None, None, 0, 0)
_NO_APPEND = (None, None, None, 0.0)


def _plane(cache: torch.Tensor, scales, zeros, fmt: int, group_size: int) -> KvPlane:
    """The ``knlp_kv_plane`` of these tensors (validated), for callers of the C
    ABI; ``tensors`` keeps what the operators take."""
    p = KvPlane()
    host().plane(cache, scales, zeros, fmt, group_size, ctypes.addressof(p))
    p.tensors = (cache, scales, zeros, fmt, group_size)
    return p


def _check_plane(p: KvPlane, name: str, num_heads: int, head_size: int) -> None:
    """Raise ValueError unless the cache of plane ``p`` holds ``num_heads``
    heads of ``head_size`` elements and its scales / zero-points cover every
    (block, slot, head, group) of it.  The kernels index these tensors
    through their strides without bounds checks (as the reference's Triton
    kernels do), so a cache with fewer heads, a shorter packed axis or
    smaller scale arrays than the call implies would be read or written out
    of bounds; every operator makes this check."""
    host().check_plane(*p.tensors, name, num_heads, head_size)


def _append(key, value, kplane, vplane, slot_mapping, clip_ratio, block_size) -> None:
    host().append(key, value, *(kplane.tensors if kplane is not None else _NO_PLANE),
                  *(vplane.tensors if vplane is not None else _NO_PLANE), slot_mapping,
                  clip_ratio, block_size)


def reshape_and_cache_int4(key, value, key_cache, value_cache, k_scales, v_scales,
                           slot_mapping, k_zeros=None, v_zeros=None, asymmetric=False, *,
                           group_size=None, clip_ratio=None) -> None:
    """Quantise fp16/bf16 K and V to packed INT4 and write them at
    ``slot_mapping`` into the paged caches (F:418-472).  Symmetric mode uses
    the trimmed-mean outlier clip (F:328-357); asymmetric stores zero-points."""
    gs = group_size or GROUP_SIZE
    fmt = KV_INT4_ASYM if asymmetric else KV_INT4_SYM
    host().append(key, value, key_cache, k_scales, k_zeros, fmt, gs, value_cache, v_scales,
                  v_zeros, fmt, gs, slot_mapping,
                  OUTLIER_CLIP_RATIO if clip_ratio is None else clip_ratio, key_cache.shape[1])


def reshape_and_cache_v_only_int4(value, value_cache, v_scales, slot_mapping, v_zeros=None,
                                  asymmetric=False, *, group_size=None,
                                  clip_ratio=None) -> None:
    """V-only INT4 quantise-and-cache (F:603-647)."""
    host().append(None, value, *_NO_PLANE, value_cache, v_scales, v_zeros,
                  KV_INT4_ASYM if asymmetric else KV_INT4_SYM, group_size or GROUP_SIZE,
                  slot_mapping, OUTLIER_CLIP_RATIO if clip_ratio is None else clip_ratio,
                  value_cache.shape[1])


def reshape_and_cache_k_int8(key, key_cache_int8, k_scales, slot_mapping, *,
                             group_size=None) -> None:
    """Symmetric INT8 K quantise-and-cache (F:1287-1312)."""
    host().append(key, None, key_cache_int8, k_scales, None, KV_INT8_SYM,
                  group_size or GROUP_SIZE, *_NO_PLANE, slot_mapping, 0.0,
                  key_cache_int8.shape[1])


def reshape_and_cache_v_int8(value, value_cache_int8, v_scales, slot_mapping, *,
                             group_size=None) -> None:
    """Symmetric INT8 V quantise-and-cache (F:1619-1650)."""
    host().append(None, value, *_NO_PLANE, value_cache_int8, v_scales, None, KV_INT8_SYM,
                  group_size or GROUP_SIZE, slot_mapping, 0.0, value_cache_int8.shape[1])


def reshape_and_cache_fp16(key, value, key_cache, value_cache, slot_mapping) -> None:
    """Plain fp16 K and V rows into fp16 paged caches at ``slot_mapping``
    (``slot < 0`` skipped).  Not a function of the reference module: it is
    the write vLLM's ``reshape_and_cache_flash`` does for the fp16 planes
    (F:2535-2544), on this library's append kernel.  Either side may be
    None."""
    src = key if key is not None else value
    if src is None:
        raise ValueError("reshape_and_cache_fp16 needs key or value")
    if src.dtype != torch.float16:
        raise ValueError("reshape_and_cache_fp16 writes fp16 caches from fp16 rows")
    d = src.shape[2]
    kp = _NO_PLANE if key is None else (key_cache, None, None, KV_FP16, d)
    vp = _NO_PLANE if value is None else (value_cache, None, None, KV_FP16, d)
    host().append(key, value, *kp, *vp, slot_mapping, 0.0,
                  (key_cache if key is not None else value_cache).shape[1])


def _run(query, k, v, block_size, block_table, seq_lens, num_kv_heads, head_size, scale,
         split_tokens, total_context, append=_NO_APPEND) -> torch.Tensor:
    """One decode; ``k`` and ``v`` are (cache, scales, zeros, format, group size)."""
    if split_tokens is None:
        split_tokens = config.DECODE_SPLIT_TOKENS or None
    if split_tokens is None:
        split_tokens = -1                                         # the library's schedule
    elif split_tokens < 0:
        raise ValueError("split_tokens must not be negative")
    return host().decode(query, *k, *v, block_size, block_table, seq_lens, num_kv_heads, head_size,
                         scale, int(split_tokens), int(total_context), *append)


def _decode(query, kp: KvPlane, vp: KvPlane, block_size, block_table, seq_lens, num_kv_heads,
            head_size, scale=None, split_tokens=None, append=None,
            total_context=0) -> torch.Tensor:
    return _run(query, kp.tensors, vp.tensors, block_size, block_table, seq_lens, num_kv_heads,
                head_size, scale, split_tokens, total_context, append or _NO_APPEND)


def prefill_supported(query, key, value, out, scale) -> bool:
    """Whether :func:`prefill_attention` takes these tensors: device tensors of
    one 16-bit dtype, heads of 64 or 128, rows that 16-byte loads can read, K
    and V rows in order, an output apart from them (its rows are written while
    other blocks still read), a scale that is finite in fp32 (None: 1/sqrt(D))."""
    if not (query.is_cuda and query.dtype in _SRC_DTYPES and query.dim() == 3 and
            query.shape[2] in (64, 128) and (scale is None or abs(scale) < 2.0 ** 127)):
        return False
    d = query.shape[2]
    spans = []                             # first byte and the one past the last
    for t in (query, key, value, out):
        if t.dim() != 3 or t.dtype != query.dtype or t.device != query.device:
            return False
        (n, h, last), (st, sh, one), p = t.shape, t.stride(), t.data_ptr()
        if last != d or one != 1 or st % 8 or sh % 8 or p % 16:
            return False
        spans.append((p, p + 2 * ((n - 1) * st + (h - 1) * sh + d)))
    if not all(d <= t.stride(0) < 1 << 24 for t in (key, value)):
        return False                       # repeated or overlapping rows
    first, end = spans[3]
    if any(first < e and s < end for s, e in spans[1:3]):
        return False
    if first < spans[0][1] and spans[0][0] < end and (first != spans[0][0] or
                                                      out.stride() != query.stride()):
        return False                       # (in place: a block reads only the rows it writes)
    return (out.shape[1] == query.shape[1] and key.shape[1] == value.shape[1] > 0 and
            query.shape[1] % key.shape[1] == 0)


def prefill_attention(query, key, value, query_start_loc, out, *, scale=None,
                      min_len=1) -> torch.Tensor:
    """Causal attention of fresh prompts into ``out`` (the reference's prefill,
    F:3127-3198): sequence s is the tokens ``query_start_loc[s]`` ..
    ``query_start_loc[s + 1] - 1`` of ``query`` / ``out`` ``[tokens, Hq, D]``
    and of ``key`` / ``value`` ``[tokens, Hkv, D]``.  Sequences of fewer than
    ``min_len`` tokens are left out.  No host synchronisation.  Not a function
    of the reference module."""
    _require_cuda(query, key, value, query_start_loc, out)
    if scale is None:
        scale = 1.0 / (query.shape[-1] ** 0.5)
    if not prefill_supported(query, key, value, out, scale):
        raise ValueError("prefill_attention needs fp16 or bf16 [tokens, heads, 64 or 128] tensors "
                         "of one dtype with 16-byte aligned rows")
    if query_start_loc.dtype != torch.int32 or not query_start_loc.is_contiguous():
        query_start_loc = query_start_loc.to(torch.int32).contiguous()
    tokens = min(t.shape[0] for t in (query, key, value, out))
    st = lib().knlp_prefill_attention(
        query.data_ptr(), key.data_ptr(), value.data_ptr(), _SRC_DTYPES[query.dtype],
        query.stride(0), query.stride(1), key.stride(0), key.stride(1), value.stride(0),
        value.stride(1), tokens, query.shape[1], key.shape[1], query.shape[2],
        query_start_loc.data_ptr(), query_start_loc.numel() - 1, int(min_len), float(scale),
        out.data_ptr(), out.stride(0), out.stride(1), _stream())
    check(st, "knlp_prefill_attention")
    return out


def int4_twos_to_offset(packed: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """Re-encode packed INT4 codes from the gpt2 compression path's
    two's-complement nibbles (gpt2/compression/kv_plugin.py:212-257) into
    this library's offset nibbles (n = t + 8, F:359).  ``packed``: uint8
    ``[..., D/2]`` with a contiguous last axis; ``out`` may be ``packed``
    itself (in place) or None (new tensor).  With that path's per-row fp16
    scale ``[..., 1]`` the result decodes as a symmetric INT4 plane of group
    size D.  Not a function of the reference module."""
    _require_cuda(packed, out)
    if packed.dtype != torch.uint8 or packed.dim() < 1 or packed.stride(-1) != 1:
        raise ValueError("packed must be uint8 with a contiguous last axis")
    if out is None:
        out = torch.empty_like(packed)
    if out.shape != packed.shape or out.dtype != torch.uint8 or out.stride(-1) != 1:
        raise ValueError("out must be uint8 shaped like packed, last axis contiguous")
    rb = packed.shape[-1]
    src2, dst2 = packed.reshape(-1, rb), out.reshape(-1, rb)
    if dst2.data_ptr() != out.data_ptr() or (out.numel() and not _same_storage(dst2, out)):
        raise ValueError("out must be reshapeable to rows without a copy")
    st = lib().knlp_int4_twos_to_offset(src2.data_ptr(), src2.stride(0) if src2.dim() else rb,
                                         dst2.data_ptr(), dst2.stride(0) if dst2.dim() else rb,
                                         src2.shape[0], rb, _stream())
    check(st, "knlp_int4_twos_to_offset")
    return out


def _same_storage(a: torch.Tensor, b: torch.Tensor) -> bool:
    return a.untyped_storage().data_ptr() == b.untyped_storage().data_ptr()


_FORMATS = {"int8": KV_INT8_SYM, "fp16": KV_FP16}


def _fmt(name: str, asymmetric: bool) -> int:
    if name == "int4":
        return KV_INT4_ASYM if asymmetric else KV_INT4_SYM
    if name not in _FORMATS:
        raise ValueError(f"unknown cache format {name!r} (int4, int8 or fp16)")
    return _FORMATS[name]


def append_and_decode(query, key, value, slot_mapping, key_cache, value_cache, k_scales,
                      v_scales, block_table, seq_lens, num_kv_heads, head_size, *,
                      k_format="int4", v_format="int4", k_zeros=None, v_zeros=None,
                      asymmetric=False, k_group_size=None, v_group_size=None,
                      clip_ratio=None, scale=None, split_tokens=None,
                      total_context=0) -> torch.Tensor:
    """Quantise the token being decoded into the caches and decode, in the
    launches of one decode (no separate append launch).

    Not a function of the reference module: it fuses the
    ``reshape_and_cache_*`` call that F's backend makes before every decode
    (F:2600-2689) into the decode, as docs/fused-quant/latency.md:41
    proposes.  ``key`` / ``value`` are ``[num_seqs, num_kv_heads, head_size]``
    rows of the new token (either may be None), ``slot_mapping[s]`` the slot
    of position ``seq_lens[s] - 1`` (``< 0``: no write).  ``k_format`` /
    ``v_format`` are "int4" (``asymmetric`` selects zero-points), "int8" or
    "fp16"; the caches, scales and zeros are the reference's tensors.  The
    written codes equal those of the separate append; the output equals the
    decode after it."""
    if query.shape[0] and (slot_mapping is None or (key is None and value is None)):
        raise ValueError("append_and_decode needs slot_mapping, and key or value")
    kf, vf = _fmt(k_format, asymmetric), _fmt(v_format, asymmetric)
    k = (key_cache, k_scales, k_zeros, kf,
         head_size if kf == KV_FP16 else (k_group_size or GROUP_SIZE))
    v = (value_cache, v_scales, v_zeros, vf,
         head_size if vf == KV_FP16 else (v_group_size or GROUP_SIZE))
    return _run(query, k, v, key_cache.shape[1], block_table, seq_lens, num_kv_heads, head_size,
                scale, split_tokens, total_context,
                (key, value, slot_mapping, OUTLIER_CLIP_RATIO if clip_ratio is None
                 else clip_ratio))


def fused_int4_decode(query, key_cache, value_cache, k_scales, v_scales, block_table, seq_lens,
                      num_kv_heads, head_size, block_n=64, k_zeros=None, v_zeros=None,
                      asymmetric=False, *, group_size=None, scale=None,
                      split_tokens=None, total_context=0) -> torch.Tensor:
    """Decode attention over packed INT4 K and V (F:901-979)."""
    gs = group_size or GROUP_SIZE
    fmt = KV_INT4_ASYM if asymmetric else KV_INT4_SYM
    return _run(query, (key_cache, k_scales, k_zeros, fmt, gs),
                (value_cache, v_scales, v_zeros, fmt, gs), key_cache.shape[1], block_table,
                seq_lens, num_kv_heads, head_size, scale, split_tokens, total_context)


def kint8_vint4_decode(query, key_cache_int8, value_cache_int4, k_scales, v_scales, block_table,
                       seq_lens, num_kv_heads, head_size, block_n=64, v_zeros=None,
                       asymmetric=False, *, k_group_size=None, v_group_size=None, scale=None,
                       split_tokens=None, total_context=0) -> torch.Tensor:
    """Decode with symmetric INT8 K and INT4 V (F:1496-1554)."""
    return _run(query, (key_cache_int8, k_scales, None, KV_INT8_SYM, k_group_size or GROUP_SIZE),
                (value_cache_int4, v_scales, v_zeros, KV_INT4_ASYM if asymmetric else KV_INT4_SYM,
                 v_group_size or GROUP_SIZE), key_cache_int8.shape[1], block_table,
                seq_lens, num_kv_heads, head_size, scale, split_tokens, total_context)


def kfp16_vint4_decode(query, key_cache_fp16, value_cache_int4, v_scales, block_table, seq_lens,
                       num_kv_heads, head_size, block_n=64, v_zeros=None, asymmetric=False, *,
                       v_group_size=None, scale=None, split_tokens=None,
                       total_context=0) -> torch.Tensor:
    """Decode with fp16 K and INT4 V (F:1159-1225)."""
    return _run(query, (key_cache_fp16, None, None, KV_FP16, head_size),
                (value_cache_int4, v_scales, v_zeros, KV_INT4_ASYM if asymmetric else KV_INT4_SYM,
                 v_group_size or GROUP_SIZE), key_cache_fp16.shape[1], block_table,
                seq_lens, num_kv_heads, head_size, scale, split_tokens, total_context)


def kint8_vint8_decode(query, key_cache_int8, value_cache_int8, k_scales, v_scales, block_table,
                       seq_lens, num_kv_heads, head_size, block_n=64, *, k_group_size=None,
                       v_group_size=None, scale=None, split_tokens=None,
                       total_context=0) -> torch.Tensor:
    """Decode with symmetric INT8 K and V (F:1796-1848)."""
    return _run(query, (key_cache_int8, k_scales, None, KV_INT8_SYM, k_group_size or GROUP_SIZE),
                (value_cache_int8, v_scales, None, KV_INT8_SYM, v_group_size or GROUP_SIZE), key_cache_int8.shape[1], block_table,
                seq_lens, num_kv_heads, head_size, scale, split_tokens, total_context)


def kfp16_vint8_decode(query, key_cache_fp16, value_cache_int8, v_scales, block_table, seq_lens,
                       num_kv_heads, head_size, block_n=64, *, v_group_size=None, scale=None,
                       split_tokens=None, total_context=0) -> torch.Tensor:
    """Decode with fp16 K and symmetric INT8 V (F:1975-2028)."""
    return _run(query, (key_cache_fp16, None, None, KV_FP16, head_size),
                (value_cache_int8, v_scales, None, KV_INT8_SYM, v_group_size or GROUP_SIZE), key_cache_fp16.shape[1], block_table,
                seq_lens, num_kv_heads, head_size, scale, split_tokens, total_context)


def fp16_paged_decode(query, key_cache_fp16, value_cache_fp16, block_table, seq_lens,
                      num_kv_heads, head_size, *, scale=None, split_tokens=None,
                      total_context=0) -> torch.Tensor:
    """The same split-K decode reading plain fp16 paged K and V caches.

    Not a reference function: it is the fp16-KV instantiation of this
    library's kernel used for the INT4-vs-fp16 comparison (the reference
    compares against SDPA, scripts/spev01/tier5_fused_decode.py:341-348)."""
    return _run(query, (key_cache_fp16, None, None, KV_FP16, head_size),
                (value_cache_fp16, None, None, KV_FP16, head_size), key_cache_fp16.shape[1], block_table,
                seq_lens, num_kv_heads, head_size, scale, split_tokens, total_context)


def decode_fp16_sdpa(query, fp16_k, fp16_v, seq_lens, num_kv_heads, num_heads,
                     head_size) -> torch.Tensor:
    """Decode attention over per-sequence fp16 K/V (F:2031-2071): ``fp16_k``
    and ``fp16_v`` are ``[max_seqs, max_ctx, num_kv_heads, head_size]``,
    sequence s holding its first ``seq_lens[s]`` positions; softmax scale
    1/sqrt(head_size), GQA head h reading kv head h // (num_heads /
    num_kv_heads), output shaped like ``query``.  The reference loops over
    the sequences with SDPA on repeat_interleave-expanded K/V; here the
    tensors are read in place as a paged cache (16-token pages when max_ctx
    allows, else one page per sequence) by the fp16 decode kernel, with no
    host synchronisation."""
    _require_cuda(query, fp16_k, fp16_v, seq_lens)
    if query.dim() != 3 or query.shape[1] != num_heads or query.shape[2] != head_size:
        raise ValueError("query must be [num_seqs, num_heads, head_size]")
    for t in (fp16_k, fp16_v):
        if t.dim() != 4 or t.shape[2] != num_kv_heads or t.shape[3] != head_size:
            raise ValueError("fp16_k / fp16_v must be [max_seqs, max_ctx, num_kv_heads, head_size]")
        if t.dtype != torch.float16:
            raise ValueError("fp16_k / fp16_v must be float16")
    num_seqs = query.shape[0]
    max_seqs, max_ctx = fp16_k.shape[:2]
    if fp16_v.shape[:2] != fp16_k.shape[:2] or num_seqs > max_seqs:
        raise ValueError("fp16_k / fp16_v shapes disagree or hold fewer sequences than query")
    page = 16 if max_ctx % 16 == 0 else max_ctx
    per_seq = max_ctx // page
    k = fp16_k.contiguous().view(max_seqs * per_seq, page, num_kv_heads, head_size)
    v = fp16_v.contiguous().view(max_seqs * per_seq, page, num_kv_heads, head_size)
    block_table = torch.arange(max_seqs * per_seq, dtype=torch.int32,
                               device=query.device).view(max_seqs, per_seq)[:num_seqs]
    return fp16_paged_decode(query, k, v, block_table, seq_lens, num_kv_heads, head_size)


def decode_kernel_kind(num_heads, num_kv_heads, head_size, k_format, k_group_size, v_format,
                       v_group_size, query_dtype=torch.float16) -> str:
    """'mfma' or 'valu': which decode kernel the library dispatches a shape to."""
    r = lib().knlp_kv_decode_kernel_kind(num_heads, num_kv_heads, head_size, k_format,
                                         k_group_size, v_format, v_group_size,
                                         _SRC_DTYPES[query_dtype])
    check(r, "knlp_kv_decode_kernel_kind")
    return "mfma" if r == 1 else "valu"
