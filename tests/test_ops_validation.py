"""Host-side shape guards of the Python ops (CPU; nothing launches).  The C
ABI takes strides only and its kernels index the caches unchecked, as the
reference's Triton kernels do, so ops._check_plane refuses caches, scales
and zero-points too small for the heads and head size of a call."""
import pytest
import torch

from knlp_amd import ops
from knlp_amd._lib import KV_FP16, KV_INT4_ASYM, KV_INT4_SYM, KV_INT8_SYM


def _int4(nb=4, bs=16, h=8, d=128, gs=32, asym=True, sg=None, zg=None):
    c = torch.zeros(nb, bs, h, d // 2, dtype=torch.uint8)
    s = torch.zeros(*(sg or (nb, bs, h, d // gs)), dtype=torch.float16)
    z = torch.zeros(*(zg or (nb, bs, h, d // gs)), dtype=torch.float16) if asym else None
    return ops._plane(c, s, z, KV_INT4_ASYM if asym else KV_INT4_SYM, gs)


def test_matching_planes_pass():
    ops._check_plane(_int4(), "key", 8, 128)
    ops._check_plane(_int4(asym=False), "key", 8, 128)
    ops._check_plane(_int4(), "key", 4, 128)          # a cache may hold more heads
    c8 = torch.zeros(4, 16, 8, 128, dtype=torch.int8)
    ops._check_plane(ops._plane(c8, torch.zeros(4, 16, 8, 1, dtype=torch.float16), None,
                                KV_INT8_SYM, 128), "key", 8, 128)
    c16 = torch.zeros(4, 16, 8, 128, dtype=torch.float16)
    ops._check_plane(ops._plane(c16, None, None, KV_FP16, 128), "value", 8, 128)


@pytest.mark.parametrize("heads,d", [(9, 128), (8, 256)])
def test_cache_too_small_for_the_call(heads, d):
    with pytest.raises(ValueError, match="fewer than"):
        ops._check_plane(_int4(), "key", heads, d)


@pytest.mark.parametrize("kw", [dict(sg=(4, 16, 8, 2)), dict(sg=(3, 16, 8, 4)),
                                dict(sg=(4, 8, 8, 4)), dict(sg=(4, 16, 4, 4)),
                                dict(zg=(4, 16, 8, 1))])
def test_scales_or_zeros_too_small(kw):
    with pytest.raises(ValueError, match="do not cover"):
        ops._check_plane(_int4(**kw), "value", 8, 128)


def test_int8_and_fp16_caches_need_full_rows():
    c8 = torch.zeros(4, 16, 8, 64, dtype=torch.int8)        # half a 128-element row
    p = ops._plane(c8, torch.zeros(4, 16, 8, 1, dtype=torch.float16), None, KV_INT8_SYM, 128)
    with pytest.raises(ValueError, match="fewer than"):
        ops._check_plane(p, "key", 8, 128)
    c16 = torch.zeros(4, 16, 8, 64, dtype=torch.float16)
    with pytest.raises(ValueError, match="fewer than"):
        ops._check_plane(ops._plane(c16, None, None, KV_FP16, 128), "key", 8, 128)


@pytest.mark.parametrize("kind", [int, float, torch.tensor])
def test_counts_reach_the_extension_as_integers(monkeypatch, kind):
    """split_tokens and total_context are whole numbers of any type that int()
    takes (a sum of lengths kept as a float, a 0-dim tensor)."""
    class Host:
        @staticmethod
        def decode(*a):
            return a[17], a[18]
    monkeypatch.setattr(ops, "host", lambda: Host)
    c = torch.zeros(4, 16, 8, 64, dtype=torch.uint8)
    got = ops.fused_int4_decode(None, c, c, None, None, None, None, 8, 128,
                                split_tokens=kind(128), total_context=kind(9000))
    assert got == (128, 9000) and all(type(n) is int for n in got)


@pytest.mark.parametrize("rows,slots", [((1, 1), False), ((1, 0), False), ((0, 0), True),
                                        ((0, 0), False)])
def test_fused_append_needs_slots_and_rows(monkeypatch, rows, slots):
    """A step without slots, or without any rows, is refused and not decoded
    without its new token."""
    monkeypatch.setattr(ops, "host", lambda: pytest.fail("the call reached the extension"))
    q = torch.zeros(2, 8, 128, dtype=torch.float16)
    c = torch.zeros(4, 16, 8, 64, dtype=torch.uint8)
    s = torch.zeros(4, 16, 8, 4, dtype=torch.float16)
    kv = [torch.zeros(2, 8, 128, dtype=torch.float16) if r else None for r in rows]
    with pytest.raises(ValueError, match="slot_mapping"):
        ops.append_and_decode(q, *kv, torch.zeros(2, dtype=torch.int64) if slots else None, c, c,
                              s, s, None, None, 8, 128)


def test_a_negative_split_is_refused_wherever_it_is_set(monkeypatch):
    class Host:
        @staticmethod
        def decode(*a):
            return a[17]
    monkeypatch.setattr(ops, "host", lambda: Host)
    c = torch.zeros(4, 16, 8, 64, dtype=torch.uint8)
    args = (None, c, c, None, None, None, None, 8, 128)
    for setting, want in ((0, -1), (256, 256)):                  # 0: the library's schedule
        monkeypatch.setattr(ops.config, "DECODE_SPLIT_TOKENS", setting)
        assert ops.fused_int4_decode(*args) == want
    with pytest.raises(ValueError, match="negative"):
        ops.fused_int4_decode(*args, split_tokens=-64)
    monkeypatch.setattr(ops.config, "DECODE_SPLIT_TOKENS", -64)
    with pytest.raises(ValueError, match="negative"):
        ops.fused_int4_decode(*args)


class _OnDevice:
    """A CPU tensor that says it is a device tensor (nothing is launched)."""
    is_cuda = True

    def __init__(self, t):
        self._t = t

    def __getattr__(self, name):
        return getattr(self._t, name)


def test_prefill_kernel_takes_no_overlapping_output_or_odd_scale():
    """An output in K's or V's memory would be written while other blocks read
    it; a scale of None is the default and one beyond fp32 is not taken."""
    rows = torch.zeros(4, 6, 64, dtype=torch.float16)
    q, k, v = (_OnDevice(torch.zeros(4, h, 64, dtype=torch.float16)) for h in (6, 6, 6))
    out = _OnDevice(rows)
    for scale, ok in ((0.1, True), (None, True), (-3.0, True), (1e39, False),
                      (float("inf"), False), (float("nan"), False)):
        assert ops.prefill_supported(q, k, v, out, scale) == ok, scale
    assert not ops.prefill_supported(q, out, v, out, 0.1)
    assert not ops.prefill_supported(q, k, out, out, 0.1)
    assert ops.prefill_supported(out, k, v, out, 0.1)      # a block reads only the q rows it writes
    shifted = _OnDevice(torch.zeros(5, 6, 64, dtype=torch.float16)[1:])
    before = _OnDevice(torch.as_strided(shifted._t, (4, 6, 64), (384, 64, 1), 0))
    assert not ops.prefill_supported(shifted, k, v, before, 0.1)
