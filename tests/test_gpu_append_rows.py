"""The append kernel's branches, bit for bit against the oracle: one row and
four rows per thread (from kBulkRows (token, head) rows on) with remainders, wide and narrow loads and stores (rows off the 16-byte and 4-byte grid), page
sizes that are no power of two, groups so large or small that the quotients
are divided instead of taken through the reciprocal, and values on the
rounding thresholds of their group."""
import os
import re

import numpy as np
import pytest
import torch

import knlp_amd as K
from oracle import quant as Q
from tests import kvgen

pytestmark = pytest.mark.gpu
DEV = "cuda"
with open(os.path.join(os.path.dirname(K.__file__), "csrc", "kv_append.hip")) as f:
    LINE = int(re.search(r"kBulkRows = (\d+);", f.read())[1])


def rows(n, hkv, d, seed, dtype, shift=0):
    """Rows of mixed magnitude; a quarter of the groups of 32 hold multiples of
    1/30 of their range (every other one a threshold of the asymmetric codes)
    and a few are 2^80 or 2^-80 times as large (bf16)."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, hkv, d // 16, 16, generator=g)
    pick = torch.rand(n, hkv, d // 16, 1, generator=g)
    grid = torch.randint(0, 31, x.shape, generator=g).float() * 0.0625
    grid[..., 0], grid[..., 1] = 0, 30 * 0.0625
    x = torch.where(pick < 0.25, grid, x)
    if dtype == torch.bfloat16:
        x = torch.where(pick > 0.98, x * 2.0 ** 80, x)
        x = torch.where((pick > 0.96) & (pick <= 0.98), x * 2.0 ** -80, x)
    wide = torch.zeros(n, hkv, d + 8, dtype=dtype)
    wide[:, :, shift:shift + d] = x.view(n, hkv, d).to(dtype)
    return wide.to(DEV)[:, :, shift:shift + d]


def check(fmt, tokens, hkv, d, gs, page, dtype, shift, code_shift, clip=10.0):
    nb = -(-tokens // page) + 2
    g = torch.Generator().manual_seed(tokens + d)
    slots = torch.randperm(nb * page, generator=g)[:tokens]
    slots[::37] = -1
    k = rows(tokens, hkv, d, 11 + d, dtype, shift)
    v = rows(tokens, hkv, d, 12 + d, dtype, shift)
    last = d if fmt == "int8" else d // 2
    kind = torch.int8 if fmt == "int8" else torch.uint8
    host = [torch.full((nb, page, hkv, last + 8), 90, dtype=kind) for _ in range(2)]
    dev = [t.to(DEV) for t in host]
    cut = [t[..., code_shift:code_shift + last] for t in dev]
    ref = [t[..., code_shift:code_shift + last].numpy().copy() for t in host]
    n = 4 if fmt == "int4_asym" else 2
    par = [torch.full((nb, page, hkv, d // gs), 3.0, dtype=torch.float16) for _ in range(n)]
    pref = [t.numpy().copy() for t in par] + [None, None]
    pdev = [t.to(DEV) for t in par] + [None, None]
    kf, vf, sl = k.float().cpu().numpy(), v.float().cpu().numpy(), slots.numpy()
    if fmt == "int8":
        for x, f, i in ((kf, K.reshape_and_cache_k_int8, 0), (vf, K.reshape_and_cache_v_int8, 1)):
            Q.reshape_and_cache_k_int8(x, ref[i], pref[i], sl, group_size=gs)
            f((k, v)[i], cut[i], pdev[i], slots.to(DEV), group_size=gs)
    else:
        asym = fmt == "int4_asym"
        Q.reshape_and_cache_int4(kf, vf, *ref, pref[0], pref[1], sl, pref[2], pref[3],
                                 asymmetric=asym, group_size=gs, clip_ratio=clip)
        K.reshape_and_cache_int4(k, v, *cut, pdev[0], pdev[1], slots.to(DEV), pdev[2], pdev[3],
                                 asymmetric=asym, group_size=gs, clip_ratio=clip)
    torch.cuda.synchronize()
    for got, want in zip(cut + pdev, ref + pref):
        if want is not None:
            got = got.contiguous().cpu().numpy()
            np.testing.assert_array_equal(got.view(np.uint8), want.view(np.uint8))
    for t in dev:                          # the bytes around the rows are as they were
        assert bool((t[..., :code_shift] == 90).all()) and \
            bool((t[..., code_shift + last:] == 90).all())


@pytest.mark.parametrize("fmt", ["int4_asym", "int4_sym", "int8"])
@pytest.mark.parametrize("tokens,hkv,d,gs", [(LINE // 8 - 1, 8, 32, 32), (LINE // 8, 8, 64, 16),
                                             (LINE // 7 + 1, 7, 32, 16), (LINE // 4 + 5, 4, 128, 128),
                                             (LINE // 4 + 1, 4, 256, 64), (1, 3, 32, 32),
                                             (67, 5, 256, 64)])
def test_rows_per_thread(fmt, tokens, hkv, d, gs):
    """Below the line, on it, and past it with a last block of few rows."""
    check(fmt, tokens, hkv, d, gs, 16, torch.float16, 0, 0)


def test_four_rows_per_thread_copy_fp16_and_take_unaligned_rows():
    n, hkv, d = LINE // 4 + 3, 4, 64
    for shift in (0, 2):
        k = rows(n, hkv, d, 7, torch.float16, shift)
        cache = torch.zeros(n // 16 + 2, 16, hkv, d, dtype=torch.float16, device=DEV)
        slots = torch.randperm(n + 16, generator=torch.Generator().manual_seed(6))[:n].to(DEV)
        K.reshape_and_cache_fp16(k, None, cache, None, slots)
        want = torch.zeros((n // 16 + 2) * 16, hkv, d, dtype=torch.float16, device=DEV)
        want[slots] = k
        assert torch.equal(cache.view_as(want), want)
    check("int4_asym", LINE // 8 + 1, 8, 32, 32, 24, torch.bfloat16, 2, 4)


@pytest.mark.parametrize("fmt,code_shifts", [("int4_asym", (0, 1, 4)), ("int4_sym", (2, 3)),
                                             ("int8", (2, 8))])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_alignment_and_magnitude(fmt, code_shifts, dtype):
    for i, cs in enumerate(code_shifts):
        check(fmt, 150, 4, 128, (32, 64, 16)[i], (16, 24, 5)[i], dtype, (2, 6, 0)[i], cs)


def test_symmetric_without_clip_and_with_a_tight_one():
    check("int4_sym", 100, 4, 128, 32, 16, torch.bfloat16, 0, 0, clip=0.0)
    check("int4_sym", 100, 4, 128, 128, 16, torch.bfloat16, 0, 0, clip=1e-3)


@pytest.mark.parametrize("shift", [0, 2])
def test_fp16_copy(shift):
    k, v = (rows(70, 4, 64, s, torch.float16, shift) for s in (1, 2))
    kc = torch.zeros(6, 16, 4, 72, dtype=torch.float16, device=DEV)[..., shift:shift + 64]
    vc = torch.zeros(6, 16, 4, 64, dtype=torch.float16, device=DEV)
    slots = torch.randperm(96, generator=torch.Generator().manual_seed(5))[:70].to(DEV)
    K.reshape_and_cache_fp16(k, v, kc, vc, slots)
    for x, c in ((k, kc), (v, vc)):
        want = torch.zeros(96, 4, 64, dtype=torch.float16, device=DEV)
        want[slots] = x
        assert torch.equal(c.reshape(96, 4, 64), want)
