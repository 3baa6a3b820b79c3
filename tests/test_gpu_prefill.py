"""knlp_prefill_attention against causal attention in float64 on the CPU.

Lengths sit on the edges of the kernel's tiles (32 queries a wave, 128 a
block, 64 keys a tile).  The bar: the inputs are 16-bit and exact, sums are
fp32 and the probabilities keep at least 16 bits, so an output differs from
the float64 one by its own rounding (at most 2^-11 of its value in fp16, 2^-8
in bf16) plus an absolute term of 2^-15 of the largest |v| that it averages.
"""
import math

import pytest
import torch

import knlp_amd as K
from knlp_amd import ops

pytestmark = pytest.mark.gpu


def reference(q, k, v, lens, scale):
    rep = q.shape[1] // k.shape[1]
    out, at = torch.zeros(q.shape, dtype=torch.float64), 0
    for n in lens:
        qq = q[at:at + n].double().transpose(0, 1)
        kk = k[at:at + n].double().repeat_interleave(rep, 1).transpose(0, 1)
        vv = v[at:at + n].double().repeat_interleave(rep, 1).transpose(0, 1)
        s = (qq @ kk.transpose(1, 2)) * scale
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), -math.inf)
        out[at:at + n] = (torch.softmax(s, -1) @ vv).transpose(0, 1)
        at += n
    return out


def check(got, ref, v, dtype):
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = half_ulp * ref.abs() + 2.0 ** -15 * float(v.double().abs().max())
    diff = (got.double().cpu() - ref).abs()
    assert torch.isfinite(got).all() and bool((diff <= bound).all()), float((diff / bound).max())


def starts(lens):
    return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", [(4, 1, 128), (7, 1, 64), (16, 8, 128), (6, 6, 64)])
@pytest.mark.parametrize("lens", [[1], [2, 31, 32, 33], [63, 64, 65, 0, 127], [128, 129, 1, 257],
                                  [700]])
def test_prefill_matches_float64(dtype, hq, hkv, d, lens):
    g = torch.Generator().manual_seed(len(lens) * 1000 + hq * 10 + d)
    n = sum(lens)
    q, k, v = (torch.randn(n, h, d, generator=g).to(dtype) for h in (hq, hkv, hkv))
    k[:, :, :2] *= 20                                   # outlier channels: peaked rows
    out = torch.zeros(n, hq, d, dtype=dtype, device="cuda")
    K.prefill_attention(q.cuda(), k.cuda(), v.cuda(), starts(lens), out)
    check(out, reference(q, k, v, lens, d ** -0.5), v, dtype)


@pytest.mark.parametrize("scale", [-0.2, 0.0, 3.0])
def test_prefill_any_finite_scale(scale):
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(150, 2, 64, generator=g).half() for _ in range(3))
    out = torch.zeros(150, 2, 64, dtype=torch.float16, device="cuda")
    K.prefill_attention(q.cuda(), k.cuda(), v.cuda(), starts([150]), out, scale=scale)
    check(out, reference(q, k, v, [150], scale), v, torch.float16)


@pytest.mark.parametrize("seqs", [64, 65, 130])
def test_prefill_of_many_short_prompts(seqs):
    """Up to 64 sequences the tiles of all go longest first; past that they are
    laid end to end, 64 at a time.  Empty sequences and one-token rows (left
    out, min_len = 2) among them, and two tiles in some."""
    g = torch.Generator().manual_seed(seqs)
    lens = torch.randint(0, 40, (seqs,), generator=g).tolist()
    lens[5], lens[6], lens[-1], lens[seqs // 2] = 0, 1, 200, 129
    n, hq, hkv, d = sum(lens), 4, 2, 64
    q, k, v = (torch.randn(n, h, d, generator=g).half() for h in (hq, hkv, hkv))
    out = torch.full((n, hq, d), 7.0, dtype=torch.float16, device="cuda")
    K.prefill_attention(q.cuda(), k.cuda(), v.cuda(), starts(lens), out, min_len=2)
    ref = reference(q, k, v, lens, d ** -0.5)
    one = torch.repeat_interleave(torch.tensor(lens), torch.tensor(lens)) == 1
    assert bool((out.cpu()[one] == 7.0).all()) and bool(one.any())
    check(out.cpu()[~one], ref[~one], v, torch.float16)


def test_prefill_strided_rows_and_short_rows_left_out():
    """q, k, v as views of one fused qkv tensor, an output with other rows
    around it, and the batch's one-token rows not written (min_len = 2)."""
    g = torch.Generator().manual_seed(4)
    lens, hq, hkv, d = [1, 70, 1, 200, 1], 8, 2, 128
    n = sum(lens)
    qkv = torch.randn(n, hq + 2 * hkv, d, generator=g).bfloat16()
    c = qkv.cuda()
    q, k, v = c[:, :hq], c[:, hq:hq + hkv], c[:, hq + hkv:]
    out = torch.full((n + 3, hq + 1, d), 7.0, dtype=torch.bfloat16, device="cuda")
    K.prefill_attention(q, k, v, starts(lens), out[:, 1:], min_len=2)
    ref = reference(qkv[:, :hq], qkv[:, hq:hq + hkv], qkv[:, hq + hkv:], lens, d ** -0.5)
    at = 0
    for m in lens:
        rows = out[at:at + m, 1:]
        if m == 1:
            assert bool((rows == 7.0).all())
        else:
            check(rows, ref[at:at + m], qkv, torch.bfloat16)
        at += m
    assert bool((out[n:] == 7.0).all()) and bool((out[:, 0] == 7.0).all())


def test_prefill_rows_past_the_end_do_not_leak():
    """The tokens that follow a sequence in its last key tile belong to the
    next one: Inf and NaN there change nothing."""
    g = torch.Generator().manual_seed(5)
    lens = [40, 90]
    q, k, v = (torch.randn(130, 2, 128, generator=g).half() for _ in range(3))
    bad_k, bad_v = k.clone(), v.clone()
    bad_k[40:], bad_v[40:] = math.nan, math.inf
    out = torch.zeros(130, 2, 128, dtype=torch.float16, device="cuda")
    K.prefill_attention(q.cuda(), bad_k.cuda(), bad_v.cuda(), starts(lens), out)
    check(out[:40], reference(q, k, v, lens, 128 ** -0.5)[:40], v, torch.float16)


def test_prefill_peaked_and_flat_rows():
    """Scores that rise along the keys (the running max moves in every tile)
    and equal scores (a mean of V)."""
    n, d = 300, 128
    g = torch.Generator().manual_seed(6)
    v = torch.randn(n, 1, d, generator=g).half()
    q = torch.ones(n, 1, d).half()
    k = (torch.arange(n).view(n, 1, 1) * torch.ones(1, 1, d) / 16).half()
    for keys in (k, torch.zeros_like(k)):
        out = torch.zeros(n, 1, d, dtype=torch.float16, device="cuda")
        K.prefill_attention(q.cuda(), keys.cuda(), v.cuda(), starts([n]), out)
        check(out, reference(q, keys, v, [n], d ** -0.5), v, torch.float16)


@pytest.mark.parametrize("dtype,big", [(torch.float16, 2.0 ** 5), (torch.float16, 2.0 ** 15),
                                       (torch.bfloat16, 2.0 ** 40)])
def test_prefill_scores_of_any_size(dtype, big):
    """Scores far beyond 2^24 (exact: one dimension, whole multiples of a power
    of two): the largest so far takes the whole row, two equal ones share it.
    With a scale of 1 the softmax's max in its log2 units has no bits left for
    an exponent of p beside it."""
    n, d = 300, 128
    g = torch.Generator().manual_seed(8)
    rank = torch.randperm(n, generator=g) // 2                    # each value twice
    v = torch.randn(n, 1, d, generator=g).to(dtype)
    q, k = torch.zeros(n, 1, d), torch.zeros(n, 1, d)
    q[:, 0, 3] = big
    k[:, 0, 3] = (rank - 75) * (big / 256)
    q, k = q.to(dtype), k.to(dtype)
    out = torch.zeros(n, 1, d, dtype=dtype, device="cuda")
    K.prefill_attention(q.cuda(), k.cuda(), v.cuda(), starts([n]), out, scale=1.0)
    check(out, reference(q, k, v, [n], 1.0), v, dtype)


def test_prefill_unsupported_tensors_raise():
    q = torch.zeros(4, 2, 128, dtype=torch.float16, device="cuda")
    qsl = starts([4])
    for bad in (q.float(), q[:, :, :96], torch.zeros(4, 2, 129, dtype=torch.float16,
                                                     device="cuda")[:, :, 1:]):
        assert not ops.prefill_supported(bad, q, q, q, 0.1)
        with pytest.raises(ValueError):
            K.prefill_attention(bad, q, q, qsl, q)
