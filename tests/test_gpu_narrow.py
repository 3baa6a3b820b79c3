"""The cooperative kernel's narrow instances (kv heads in fours or twos, a
tile of 64 or 128 tokens in two or four parts) and its fp16-K two-set one,
against the oracle: every format they take, head counts and group sizes at the
edges of their rule, lengths at the edges of a part (32), a tile (64, 128) and
a window of pages, both schedules, the fused append, a workspace of NaN, and
layouts that must fall back to the other kernels."""
import ctypes

import numpy as np
import pytest
import torch

import knlp_amd as K
from knlp_amd import _lib, ops
from oracle import attention as A
from tests import kvgen
from tests.test_gpu_decode import _build, _check, _query, _run

pytestmark = pytest.mark.gpu
DEV = "cuda"

# name, hq, hkv, d, kfmt, vfmt, kgs, vgs
SHAPES = [
    ("qwen7b_int4_asym", 28, 4, 128, 1, 1, 32, 32),
    ("qwen7b_int4_sym", 28, 4, 128, 0, 0, 32, 32),
    ("int4_one_set", 16, 4, 128, 1, 1, 32, 32),
    ("int4_g64_wide", 32, 4, 128, 1, 1, 64, 64),
    ("int4_g64_sym_one_head", 4, 4, 128, 0, 0, 64, 64),
    ("qwen7b_k8v4", 28, 4, 128, 2, 1, 32, 32),
    ("k8row_v4_wide", 28, 4, 128, 2, 0, 128, 32),
    ("k8row_v4_one_set", 12, 4, 128, 2, 1, 128, 32),
    ("k8_v4_one_set_12_heads", 24, 12, 128, 2, 0, 32, 32),
    ("qwen7b_k8v8", 28, 4, 128, 2, 2, 32, 32),
    ("k8row_v8", 16, 4, 128, 2, 2, 128, 32),
    ("k8row_v8_two_sets", 32, 4, 128, 2, 2, 128, 32),
    ("gpt2_d64_12_heads", 12, 12, 64, 1, 1, 32, 32),
    ("d64_hkv4_sym_g8", 32, 4, 64, 0, 0, 32, 32),
    ("qwen05b_d64_hkv2", 14, 2, 64, 0, 0, 32, 32),
    ("d64_hkv2_asym", 16, 2, 64, 1, 1, 32, 32),
    ("hkv2_int4", 8, 2, 128, 1, 1, 32, 32),
    ("hkv2_int4_two_sets", 16, 2, 128, 0, 0, 32, 32),
    ("hkv6_int4", 18, 6, 128, 1, 1, 32, 32),
    ("k16_v4_two_sets", 28, 4, 128, 3, 0, 128, 32),
    ("k16_v4_asym_two_sets", 40, 8, 128, 3, 1, 128, 32),
    ("k16_v8_two_sets", 28, 4, 128, 3, 2, 128, 32),
]
LENS = [1, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 0, 700, 1025, 2100]


TILE = {2: 128, 6: 128}            # tokens of a tile by kv heads, else 64


def planned(hq, hkv, d, kf, vf, kgs, vgs):
    """knlp_kv_decode_schedule answers for the shape where the plan does not."""
    L = _lib.lib()
    a = (16, hkv, hq, d, 4096, 0, kf, kgs, vf, vgs)
    return L.knlp_kv_decode_schedule(*a) == 0 and L.knlp_kv_decode_plan(*a) > 0


@pytest.mark.parametrize("split", [None, 0, 64, 192])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: s[0])
def test_narrow_matches_oracle(shape, split):
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    assert planned(*shape[1:]), name
    seed = SHAPES.index(shape)
    lens = LENS if split != 64 else [1, 33, 65, 128, 500]
    bt, kp, vp = _build(lens, hq, hkv, d, kf, vf, kgs, vgs, seed, bs=32 if seed % 3 == 2 else 16)
    q = _query(len(lens), hq, d, seed, torch.bfloat16 if seed % 4 == 1 else torch.float16)
    out = _run(q, kp, vp, bt, lens, hkv, d, split_tokens=split)
    _check(out, q, kp, vp, bt, lens, name=f"narrow_{name}_{split}")


@pytest.mark.parametrize("split", [0, 128])
@pytest.mark.parametrize("shape,sides", [(s, "kv") for s in SHAPES] +
                         [(s, "v") for s in SHAPES if s[4] == 3],
                         ids=lambda x: x if isinstance(x, str) else x[0])
def test_narrow_fused_append(shape, sides, split):
    """The new token's rows written by the decode launch: the codes of the
    separate append and the decode that follows it, bit for bit.  (fp16 K also
    with its row already in the cache.)"""
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    lens = [1, 32, 33, 64, 129, 600]
    bt, kp, vp = _build(lens, hq, hkv, d, kf, vf, kgs, vgs, 40)
    q = _query(len(lens), hq, d, 41).to(DEV)
    new = [kvgen.randn((len(lens), hkv, d), s, torch.float16).to(DEV) for s in (42, 43)]
    if sides == "v":
        new[0] = None
    pos = np.array(lens) - 1
    slots = torch.from_numpy(bt[np.arange(len(lens)), pos // 16].astype(np.int64) * 16 + pos % 16)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    btd = torch.from_numpy(bt).to(DEV)
    outs = []
    for fused in (True, False):
        kd, ks, kz = kvgen.plane_to_torch(kp, DEV)
        vd, vs, vz = kvgen.plane_to_torch(vp, DEV)
        planes = (ops._plane(kd, ks, kz, kf, kgs), ops._plane(vd, vs, vz, vf, vgs))
        args = (new[0], new[1], slots.to(DEV), 10.0)
        if not fused:
            ops._append(new[0], new[1], planes[0] if sides == "kv" else None, planes[1],
                        slots.to(DEV), 10.0, 16)
        out = ops._decode(q, *planes, 16, btd, sl, hkv, d, split_tokens=split,
                          append=args if fused else None)
        torch.cuda.synchronize()
        outs.append([t for t in (out, kd, vd, ks, vs, kz, vz) if t is not None])
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), name


@pytest.mark.parametrize("shape", [SHAPES[0], SHAPES[5], SHAPES[14], SHAPES[19]],
                         ids=lambda s: s[0])
@pytest.mark.parametrize("split", [0, 128])
def test_narrow_reads_only_what_it_wrote(shape, split):
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    lens = [3, 0, 65, 900, 128]
    bt, kp, vp = _build(lens, hq, hkv, d, kf, vf, kgs, vgs, 50)
    q = _query(len(lens), hq, d, 50).to(DEV)
    t = [kvgen.plane_to_torch(p, DEV) for p in (kp, vp)]
    kpl, vpl = ops._plane(*t[0], kf, kgs), ops._plane(*t[1], vf, vgs)
    btd = torch.from_numpy(bt).to(DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    L, mc = _lib.lib(), bt.shape[1] * 16
    nbytes = L.knlp_kv_decode_workspace_bytes(len(lens), hq, d, mc, split)
    ws = torch.full(((nbytes + 3) // 4,), float("nan"), dtype=torch.float32, device=DEV)
    out = torch.empty_like(q)
    st = L.knlp_kv_decode(q.data_ptr(), _lib.DT_F16, q.stride(0), q.stride(1), len(lens), hq, hkv,
                          d, ctypes.byref(kpl), ctypes.byref(vpl), btd.data_ptr(), btd.stride(0),
                          sl.data_ptr(), 16, mc, d ** -0.5, split, ws.data_ptr(), nbytes,
                          out.data_ptr(), _lib.DT_F16, out.stride(0), out.stride(1),
                          ops._stream())
    assert st == 0
    torch.cuda.synchronize()
    _check(out.cpu(), q.cpu(), kp, vp, bt, lens, name=f"narrow_nan_workspace_{name}_{split}")


@pytest.mark.parametrize("shape", [SHAPES[2], SHAPES[5], SHAPES[14], SHAPES[12]],
                         ids=lambda s: s[0])
@pytest.mark.parametrize("split", [None, 0, 128])
def test_other_layouts_run_on_the_other_kernels(shape, split):
    """Rows with gaps between them (codes and scales) and pages of 8 tokens."""
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    lens = [5, 64, 700]
    for bs, gap in ((16, True), (8, False)):
        bt, kp, vp = _build(lens, hq, hkv, d, kf, vf, kgs, vgs, 60, bs=bs)
        q = _query(len(lens), hq, d, 60)
        keep, planes = [], []
        for p, f, gs in ((kp, kf, kgs), (vp, vf, vgs)):
            t = []
            for x in kvgen.plane_to_torch(p, DEV):
                if x is not None and gap:
                    wide = torch.full((*x.shape[:2], x.shape[2] + 2, x.shape[3]), 7,
                                      dtype=x.dtype, device=DEV)
                    wide[:, :, :hkv] = x
                    x = wide[:, :, :hkv]
                t.append(x)
            keep.append(t)
            planes.append(ops._plane(*t, f, gs))
        out = ops._decode(q.to(DEV), *planes, bs, torch.from_numpy(bt).to(DEV),
                          torch.tensor(lens, dtype=torch.int32, device=DEV), hkv, d,
                          split_tokens=split)
        _check(out, q, kp, vp, bt, lens, name=f"narrow_other_layout_{name}_{bs}_{split}")
        del keep


@pytest.mark.parametrize("shape", [("coop8", 32, 8, 128, 1, 1, 32, 32), SHAPES[5], SHAPES[14],
                                   ("coop16", 16, 4, 128, 3, 1, 128, 32)], ids=lambda s: s[0])
def test_whole_row_shares(shape):
    """A variable-length batch of few rows whose shares are too small for row
    charges: each row takes whole blocks (lengths that end in every part of a
    share, one sequence empty and one of a single token)."""
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    tile = {8: 32, 2: 128}.get(hkv, 32 if kf == 3 else 64)
    lens = [n * tile // 32 for n in (2900, 1, 0, 5000, 33, 1777, 3200, 640)]
    tiles = sum(-(-n // tile) for n in lens)
    assert 256 < tiles < 7 * 256
    bt, kp, vp = _build(lens, hq, hkv, d, kf, vf, kgs, vgs, 70)
    q = _query(len(lens), hq, d, 70)
    out = _run(q, kp, vp, bt, lens, hkv, d, split_tokens=0)
    _check(out, q, kp, vp, bt, lens, name=f"whole_rows_{name}")
    again = _run(q, kp, vp, bt, lens, hkv, d, split_tokens=0)
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))


@pytest.mark.parametrize("charged", [False, True])
@pytest.mark.parametrize("shape", [SHAPES[i] for i in (0, 3, 5, 9, 12, 14, 17, 19)],
                         ids=lambda s: s[0])
def test_several_segments_in_a_block(shape, charged):
    """A batch of more rows than a quarter of the CUs and more tiles than CUs:
    equal shares, with the charge of 6 tiles a row from 7 tiles a CU on, so
    most blocks end one row and start another: partials, their combination and
    the next row's copies in the same LDS.  (All sequences draw on one small
    pool of pages.)"""
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    tile = 32 if kf == 3 else TILE.get(hkv, 64)
    heads = 4 if kf == 3 or hkv % 4 == 0 else 2
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    seqs, nhg, bs = 96, hkv // heads, 16
    g = np.random.default_rng(len(name) + charged)
    lens = [int(n) for n in g.integers(1, (44 if charged else 9) * tile // nhg, seqs)]
    lens[3], lens[7], lens[8] = 0, 1, tile + 1
    tiles = nhg * sum(-(-n // tile) for n in lens)
    rows = nhg * sum(n > 0 for n in lens)
    assert 4 * rows > cus and (tiles >= 7 * cus if charged else cus < tiles < 7 * cus)
    nb = 200
    table = g.integers(0, nb, (seqs, -(-max(lens) // bs))).astype(np.int32)
    planes = []
    for f, gs, seed in ((kf, kgs, 1), (vf, vgs, 2)):
        p = kvgen.empty_plane(f, nb, bs, hkv, d, gs)
        kvgen.fill_plane(p, kvgen.randn((nb * bs, hkv, d), seed, outlier_frac=0.01).float().numpy(),
                         np.arange(nb * bs))
        planes.append(p)
    q = _query(seqs, hq, d, 90)
    out = _run(q, *planes, table, lens, hkv, d, split_tokens=0)
    _check(out, q, *planes, table, lens, name=f"segments_{name}_{charged}")
    again = _run(q, *planes, table, lens, hkv, d, split_tokens=0)
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))


# those whose other kernel is the VALU one, which sums in fp32
FROM_VALU = [s for s in SHAPES if s[4] != s[5] or s[4] == 2 or (s[1] // s[2]) * (s[3] // s[7]) > 16]


@pytest.mark.parametrize("shape", FROM_VALU, ids=lambda s: s[0])
@pytest.mark.parametrize("split", [0, 128])
def test_shapes_of_the_valu_kernel_keep_32_bit_sums(shape, split):
    """An fp16 output differs from float64 by its own rounding (2e-4 of the
    result here) and, beside it, by what 32-bit sums leave: 1e-5.  V codes as
    fp16 subnormals lost 1.2e-4 in the matrix cores."""
    name, hq, hkv, d, kf, vf, kgs, vgs = shape
    lens = [1500, 700, 2100]
    bt, kp, vp = _build(lens, hq, hkv, d, kf, vf, kgs, vgs, 80)
    q = _query(len(lens), hq, d, 80)
    out = _run(q, kp, vp, bt, lens, hkv, d, split_tokens=split).cpu().double().numpy()
    ref = A.decode_reference_f64(q.float().numpy(), kp, vp, bt, lens)
    norm = np.sqrt(np.mean(ref ** 2))
    rounding = np.mean((ref.astype(np.float16).astype(np.float64) - ref) ** 2)
    beside = np.sqrt(max(np.mean((out - ref) ** 2) - rounding, 0.0)) / norm
    print(f"{name} {split}: {beside:.2e} beside a rounding of {np.sqrt(rounding) / norm:.2e}")
    assert beside <= 1e-5
