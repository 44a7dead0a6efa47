"""The form a launch runs, as the launcher decides it (host only; 256 compute
units and 8 XCDs where there is no GPU, as on the MI355X)."""
import random

import pytest

import fmha_native_amd as fmha

AUTO, REF = fmha.VARIANT_AUTO, fmha.VARIANT_REFERENCE_ORDER
BIG = 1 << 40


def params(h, hk, sq, sk, varlen=False):
    p = fmha.FmhaFwdParams()
    p.q = p.k = p.v = p.o = 1 << 20
    p.scale, p.nhead_q, p.nhead_k, p.seqlen_q, p.seqlen_k = 0.18, h, hk, sq, sk
    for n in "qkvo":
        for f in ("stride", "nhead_stride", "batch_stride"):
            setattr(p, f"{f}_{n}", 64)
    if varlen:
        p.seqstart_q = p.seqstart_k = 1 << 20
    return p


def form(b, h, hk, sq, sk, causal, ws=0, variant=AUTO, varlen=False):
    return fmha.FORMS.get(fmha.launch_form(params(h, hk, sq, sk, varlen), b, causal, variant, ws))


@pytest.mark.parametrize("b,h,hk,sq,sk,causal,plain,with_ws", [
    (1, 2, 2, 128, 128, 0, "regular", "regular"),
    (4, 16, 16, 2048, 2048, 0, "wide", "wide"),
    (1, 16, 16, 8192, 8192, 1, "pair", "pair"),
    (1, 2, 2, 40000, 40000, 1, "regular", "balanced"),
    (128, 16, 16, 128, 128, 0, "short", "short"),
    (16, 32, 8, 1, 4100, 1, "decode", "decode"),
    (1, 16, 4, 512, 16384, 1, "decode", "chunk"),
    (1, 4, 4, 4096, 4096, 0, "splitkv", "chunk"),
    (1, 8, 8, 512, 512, 0, "decode", "decode"),
])
def test_forms_of_common_launches(b, h, hk, sq, sk, causal, plain, with_ws):
    assert form(b, h, hk, sq, sk, causal) == plain
    assert form(b, h, hk, sq, sk, causal, BIG) == with_ws


def test_named_variants_and_order_flags_keep_their_form():
    for v in ("regular", "splitkv", "pair", "short", "pair_stream"):
        for ws in (0, BIG):
            assert form(2, 8, 8, 1, 4096, 1, ws, fmha.VARIANTS[v]) == v
            assert form(2, 8, 8, 1, 4096, 1, ws, fmha.VARIANTS[v] | REF) == v
    for flag in (REF, fmha.VARIANT_TILE_MAJOR_ORDER, fmha.VARIANT_SEQUENCE_ORDER):
        assert form(4, 16, 16, 2048, 2048, 0, 0, AUTO | flag) == "pair"      # wide without the flag
        assert form(16, 32, 8, 1, 4100, 1, BIG, AUTO | flag) == "regular"    # decode without it
        assert form(1, 16, 4, 512, 16384, 1, BIG, AUTO | flag) == "balanced"  # chunk without it
        assert form(1, 2, 2, 40000, 40000, 1, BIG, AUTO | flag) == "balanced"


def test_rejected_and_empty_launches():
    p = params(2, 2, 40000, 40000)
    f = lambda v, ws=0, b=1, c=1, q=p: fmha.launch_form(q, b, c, v, ws)
    for v in (fmha.VARIANT_BALANCED, fmha.VARIANT_BALANCED_PAIR):
        need = fmha.workspace_size(p, 1, 1, v)
        assert need > 0 and f(v, need) == v and f(v, need - 1) == -1 and f(v, BIG, c=0) == -1
        assert f(v, 0, b=0) == 0
    assert f(4) == f(99) == f(REF | fmha.VARIANT_TILE_MAJOR_ORDER) == f(AUTO, -1) == f(AUTO, 0, c=2) == -1
    v = params(2, 2, 400, 400, varlen=True)
    assert f(fmha.VARIANT_PAIR_STREAM, q=v) == f(fmha.VARIANT_PAIR_STREAM, b=0, q=v) == -1
    assert f(AUTO, b=0) == f(AUTO, q=params(2, 2, 0, 400)) == f(fmha.VARIANT_PAIR, b=0) == 0


def test_workspace_and_form_agree():
    """The bytes workspace_size asks for are those its form needs: one byte
    less and another form runs (decode: the same, unsplit); none and the
    launch needs none."""
    r = random.Random(5)
    seen = set()
    for _ in range(3000):
        h, hk = r.choice([(1, 1), (2, 2), (4, 4), (8, 8), (16, 16), (32, 8), (16, 2), (6, 3)])
        sq, sk = int(2 ** r.uniform(0, 14)), int(2 ** r.uniform(0, 15))
        b, causal, varlen = int(2 ** r.uniform(0, 7)), r.randrange(2), r.random() < 0.2
        p = params(h, hk, sq, sk, varlen)
        need = fmha.workspace_size(p, b, causal)
        f = fmha.launch_form(p, b, causal, AUTO, need)
        tag = (b, h, hk, sq, sk, causal, varlen, need, f)
        seen.add((f, need > 0))
        if f in (fmha.FORM_CHUNK, fmha.VARIANT_BALANCED):
            assert need > 0 and not varlen and need % 34816 == 0, tag
            assert fmha.launch_form(p, b, causal, AUTO, need - 1) != f, tag
        elif f != fmha.FORM_DECODE:
            assert need == 0, tag
        if need == 0 and f not in (fmha.FORM_DECODE, fmha.FORM_WIDE):
            assert f == fmha.pick_variant(p, b, causal), tag
    assert {(fmha.FORM_DECODE, True), (fmha.FORM_DECODE, False), (fmha.FORM_CHUNK, True), (fmha.FORM_WIDE, False),
            (fmha.VARIANT_BALANCED, True)} <= seen


@pytest.mark.parametrize("b,h,hk,sq,sk,causal,wide", [
    (64, 8, 8, 256, 256, 0, True), (4, 16, 16, 2048, 2048, 0, True), (12, 16, 16, 1000, 1000, 0, True),  # two or more
    (28, 8, 1, 703, 4872, 1, True), (12, 32, 32, 406, 1584, 1, True), (13, 8, 2, 1011, 4696, 1, True),
    (58, 8, 2, 193, 193, 1, False), (50, 8, 2, 206, 206, 1, False), (26, 16, 4, 129, 129, 1, False),  # a light M-tile
    # at most one 256-row block per compute unit: one wave per SIMD
    (1, 40, 40, 1024, 512, 0, False), (1, 32, 32, 2048, 256, 0, False), (1, 64, 64, 767, 512, 0, False),
    (3, 24, 24, 445, 870, 1, False), (2, 16, 4, 1918, 1918, 0, False), (20, 4, 1, 389, 479, 1, False),
    (32, 8, 8, 132, 76, 0, False), (18, 8, 2, 155, 324, 0, False),
    # ... but a head's two M-tiles would run on two XCDs and its keys are few
    (26, 6, 6, 153, 848, 0, True), (54, 4, 1, 132, 1159, 0, True), (14, 12, 12, 238, 238, 0, True),
    (14, 12, 12, 238, 1281, 0, False), (1, 129, 129, 256, 64, 0, False), (14, 12, 12, 238, 238, 1, False), (9, 6, 6, 546, 135, 0, False),
])
def test_wide_rule(b, h, hk, sq, sk, causal, wide):
    assert (form(b, h, hk, sq, sk, causal) == "wide") == wide


@pytest.mark.parametrize("b,h,sq,sk,causal,chunk", [
    (1, 16, 512, 16384, 1, True), (1, 4, 4096, 4096, 0, True), (1, 2, 4096, 4096, 1, True), (2, 24, 124, 9467, 0, True),
    # causal M-tiles of nearly one length: a chunk length that cuts the longest
    # ones alone leaves the others whole, as long as they were
    (1, 72, 256, 2048, 1, False), (1, 80, 256, 2048, 1, False), (1, 40, 512, 2048, 1, False),
    (1, 32, 640, 2048, 1, False), (2, 24, 298, 5399, 1, False),
    (1, 16, 1024, 1024, 0, False), (5, 32, 128, 9000, 0, True), (161, 1, 128, 9000, 0, False),  # 5/8 per CU: 160
])
def test_chunk_form_rule(b, h, sq, sk, causal, chunk):
    assert (form(b, h, h, sq, sk, causal, BIG) == "chunk") == chunk


@pytest.mark.parametrize("b,h,hk,sq,sk,causal,ws,expect", [
    # every row tile of a head on an XCD of its own: K and V come once per tile
    (7, 6, 6, 165, 5698, 1, BIG, "chunk"), (8, 12, 12, 66, 19520, 1, BIG, "chunk"),
    (14, 2, 2, 83, 14968, 0, BIG, "chunk"), (10, 3, 3, 116, 10835, 0, BIG, "chunk"),
    # the chain of key steps bounds these
    (1, 8, 8, 512, 512, 0, 0, "decode"), (1, 4, 4, 256, 8192, 0, BIG, "decode"), (1, 2, 2, 2048, 2048, 0, BIG, "decode"),
    (8, 16, 2, 64, 1000, 0, BIG, "decode"),
])
def test_decode_estimate_counts_the_memory(b, h, hk, sq, sk, causal, ws, expect):
    assert form(b, h, hk, sq, sk, causal, ws) == expect


@pytest.mark.parametrize("b,h,hk,sq,sk,causal,varlen,decode", [
    (16, 32, 8, 1, 4100, 1, False, True), (512, 16, 16, 8, 1000, 0, False, True), (16, 8, 8, 32, 2000, 1, True, True),
    (4, 16, 16, 48, 2000, 0, False, True), (4, 16, 16, 48, 2000, 0, True, True),  # two row tiles, within one round
    # two row tiles per head, more than one per compute unit
    (32, 16, 16, 48, 1024, 0, False, False), (76, 6, 6, 64, 1787, 1, False, False), (100, 2, 2, 48, 5550, 1, False, False),
    (58, 4, 4, 52, 7077, 1, False, False), (32, 32, 16, 64, 2048, 1, False, False),
    (32, 16, 16, 48, 1024, 0, True, False), (100, 2, 2, 48, 5550, 1, True, False),
    (4, 16, 16, 48, 900, 0, True, False),
])
def test_decode_rule_past_32_queries(b, h, hk, sq, sk, causal, varlen, decode):
    for ws in (0, BIG):
        assert (form(b, h, hk, sq, sk, causal, ws, varlen=varlen) == "decode") == decode


@pytest.mark.parametrize("varlen", [False, True])
@pytest.mark.parametrize("b,h,hk,sq,sk,causal,expect", [
    (128, 16, 16, 32, 128, 0, "short"), (128, 16, 16, 32, 192, 1, "short"), (512, 16, 16, 8, 130, 0, "short"),
    (600, 16, 16, 32, 380, 1, "short"), (200, 32, 8, 32, 150, 0, "short"),  # four row tiles for four heads
    (400, 32, 8, 24, 150, 0, "decode"), (400, 32, 8, 16, 150, 0, "decode"), (600, 64, 8, 16, 150, 0, "decode"),
    (128, 16, 16, 31, 128, 0, "decode"), (128, 16, 16, 32, 193, 0, "decode"),  # not the short form's
])
def test_decode_leaves_the_short_form(b, h, hk, sq, sk, causal, expect, varlen):
    assert form(b, h, hk, sq, sk, causal, varlen=varlen) == expect


@pytest.mark.parametrize("varlen", [False, True])
def test_decode_grid_stays_within_the_launch_limit(varlen):
    """A grid holds fewer than 2^32 threads; eight-wave decode blocks reach it
    at half the heads the M-tile grid takes (K and V of all heads may be one:
    head stride 0)."""
    limit = (1 << 32) // 512
    assert form(1, limit - 1, limit - 1, 1, 4096, 0, varlen=varlen) == "decode"
    assert form(1, limit + 1, limit + 1, 1, 4096, 0, varlen=varlen) == "regular"
    assert form(1, 2 * limit - 2, limit - 1, 1, 4096, 0, varlen=varlen) == "decode"
