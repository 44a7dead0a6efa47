"""Decode form: packed query rows of a KV head over many keys, whole or split
over key chunks, against float64 attention."""
import ctypes
import math

import numpy as np
import pytest
import torch

import fmha_native_amd as fmha

INF = float("inf")


def _f64(q, k, v, causal):
    """float64 attention of one sequence on the CPU: q [H, Sq, 64], k/v [Hk, Sk, 64]."""
    h, sq, _ = q.shape
    hk, sk, _ = k.shape
    q, k, v = (t.double().cpu() for t in (q, k, v))
    k, v = (t.repeat_interleave(h // hk, 0) for t in (k, v))
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / 8.0
    if causal:
        lim = torch.arange(sq)[:, None] + (sk - sq)
        s = s.masked_fill(torch.arange(sk)[None] > lim, -INF)
    lse = torch.logsumexp(s, -1) if sk else torch.full((h, sq), -INF, dtype=torch.float64)
    p = torch.exp(s - torch.where(lse == -INF, torch.zeros_like(lse), lse)[..., None])
    return torch.matmul(p, v), lse


def _check(o, lse, ref_o, ref_l, tag):
    # bf16 rounding of P and O: the benchmark rule 1e-2 + 1e-2|O| (half an ulp of
    # each is 2^-9 relative; |V| rows average out); LSE is fp32 throughout
    o, lse = o.double().cpu(), lse.double().cpu()
    # written so that NaN, the outputs' poison, is a miss
    bad = ~((o - ref_o).abs() <= 1e-2 + 1e-2 * ref_o.abs())
    assert not bool(bad.any()), (tag, int(bad.sum()), float((o - ref_o).abs().max()))
    fin = ref_l != -INF
    assert bool((lse[~fin] == -INF).all()), tag
    assert bool(((lse - ref_l).abs()[fin] <= 1e-3).all()), tag


def _params(h, hk, sq, sk):
    p = fmha.FmhaFwdParams()
    p.q = p.k = p.v = p.o = 1 << 20
    p.scale, p.nhead_q, p.nhead_k, p.seqlen_q, p.seqlen_k = 0.18, h, hk, sq, sk
    for n in "qkvo":
        for f in ("stride", "nhead_stride", "batch_stride"):
            setattr(p, f"{f}_{n}", 64)
    return p


def test_check_misses_nan():
    """Outputs start as NaN: one left unwritten fails the comparison."""
    ref = torch.ones(2, 64, dtype=torch.float64)
    ok, nan = torch.ones(2, 64), torch.ones(2, 64)
    nan[1, 3] = float("nan")
    _check(ok, torch.ones(2), ref, torch.ones(2, dtype=torch.float64), "written")
    with pytest.raises(AssertionError):
        _check(nan, torch.ones(2), ref, torch.ones(2, dtype=torch.float64), "O")
    with pytest.raises(AssertionError):
        _check(ok, nan[:, 3], ref, torch.ones(2, dtype=torch.float64), "LSE")


@pytest.mark.parametrize("h,hk,sq,sk,batch,chunks", [
    (32, 8, 1, 1280, 4, 1), (32, 8, 1, 1281, 4, 6),      # at most five steps: whole
    (32, 8, 1, 4100, 16, 1), (32, 8, 1, 4100, 15, 2),    # half the CUs busy: whole
    (32, 8, 1, 32768, 1, 32), (32, 8, 1, 1 << 20, 1, 32), (8, 1, 1, 1 << 20, 1, 64),  # one round; the most chunks
    (32, 8, 32, 4096, 1, 8), (32, 8, 32, 4096, 0, 1), (4, 4, 64, 4096, 1, 16),
])
def test_decode_split_rule(h, hk, sq, sk, batch, chunks):
    """The workspace holds rows x (64 + 2) floats per chunk of a split launch
    (256 compute units); a launch with an order flag never splits."""
    p = _params(h, hk, sq, sk)
    rows = h // hk * sq
    assert fmha.workspace_size(p, batch, 0) == (0 if chunks == 1 else batch * hk * chunks * rows * 66 * 4)
    assert fmha.workspace_size(p, batch, 0, fmha.VARIANT_REFERENCE_ORDER) == 0


@pytest.mark.parametrize("b,h,hk,sq,sk,decode", [
    (1, 16, 16, 100, 8192, True), (1, 1, 1, 200, 9000, True), (2, 8, 1, 64, 3000, True),  # one row tile per CU at most
    (16, 16, 16, 100, 8192, False), (1, 16, 4, 512, 16384, False), (1, 8, 8, 0, 4096, False)])
def test_decode_takes_small_launches(b, h, hk, sq, sk, decode):
    """Past 128 rows or 64 queries: where one 32-row tile per compute unit
    holds the launch and the estimates say so (seen in the workspace: the
    M-tile forms' are whole 34,816-byte partial results)."""
    assert (fmha.workspace_size(_params(h, hk, sq, sk), b, 0) % 34816 != 0) == decode


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("b,h,hk,sq,sk", [
    (3, 8, 2, 1, 128), (2, 16, 2, 4, 255), (1, 3, 3, 31, 257), (40, 16, 16, 2, 300),   # 640 pairs: four-wave blocks
    (1, 8, 2, 1, 1281), (2, 32, 4, 16, 4100), (1, 2, 2, 64, 5000), (1, 8, 1, 7, 20011), (20, 32, 8, 1, 2048),
    (1, 4, 4, 512, 512), (1, 6, 3, 1000, 1000), (2, 2, 1, 700, 701), (1, 2, 2, 2049, 2047), (1, 1, 1, 200, 9000)])
def test_decode_matches_float64(b, h, hk, sq, sk, causal):
    """Whole and split, from a KV cache whose tail is NaN and with O and LSE
    poisoned; the split launch twice on a dirty workspace (equal bits)."""
    g = torch.Generator(device="cuda").manual_seed(sk * 7 + sq)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    q = rnd(b, sq, h, 64).transpose(1, 2)                       # BSHD rows
    kc, vc = rnd(b, hk, sk + 37, 64), rnd(b, hk, sk + 37, 64)
    kc[:, :, sk:] = float("nan")
    vc[:, :, sk:] = float("nan")
    k, v = kc[:, :, :sk], vc[:, :, :sk]
    refs = [_f64(q[i], k[i], v[i], causal) for i in range(b)]
    o = torch.empty_strided(q.shape, q.stride(), dtype=q.dtype, device="cuda")
    lse = torch.empty(q.shape[:-1], dtype=torch.float32, device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse)
    need = fmha.workspace_size(p, b, causal)
    ws = torch.full((max(need, 256),), 0xFF, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    outs = []
    for size in (0, need, need):
        assert fmha.launch_form(p, b, causal, fmha.VARIANT_AUTO, size) == fmha.FORM_DECODE
        o.fill_(float("nan"))
        lse.fill_(float("nan"))
        fmha.fmha_fwd_d64_bf16_ws(p, b, causal, ws.data_ptr() if size else None, size, stream)
        torch.cuda.synchronize()
        for i in range(b):
            _check(o[i], lse[i], *refs[i], (size, i))
        outs.append((o.clone(), lse.clone()))
    assert torch.equal(outs[1][0], outs[2][0]) and torch.equal(outs[1][1], outs[2][1])


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("bound", [None, 700])
def test_decode_varlen_matches_float64(causal, bound):
    """Ragged key lengths (an empty one among them) and query counts; with a
    key bound below the longest sequence the last chunk takes the rest."""
    lk = [1500, 0, 1, 4097, 31, 257, 6000, 33, 1281, 2]
    lq = [1, 2, 4, 3, 1, 4, 2, 1, 0, 4]  # causal: rows with no key where lq > lk
    h, hk = 8, 2
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(h, sum(lq), 64), rnd(hk, sum(lk), 64), rnd(hk, sum(lk), 64)
    ss = [torch.from_numpy(np.cumsum([0] + l).astype(np.int32)).cuda() for l in (lq, lk)]
    o = torch.full_like(q, float("nan"))
    lse = torch.full(q.shape[:-1], float("nan"), device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse, ss[0], ss[1], 4, max(lk))
    full = fmha.workspace_size(p, len(lk), causal)
    assert full > 0
    if bound:
        p.seqlen_k = bound
    for size in (0, fmha.workspace_size(p, len(lk), causal)):
        assert fmha.launch_form(p, len(lk), causal, fmha.VARIANT_AUTO, size) == fmha.FORM_DECODE
        ws = torch.full((max(size, 256),), 0xFF, dtype=torch.uint8, device="cuda")
        o.fill_(float("nan"))
        lse.fill_(float("nan"))
        fmha.fmha_fwd_d64_bf16_ws(p, len(lk), causal, ws.data_ptr() if size else None, size,
                                  torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        a = c = 0
        for nq, nk in zip(lq, lk):
            _check(o[:, a:a + nq], lse[:, a:a + nq], *_f64(q[:, a:a + nq], k[:, c:c + nk], v[:, c:c + nk], causal),
                   (size, nq, nk))
            a, c = a + nq, c + nk


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("h,hk,lq,lk,bound", [
    (8, 2, [1, 100, 9, 128, 0, 33], [700, 300, 4000, 128, 64, 2500], 1),   # split with a workspace
    (16, 16, [3, 128, 40, 2], [900, 200, 1000, 1], 3),                     # no split, one head per KV head
    (12, 4, [64, 65, 97, 11], [2000, 1030, 70, 1500], 10),                 # the bound inside a packed tile
    (128, 128, [1, 300, 130, 200], [2048, 300, 2048, 64], 1)])             # unmasked: two M-tiles per pair block
def test_decode_varlen_rows_past_the_query_bound(h, hk, lq, lk, bound, causal):
    """seqlen_q sizes a varlen launch's grid: the rows past it that the grid's
    M-tiles reach (128 per sequence, 256 where the pair form would run) are
    computed too, and no other row is written."""
    batch = len(lq)
    g = torch.Generator(device="cuda").manual_seed(h + bound)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(h, sum(lq), 64), rnd(hk, sum(lk), 64), rnd(hk, sum(lk), 64)
    ss = [torch.from_numpy(np.cumsum([0] + l).astype(np.int32)).cuda() for l in (lq, lk)]
    o = torch.empty_like(q)
    lse = torch.empty(q.shape[:-1], device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse, ss[0], ss[1], bound, max(lk))
    tile = 256 if fmha.pick_variant(p, batch, causal) == fmha.VARIANT_PAIR else 128
    assert (tile == 256) == (h == 128 and not causal)
    need = fmha.workspace_size(p, batch, causal)
    ws = torch.full((max(need, 256),), 0xFF, dtype=torch.uint8, device="cuda")
    for size in sorted({0, need}):
        assert fmha.launch_form(p, batch, causal, fmha.VARIANT_AUTO, size) == fmha.FORM_DECODE
        o.fill_(float("nan"))
        lse.fill_(float("nan"))
        fmha.fmha_fwd_d64_bf16_ws(p, batch, causal, ws.data_ptr() if size else None, size,
                                  torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        a = c = 0
        for nq, nk in zip(lq, lk):
            n = min(nq, tile)
            ref_o, ref_l = _f64(q[:, a:a + nq], k[:, c:c + nk], v[:, c:c + nk], causal)
            _check(o[:, a:a + n], lse[:, a:a + n], ref_o[:, :n], ref_l[:, :n], (size, nq, nk))
            assert bool(torch.isnan(o[:, a + n:a + nq].float()).all()), (size, nq, nk)
            a, c = a + nq, c + nk


@pytest.mark.gpu
def test_decode_split_replays_in_a_graph():
    """A captured split launch, replayed with eager work between, equals the
    eager launch on each replay's inputs."""
    g = torch.Generator(device="cuda").manual_seed(9)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(2, 16, 1, 64), rnd(2, 4, 9000, 64), rnd(2, 4, 9000, 64)
    o = torch.empty_like(q)
    lse = torch.empty(q.shape[:-1], device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse)
    need = fmha.workspace_size(p, 2, 1)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    run = lambda: fmha.fmha_fwd_d64_bf16_ws(p, 2, 1, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for i in range(4):
        q.copy_(rnd(2, 16, 1, 64))
        ws.fill_(0xA5)
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = o.clone(), lse.clone()
        o.zero_()
        run()
        torch.cuda.synchronize()
        assert torch.equal(got[0], o) and torch.equal(got[1], lse)
        assert math.isfinite(float(lse.sum()))


@pytest.mark.gpu
def test_workspace_outlives_the_call_on_another_stream(monkeypatch):
    """fmha_fwd on a stream that is not torch's current one: its workspace is
    not handed out again while that stream still has work.  The launch is
    replaced by a recorder, so nothing is written either way."""
    q = torch.zeros(2, 16, 1, 64, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(2, 4, 9000, 64, device="cuda", dtype=torch.bfloat16)
    need = fmha.workspace_size(fmha.params_from_tensors(q, k, k, torch.empty_like(q)), 2, 1)
    assert need > 0
    seen = []
    monkeypatch.setattr(fmha, "fmha_fwd_d64_bf16_ws", lambda p, b, c, ws, n, stream: seen.append((ws, n, stream)))
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)  # ~0.1 s of bounded work
    out = fmha.fmha_fwd(q, k, k, causal=True, stream=side.cuda_stream)  # kept: a free O would join the block
    busy = not side.query()
    again = torch.empty(need, dtype=torch.uint8, device="cuda")
    (ptr, size, stream), = seen
    assert busy and (size, stream) == (need, side.cuda_stream)
    assert again.data_ptr() + need <= ptr or ptr + need <= again.data_ptr()
    torch.cuda.synchronize()
    del out


@pytest.mark.gpu
@pytest.mark.parametrize("h,hk,sq,sk", [(8, 8, 3, 9001), (4, 4, 700, 700), (4, 4, 4161, 4161), (2, 2, 9000, 9000)])
def test_static_array_gives_the_plans_bytes_or_none(h, hk, sq, sk):
    """The entry point on the static array runs what a workspace of the
    balanced plan's bytes (0 without a plan) runs, bit for bit: decode, split
    and whole, chunk and balanced."""
    g = torch.Generator(device="cuda").manual_seed(sk)
    rnd = lambda n, s: torch.randn((1, n, s, 64), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(h, sq), rnd(hk, sk), rnd(hk, sk)
    lib, stream = fmha.load_library(), torch.cuda.current_stream().cuda_stream
    outs = []
    for entry in ("ws", "noalloc"):
        o, lse = torch.full_like(q, float("nan")), torch.full(q.shape[:-1], float("nan"), device="cuda")
        p = fmha.params_from_tensors(q, k, v, o, lse)
        plan = fmha.workspace_size(p, 1, 1, fmha.VARIANT_REFERENCE_ORDER)  # the flag leaves the balanced form alone
        ws = torch.empty(max(plan, 256), dtype=torch.uint8, device="cuda")
        if entry == "ws":
            fmha.fmha_fwd_d64_bf16_ws(p, 1, 1, ws.data_ptr() if plan else None, plan, stream)
        else:
            assert lib.fmha_fwd_d64_bf16_noalloc(ctypes.byref(p), 1, 1, fmha.VARIANT_AUTO, stream) == 0
        torch.cuda.synchronize()
        outs.append((o, lse))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    _check(outs[1][0][0], outs[1][1][0], *_f64(q[0], k[0], v[0], 1), (sq, sk))
