"""Chunk form: M-tiles of dense launches too small to fill the GPU, cut into
key chunks, against float64 attention and the other forms."""
import pytest
import torch

import fmha_native_amd as fmha
from test_decode_gpu import _check, _f64, _params

PART = 34816  # bytes of one chunk's partial result


def _tiles(sq, sk, causal):
    n = -(-sq // 128)
    if not causal:
        return [-(-sk // 64)] * n
    return [max(0, -(-min(sk, min(mt * 128 + 127, sq - 1) + sk - sq + 1) // 64)) for mt in range(n)]


@pytest.mark.parametrize("b,h,sq,sk,causal", [
    (1, 16, 512, 16384, 1), (1, 4, 4096, 4096, 1), (1, 4, 4096, 4096, 0), (1, 8, 2048, 2048, 0), (1, 1, 16384, 16384, 1),
    (2, 4, 1500, 1500, 1), (1, 24, 512, 8192, 1), (1, 3, 6000, 6000, 0), (1, 32, 300, 20000, 0)])
def test_chunk_rule(b, h, sq, sk, causal):
    """The workspace holds one slot per chunk of every cut M-tile for some
    chunk length, all chunks resident at once (two blocks per CU)."""
    need = fmha.workspace_size(_params(h, h, sq, sk), b, causal)
    slots, rest = divmod(need, PART * b * h)
    tiles = _tiles(sq, sk, causal)
    cut = {sum(c for c in (-(-t // ct) for t in tiles) if c > 1): sum(max(1, -(-t // ct)) for t in tiles)
           for ct in range(4, max(tiles))}
    assert rest == 0 and slots in cut and b * h * cut[slots] <= 512


@pytest.mark.parametrize("b,h,sq,sk,causal", [
    (4, 16, 2048, 2048, 0), (1, 16, 8192, 8192, 1), (1, 16, 1024, 1024, 0), (1, 2, 700, 700, 0), (1, 2, 128, 128, 0),
    (3, 8, 700, 700, 0)])
def test_chunk_leaves_other_launches(b, h, sq, sk, causal):
    assert fmha.workspace_size(_params(h, h, sq, sk), b, causal) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("b,h,hk,sq,sk,causal", [
    (1, 6, 2, 1500, 1500, 1), (1, 6, 6, 2500, 2501, 0), (2, 8, 4, 600, 5003, 1), (1, 2, 2, 4100, 4000, 1),  # Sq > Sk
    (1, 16, 4, 513, 8192, 0), (1, 4, 4, 4161, 4161, 1), (1, 32, 8, 257, 20011, 1)])
def test_chunk_matches_float64(b, h, hk, sq, sk, causal):
    """From BSHD storage, O and LSE poisoned, twice on a dirty workspace; a
    workspace one byte short takes another form."""
    g = torch.Generator(device="cuda").manual_seed(sk + sq)
    rnd = lambda s, n: torch.randn((b, s, n, 64), generator=g, device="cuda").to(torch.bfloat16).transpose(1, 2)
    q, k, v = rnd(sq, h), rnd(sk, hk), rnd(sk, hk)
    o = torch.empty_strided(q.shape, q.stride(), dtype=q.dtype, device="cuda")
    lse = torch.empty(q.shape[:-1], dtype=torch.float32, device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse)
    need = fmha.workspace_size(p, b, causal)
    assert need > 0 and need % PART == 0
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    refs = [_f64(q[i], k[i], v[i], causal) for i in range(b)]
    outs = []
    for size in (need, need, need - 1):
        assert (fmha.launch_form(p, b, causal, fmha.VARIANT_AUTO, size) == fmha.FORM_CHUNK) == (size == need)
        o.fill_(float("nan"))
        lse.fill_(float("nan"))
        fmha.fmha_fwd_d64_bf16_ws(p, b, causal, ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        for i in range(b):
            _check(o[i], lse[i], *refs[i], (size, i))
        outs.append((o.clone(), lse.clone()))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.gpu
def test_chunk_replays_in_a_graph():
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda s: torch.randn((1, 16, s, 64), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(400), rnd(6000), rnd(6000)
    o = torch.empty_like(q)
    lse = torch.empty(q.shape[:-1], device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse)
    need = fmha.workspace_size(p, 1, 1)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    run = lambda: fmha.fmha_fwd_d64_bf16_ws(p, 1, 1, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(3):
        q.copy_(rnd(400))
        ws.fill_(0xA5)
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = o.clone(), lse.clone()
        o.zero_()
        run()
        torch.cuda.synchronize()
        assert torch.equal(got[0], o) and torch.equal(got[1], lse)
