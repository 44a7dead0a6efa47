"""Wide form (64 query rows per wave): automatic launches on grids it takes,
against float64 attention on sampled heads and the regular form everywhere."""
import pytest
import torch

import fmha_native_amd as fmha
from test_decode_gpu import _check, _f64


def _run(q, k, v, causal, variant):
    o = torch.full_like(q, float("nan"))
    lse = torch.full(q.shape[:-1], float("nan"), device="cuda")
    p = fmha.params_from_tensors(q, k, v, o, lse)
    form = fmha.FORM_WIDE if variant == fmha.VARIANT_AUTO else variant
    assert fmha.launch_form(p, q.shape[0], causal, variant) == form
    fmha.fmha_fwd_d64_bf16(p, q.shape[0], causal, torch.cuda.current_stream().cuda_stream, variant)
    torch.cuda.synchronize()
    return o, lse


@pytest.mark.gpu
@pytest.mark.parametrize("rising", [False, True])
@pytest.mark.parametrize("b,h,hk,sq,sk,causal", [
    (64, 8, 8, 256, 256, 0), (64, 8, 2, 225, 1001, 0), (32, 16, 16, 801, 193, 0),  # a dead wave; a dead M-tile
    (64, 8, 8, 129, 449, 0), (64, 8, 8, 256, 511, 0),                              # every remainder of four tiles
    (32, 16, 4, 256, 4001, 1), (1, 94, 94, 2600, 2600, 1), (3, 32, 8, 2563, 2563, 1)])
def test_wide_matches_regular_and_float64(b, h, hk, sq, sk, causal, rising):
    """Also with scores that rise by ~23 (log2 units) per 32 keys, which moves
    every row's reference maximum at every step.  Two bf16 roundings apart:
    the benchmark rule 1e-2 + 1e-2|O| between the forms."""
    g = torch.Generator(device="cuda").manual_seed(sq + sk)
    rnd = lambda n, s: torch.randn((b, n, s, 64), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v = rnd(h, sq), rnd(hk, sk), rnd(hk, sk)
    if rising:
        q[..., 0] = 4.0
        k[..., 0] = torch.arange(sk, device="cuda").to(torch.bfloat16)
    o, lse = _run(q, k, v, causal, fmha.VARIANT_AUTO)
    o_r, lse_r = _run(q, k, v, causal, fmha.VARIANT_REGULAR)
    d = (o.float() - o_r.float()).abs()
    assert bool((d <= 1e-2 + 1e-2 * o_r.float().abs()).all()), float(d.max())  # NaN misses
    if not rising:  # no row re-frames: the same operations in the same order
        assert torch.equal(o, o_r) and torch.equal(lse, lse_r)
    # LSE: fp32 sums of the same weights in another order, on values up to |LSE|
    assert bool(((lse - lse_r).abs() <= 1e-4 + 1e-6 * lse_r.abs()).all())
    for i, j in ((0, 0), (b - 1, h - 1)):
        kv = j // (h // hk)
        ref = _f64(q[i, j:j + 1], k[i, kv:kv + 1], v[i, kv:kv + 1], causal)
        _check(o[i, j:j + 1], lse[i, j:j + 1], *ref, (i, j))
