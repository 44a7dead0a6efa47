"""Last M-tiles with fewer live rows than a block has waves for: the waves
without rows compute nothing and change no other row's bits."""
import pytest
import torch

import fmha_native_amd as fmha

FORMS = {"regular": fmha.VARIANT_REGULAR, "splitkv": fmha.VARIANT_SPLITKV, "pair": fmha.VARIANT_PAIR,
         "short": fmha.VARIANT_SHORT}


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("form", list(FORMS))
def test_dead_waves_change_no_row(form, causal):
    """Rows 0 .. n-1 equal, bit for bit, those of the same queries followed by
    more rows (causal: as many more keys, so that every row sees the same
    ones), for every count of live waves and key-tile remainder; O past row n
    stays unwritten."""
    g = torch.Generator(device="cuda").manual_seed(17)
    rnd = lambda s: torch.randn((2, 3, s, 64), generator=g, device="cuda").to(torch.bfloat16)
    full = 512
    for n in (1, 32, 33, 65, 97, 129, 161, 225, 257, 300):
        sk = n + 40 if causal else 40 * (n % 7) + 33
        k, v = rnd(sk + full - n), rnd(sk + full - n)
        q = rnd(full)
        outs = []
        for rows, keys in ((n, sk), (full, sk + full - n if causal else sk)):
            o = torch.full_like(q, float("nan"))
            p = fmha.params_from_tensors(q[:, :, :rows], k[:, :, :keys], v[:, :, :keys], o[:, :, :rows])
            fmha.fmha_fwd_d64_bf16(p, 2, causal, torch.cuda.current_stream().cuda_stream,
                                   FORMS[form] | fmha.VARIANT_REFERENCE_ORDER)
            torch.cuda.synchronize()
            outs.append(o)
        assert bool(outs[0][:, :, n:].isnan().all()), n
        if form != "splitkv" or not causal:  # a longer M-tile's key halves meet elsewhere
            assert torch.equal(outs[0][:, :, :n], outs[1][:, :, :n]), n
        else:
            d = (outs[0][:, :, :n].float() - outs[1][:, :, :n].float()).abs()
            assert bool((d <= 1e-2 + 1e-2 * outs[1][:, :, :n].float().abs()).all()), n  # NaN misses
