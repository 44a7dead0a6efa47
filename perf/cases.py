"""The attention calls this library is used for, as timed cases.

Each case is one call as a program makes it: inputs and outputs resident in
GPU memory, the parameter block and the workspace prepared once (as a serving
or training loop keeps them), the launch on torch's current stream.  Kinds:

* ``prefill``  dense [B, H, S, 64] attention, square or a chunk of queries
  over a longer key range (bottom-right causal), from contiguous BHSD tensors
  or from BSHD activations viewed as BHSD;
* ``wrapper``  the same through ``fmha_fwd`` on torch tensors, outputs and
  workspace allocated per call;
* ``decode``   a few new tokens per sequence against a preallocated KV cache;
* ``varlen``   packed sequences of different lengths, self-attention;
* ``varlen_decode``  one new token per sequence against packed K/V of
  different lengths;
* ``merge``    partial results over disjoint key sets merged into one.
"""
import math

import torch

import fmha_native_amd as fmha

D = 64
DEV = "cuda:0"


def _prefill(name, b, h, hk, sq, sk, causal, lse, layout="bhsd", mult=1.0, kind="prefill"):
    return {"name": name, "kind": kind, "batch": b, "heads": h, "kv_heads": hk, "seqlen_q": sq, "seqlen_k": sk,
            "causal": causal, "lse": lse, "layout": layout, "mult": mult}


def listed():
    return [
        # the smallest call: one M-tile per head; launch and one block's latency
        _prefill("tiny_dense", 1, 2, 2, 128, 128, False, True),
        # the headline dense shape: a batch of medium prompts, no mask
        _prefill("dense_b4_h16_s2048", 4, 16, 16, 2048, 2048, False, False),
        # the headline causal shape: one long prompt, LSE kept for a backward pass
        _prefill("causal_b1_h16_s8192", 1, 16, 16, 8192, 8192, True, True),
        # one very long prompt on few heads (a tensor-parallel shard); peaked scores
        _prefill("causal_b1_h2_s40000", 1, 2, 2, 40000, 40000, True, True, mult=2.0),
        # many short sequences (classification, embedding batches): memory-bound
        _prefill("short_b128_h16_s128", 128, 16, 16, 128, 128, False, True),
        # an ordinary GQA training forward on BSHD activations with an odd length,
        # through the torch wrapper
        _prefill("wrapper_gqa_b5_s1027", 5, 16, 4, 1027, 1027, True, True, layout="bshd", kind="wrapper"),
        # chunked prefill: the next 512 tokens of a prompt over its 16,384 keys
        _prefill("chunk_gqa_sq512_sk16384", 1, 16, 4, 512, 16384, True, True),
        # a decode step: one token per sequence over a half-filled KV cache
        {"name": "decode_b16_gqa_sk4100", "kind": "decode", "batch": 16, "heads": 32, "kv_heads": 8, "new": 1,
         "seqlen_k": 4100, "cache": 8192, "lse": False},
        # a continuous-batching decode step: every sequence at another length
        {"name": "varlen_decode_n12", "kind": "varlen_decode", "heads": 16, "kv_heads": 2, "n": 12, "lo": 500,
         "hi": 16000, "lens": 7, "lse": True},
        # packed causal prompts of mixed lengths
        {"name": "varlen_causal_n8", "kind": "varlen", "heads": 16, "kv_heads": 16, "n": 8, "lo": 128, "hi": 4096,
         "lens": 42, "causal": True, "lse": True},
        # packed encoder inputs of mixed short lengths, no mask
        {"name": "varlen_dense_n64", "kind": "varlen", "heads": 12, "kv_heads": 12, "n": 64, "lo": 16, "hi": 640,
         "lens": 11, "causal": False, "lse": False},
        # partial results of four key shards of one long prompt
        {"name": "merge_n4_rows131072", "kind": "merge", "parts": 4, "rows": 131072},
    ]


MAX_FLOPS = 2.0e11   # below the largest listed case
MAX_BYTES = 3.0e8


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    h = rng.choice([2, 3, 4, 6, 8, 12, 16, 24, 32])
    hk = h // rng.choice([r for r in (1, 1, 2, 4, 8) if h % r == 0])
    return h, hk


def _draw_one(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "chunk", "wrapper", "decode", "decode", "varlen_decode",
                       "varlen", "varlen", "merge"])
    h, hk = _heads(rng)
    lse = rng.random() < 0.5
    if kind in ("prefill", "wrapper"):
        s = _log(rng, 64, 16384)
        b = max(1, min(128, _log(rng, 1024, 65536) // s))
        return _prefill("", b, h, hk, s, s, rng.random() < 0.6, lse, rng.choice(["bhsd", "bshd"]), 1.0, kind)
    if kind == "chunk":
        sq = _log(rng, 32, 2048)
        sk = max(sq, _log(rng, 1024, 32768))
        return _prefill("", rng.choice([1, 1, 2, 4]), h, hk, sq, sk, True, lse, "bhsd", 1.0)
    if kind == "decode":
        sk = _log(rng, 128, 32768)
        return {"kind": kind, "batch": _log(rng, 1, 64), "heads": h, "kv_heads": hk, "new": rng.choice([1, 1, 1, 2, 4]),
                "seqlen_k": sk, "cache": sk + rng.randrange(0, 1 + sk // 2), "lse": lse}
    if kind == "varlen_decode":
        lo = _log(rng, 32, 2000)
        return {"kind": kind, "heads": h, "kv_heads": hk, "n": _log(rng, 2, 64), "lo": lo, "hi": lo * rng.choice([2, 8, 16]),
                "lens": rng.randrange(1 << 20), "lse": lse}
    if kind == "varlen":
        lo = _log(rng, 8, 512)
        return {"kind": kind, "heads": h, "kv_heads": hk, "n": _log(rng, 2, 96), "lo": lo, "hi": lo * rng.choice([2, 4, 16]),
                "lens": rng.randrange(1 << 20), "causal": rng.random() < 0.6, "lse": lse}
    return {"kind": "merge", "parts": rng.randrange(2, 9), "rows": _log(rng, 1000, 131072)}


def draw(rng):
    while True:
        case = _draw_one(rng)
        case.pop("name", None)
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


def _lengths(case):
    """The packed sequences' (query, key) lengths."""
    lens = fmha.varlen_lengths(case["lens"], case["n"], case["lo"], case["hi"])
    return ([1] * len(lens) if case["kind"] == "varlen_decode" else lens), lens


def _causal(case):
    return case["kind"] in ("decode", "varlen_decode") or bool(case.get("causal"))


def _inputs(case, seed):
    """(q, k, v) in the layouts the call takes, bf16 on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(*shape):
        x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
        return (x * case.get("mult", 1.0)).to(torch.bfloat16)

    h, hk = case["heads"], case["kv_heads"]
    if case["kind"] in ("varlen", "varlen_decode"):
        lq, lk = _lengths(case)
        return normal(h, sum(lq), D), normal(hk, sum(lk), D), normal(hk, sum(lk), D)
    b = case["batch"]
    if case["kind"] == "decode":
        cache, sk = case["cache"], case["seqlen_k"]
        return normal(b, h, case["new"], D), normal(b, hk, cache, D)[:, :, :sk], normal(b, hk, cache, D)[:, :, :sk]
    sq, sk = case["seqlen_q"], case["seqlen_k"]
    if case["layout"] == "bshd":
        return (normal(b, sq, h, D).transpose(1, 2), normal(b, sk, hk, D).transpose(1, 2),
                normal(b, sk, hk, D).transpose(1, 2))
    return normal(b, h, sq, D), normal(b, hk, sk, D), normal(b, hk, sk, D)


def _merge_inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    n, rows = case["parts"], case["rows"]
    o = torch.randn((n, rows, D), generator=g, device=DEV, dtype=torch.float32).mul_(0.3).to(torch.bfloat16)
    lse = torch.randn((n, rows), generator=g, device=DEV, dtype=torch.float32).add_(8.0)
    # a key shard past a causal row's diagonal sees no key
    lse[1:][torch.rand((n - 1, rows), generator=g, device=DEV) < 0.05] = -math.inf
    return o, lse


def prepare(case, seed):
    if case["kind"] == "merge":
        o, lse = _merge_inputs(case, seed)
        return {"case": case, "o_parts": o, "lse_parts": lse,
                "o": torch.empty(o.shape[1:], dtype=o.dtype, device=DEV),
                "lse": torch.empty(lse.shape[1:], dtype=torch.float32, device=DEV)}
    q, k, v = _inputs(case, seed)
    st = {"case": case, "q": q, "k": k, "v": v}
    if case["kind"] == "wrapper":
        return st
    # O in q's layout, as a program that feeds the output projection keeps it
    o = torch.empty_strided(q.shape, q.stride(), dtype=q.dtype, device=DEV)
    lse = torch.empty(q.shape[:-1], dtype=torch.float32, device=DEV) if case["lse"] else None
    ssq = ssk = mq = mk = None
    batch = q.shape[0]
    if case["kind"] in ("varlen", "varlen_decode"):
        lq, lk = _lengths(case)
        batch, mq, mk = len(lq), max(lq), max(lk)
        ssq, ssk = (torch.tensor([0] + l, dtype=torch.int32).cumsum(0, dtype=torch.int32).to(DEV) for l in (lq, lk))
    p = fmha.params_from_tensors(q, k, v, o, lse, ssq, ssk, mq, mk)
    causal = int(_causal(case))
    need = fmha.workspace_size(p, batch, causal)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV) if need > 0 else None
    st.update(o=o, lse=lse, ssq=ssq, ssk=ssk, params=p, batch=batch, causal=causal, ws=ws, ws_bytes=max(need, 0))
    return st


def run(state):
    kind = state["case"]["kind"]
    if kind == "merge":
        return fmha.merge_partials(state["o_parts"], state["lse_parts"], state["o"], state["lse"])
    if kind == "wrapper":
        c = state["case"]
        o, lse = fmha.fmha_fwd(state["q"], state["k"], state["v"], causal=c["causal"], return_lse=c["lse"])
    else:
        ws = state["ws"]
        fmha.fmha_fwd_d64_bf16_ws(state["params"], state["batch"], state["causal"],
                                  ws.data_ptr() if ws is not None else None, state["ws_bytes"],
                                  torch.cuda.current_stream().cuda_stream)
        o, lse = state["o"], state["lse"]
    return (o, lse) if lse is not None else (o,)


def _pairs(sq, sk, causal):
    """Visible (query, key) pairs, bottom-right causal, sq <= sk."""
    return sq * sk - sq * (sq - 1) // 2 if causal else sq * sk


def work(case):
    if case["kind"] == "merge":
        n, rows = case["parts"], case["rows"]
        return {"bytes": (n + 1) * rows * (2 * D + 4), "flops": 2 * n * rows * D}
    h, hk = case["heads"], case["kv_heads"]
    if case["kind"] in ("varlen", "varlen_decode"):
        lq, lk = _lengths(case)
    else:
        b = case["batch"]
        lq = [case["new"] if case["kind"] == "decode" else case["seqlen_q"]] * b
        lk = [case["seqlen_k"]] * b
    tq, tk = sum(lq), sum(lk)
    pairs = sum(_pairs(a, c, _causal(case)) for a, c in zip(lq, lk))
    return {"bytes": 2 * D * 2 * (h * tq + hk * tk) + (4 * h * tq if case["lse"] else 0),
            "flops": 4 * D * h * pairs}


def tolerance(case):
    """O is rounded to bf16 once (half an ulp: 1.1e-3 relative, 2-norm) and P
    once before P.V, so two correct kernels differ by about 2e-3; peaked rows
    (inputs x2) show P's rounding more.  A merge only rounds its result."""
    return {"rel": 8e-3}


def _exact_rows(q, k, v, causal, scale, o, lse):
    """One sequence in float64: q [H, Sq, 64], k/v [Hk, Sk, 64] -> o, lse filled."""
    h, sq, _ = q.shape
    hk, sk, _ = k.shape
    rep = h // hk
    kd = k.double().transpose(1, 2).contiguous()
    vd = v.double().contiguous()
    step = max(1, (1 << 26) // max(1, rep * sk))
    for g in range(hk):
        for r0 in range(0, sq, step):
            r1 = min(sq, r0 + step)
            s = torch.matmul(q[g * rep:(g + 1) * rep, r0:r1].double().contiguous().view(-1, D), kd[g]) * scale
            s = s.view(rep, r1 - r0, sk)
            if causal:
                lim = torch.arange(r0, r1, device=DEV) + (sk - sq)
                s.masked_fill_(torch.arange(sk, device=DEV)[None, :] > lim[:, None], -math.inf)
            l = torch.logsumexp(s, dim=-1)
            p = torch.exp_(s.sub_(l[..., None]))
            o[g * rep:(g + 1) * rep, r0:r1] = torch.matmul(p.view(-1, sk), vd[g]).view(rep, r1 - r0, D)
            lse[g * rep:(g + 1) * rep, r0:r1] = l


def exact(case, seed):
    if case["kind"] == "merge":
        o, lse = _merge_inputs(case, seed)
        ld = lse.double()
        tot = torch.logsumexp(ld, dim=0)
        out = torch.zeros(o.shape[1:], dtype=torch.float64, device=DEV)
        for i in range(o.shape[0]):
            out += torch.exp(ld[i] - tot)[:, None] * o[i].double()
        return out, tot
    q, k, v = _inputs(case, seed)
    scale = 1.0 / math.sqrt(D)
    causal = _causal(case)
    o = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    lse = torch.empty(q.shape[:-1], dtype=torch.float64, device=DEV)
    if case["kind"] in ("varlen", "varlen_decode"):
        lq, lk = _lengths(case)
        a = c = 0
        for nq, nk in zip(lq, lk):
            _exact_rows(q[:, a:a + nq], k[:, c:c + nk], v[:, c:c + nk], causal, scale, o[:, a:a + nq],
                        lse[:, a:a + nq])
            a, c = a + nq, c + nk
    else:
        for b in range(q.shape[0]):
            _exact_rows(q[b], k[b], v[b], causal, scale, o[b], lse[b])
    return (o, lse) if case["lse"] else (o,)
