"""GPU parity of the elementwise / attention operators against the oracle."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("n", [4, 768, 2048, 5000])
def test_rmsnorm_layernorm(gpu, n):
    from smallmind_amd.quantization import layernorm, rmsnorm
    rng = np.random.default_rng(n)
    x = rng.normal(0, 2, (3, n)).astype(np.float32)
    g = rng.normal(1, 0.2, n).astype(np.float32)
    b = rng.normal(0, 0.2, n).astype(np.float32)
    assert rel_err(rmsnorm(_dev(x), _dev(g)).cpu().numpy(), O.rmsnorm(x, g)) < 2e-6
    assert rel_err(layernorm(_dev(x), _dev(g), _dev(b)).cpu().numpy(), O.layernorm(x, g, b)) < 2e-6


def test_rmsnorm_reference_values(gpu):
    from smallmind_amd.quantization import rmsnorm
    x = np.array([[0.5, 1.5, 2.5, 3.5]], np.float32)
    g = np.array([1.2, 0.8, 1.5, 0.5], np.float32)
    inv = 1.0 / np.sqrt((0.25 + 2.25 + 6.25 + 12.25) / 4 + 1e-5)
    assert np.allclose(rmsnorm(_dev(x), _dev(g)).cpu().numpy(), g * x * inv, atol=1e-4)


def test_rope_tables_equal_oracle_and_apply(gpu):
    from smallmind_amd.quantization import rope_, rope_tables
    c, s = rope_tables(300, 64, 10000.0)
    oc, os_ = O.rope_tables(300, 64, 10000.0)
    assert np.array_equal(c, oc) and np.array_equal(s, os_)
    rng = np.random.default_rng(0)
    x = rng.normal(0, 1, (4, 6, 64)).astype(np.float32)
    got = rope_(_dev(x), 37, _dev(c), _dev(s)).cpu().numpy()
    assert np.array_equal(got, O.rope_apply(x, 37, oc, os_))
    got0 = rope_(_dev(x), 0, _dev(c), _dev(s)).cpu().numpy()
    assert np.array_equal(got0[:, 0], x[:, 0])   # position 0 is the identity


@pytest.mark.parametrize("seq,kseq,off", [(1, 1, 0), (1, 700, 699), (5, 9, 4), (3, 3000, 2997)])
def test_scale_mask_softmax(gpu, seq, kseq, off):
    from smallmind_amd.quantization import scale_mask_softmax_
    s = np.random.default_rng(kseq).normal(0, 3, (seq, kseq)).astype(np.float32)
    got = scale_mask_softmax_(_dev(s), 0.125, off).cpu().numpy()
    ref = O.scale_mask_softmax(s, 0.125, off)
    assert np.abs(got - ref).max() < 1e-6
    for i in range(seq):
        assert np.all(got[i, off + i + 1:] == 0)


@pytest.mark.parametrize("H,Hkv,hd,npos", [(32, 4, 64, 1), (32, 4, 64, 513), (12, 12, 64, 160),
                                           (32, 32, 64, 300), (8, 2, 128, 1000), (32, 4, 64, 4096),
                                           (12, 4, 32, 33), (16, 1, 16, 95), (4, 4, 128, 31),
                                           (16, 2, 64, 767), (32, 4, 64, 1500), (8, 8, 64, 2500),
                                           (32, 4, 64, 4608), (4, 2, 64, 5000)])
def test_attention_decode_vs_oracle(gpu, H, Hkv, hd, npos):
    from smallmind_amd.quantization import attention_decode
    rng = np.random.default_rng(npos)
    ctx = npos + 7
    q = rng.normal(0, 1, (H, hd)).astype(np.float32)
    kc = rng.normal(0, 1, (Hkv, ctx, hd)).astype(np.float32)
    vc = rng.normal(0, 1, (Hkv, ctx, hd)).astype(np.float32)
    kt = np.ascontiguousarray(kc.transpose(0, 2, 1))   # the backend keeps K dimension-major
    got = attention_decode(_dev(q), _dev(kt), _dev(vc), H, Hkv, hd, ctx, npos).cpu().numpy()
    scale = np.float32(1.0) / np.sqrt(np.float32(hd))
    ref = np.empty((H, hd), np.float32)
    for h in range(H):
        kv = h // (H // Hkv)
        sc = (kc[kv, :npos].astype(np.float64) @ q[h].astype(np.float64)).astype(np.float32)[None]
        p = O.scale_mask_softmax(sc, float(scale), cache_off=npos - 1)[0]
        ref[h] = p.astype(np.float64) @ vc[kv, :npos].astype(np.float64)
    assert rel_err(got.reshape(H, hd), ref) < 1e-5


@pytest.mark.parametrize("H,Hkv,hd,npos,ctx", [(32, 4, 64, 1, 4), (32, 4, 64, 160, 160), (12, 12, 64, 255, 256),
                                               (32, 4, 64, 256, 260), (8, 2, 64, 257, 512), (32, 4, 64, 511, 512),
                                               (32, 4, 64, 700, 768), (32, 4, 64, 768, 768), (16, 4, 64, 769, 1024),
                                               (32, 8, 64, 1024, 1024), (12, 4, 32, 600, 604), (16, 1, 16, 95, 100),
                                               (4, 4, 32, 1000, 1000)])
def test_attention_decode_one_launch_vs_oracle(gpu, H, Hkv, hd, npos, ctx):
    """Contexts up to 1024 positions with 16-byte aligned cache rows (ctx % 4 == 0) run as one
    launch that computes the scores inside the P.V workgroups.  Cache entries past n_pos hold
    NaN: they must never reach the output."""
    from smallmind_amd.quantization import attention_decode
    rng = np.random.default_rng(npos * 3 + hd)
    q = rng.normal(0, 1, (H, hd)).astype(np.float32)
    kc = rng.normal(0, 1, (Hkv, ctx, hd)).astype(np.float32)
    vc = rng.normal(0, 1, (Hkv, ctx, hd)).astype(np.float32)
    kc[:, npos:] = np.nan
    vc[:, npos:] = np.nan
    kt = np.ascontiguousarray(kc.transpose(0, 2, 1))
    got = attention_decode(_dev(q), _dev(kt), _dev(vc), H, Hkv, hd, ctx, npos).cpu().numpy().reshape(H, hd)
    scale = np.float32(1.0) / np.sqrt(np.float32(hd))
    ref = np.empty((H, hd), np.float32)
    for h in range(H):
        kv = h // (H // Hkv)
        sc = (kc[kv, :npos].astype(np.float64) @ q[h].astype(np.float64)).astype(np.float32)[None]
        p = O.scale_mask_softmax(sc, float(scale), cache_off=npos - 1)[0]
        ref[h] = p.astype(np.float64) @ vc[kv, :npos].astype(np.float64)
    assert np.isfinite(got).all()
    assert rel_err(got, ref) < 1e-5


@pytest.mark.parametrize("H,Hkv,p0,n", [(32, 4, 0, 37), (32, 4, 300, 64), (12, 12, 5, 33),
                                        (16, 1, 0, 20), (8, 8, 1000, 17), (4, 2, 0, 1),
                                        (32, 32, 255, 256), (32, 4, 3840, 256), (2, 2, 16, 48)])
def test_attention_prefill_vs_oracle(gpu, H, Hkv, p0, n):
    """Causal attention of n tokens at positions p0.. over the cache (MultiHeadAttention T > 1).
    Cache entries past the last token hold NaN: they must never reach the output."""
    from smallmind_amd.quantization import attention_prefill
    hd = 64
    rng = np.random.default_rng(p0 * 7 + n)
    ctx = p0 + n + 9
    q = rng.normal(0, 1, (n, H, hd)).astype(np.float32)
    kc = rng.normal(0, 1, (Hkv, ctx, hd)).astype(np.float32)
    vc = rng.normal(0, 1, (Hkv, ctx, hd)).astype(np.float32)
    kc[:, p0 + n:] = np.nan
    vc[:, p0 + n:] = np.nan
    kt = np.ascontiguousarray(kc.transpose(0, 2, 1))   # the backend keeps K dimension-major
    got = attention_prefill(_dev(q), _dev(kt), _dev(vc), H, Hkv, hd, ctx, p0, n).cpu().numpy()
    got = got.reshape(n, H, hd)
    scale = np.float32(1.0) / np.sqrt(np.float32(hd))
    ref = np.empty((n, H, hd), np.float32)
    kl = p0 + n
    for h in range(H):
        kv = h // (H // Hkv)
        sc = (q[:, h].astype(np.float64) @ kc[kv, :kl].astype(np.float64).T).astype(np.float32)
        p = O.scale_mask_softmax(sc, float(scale), cache_off=p0)
        ref[:, h] = p.astype(np.float64) @ vc[kv, :kl].astype(np.float64)
    assert np.isfinite(got).all()
    assert rel_err(got, ref) < 2e-5


@pytest.mark.parametrize("H,Hkv,p0,n", [(32, 4, 0, 401),     # 128-row workgroups of 16 tokens, the last with one
                                        (32, 32, 37, 420),   # 128 tokens per workgroup, ragged; keys split 8 + 7 tiles
                                        (32, 1, 95, 405),    # 4 tokens per workgroup
                                        (12, 12, 5, 1070)])
def test_attention_prefill_many_rows_vs_float64(gpu, H, Hkv, p0, n):
    """The 128-row kernel (12800 query rows and more): against float64 with the same FastExp, cache
    entries past the last token NaN, q at an address that is only 4-byte aligned.  Bound: the op
    bound of this file."""
    import torch
    from smallmind_amd.quantization import attention_prefill
    hd, ctx, kl = 64, p0 + n + 3, p0 + n
    g = torch.Generator("cuda").manual_seed(H * 7 + n)
    q = torch.randn(n * H * hd + 1, device="cuda", generator=g)[1:].reshape(n, H, hd)
    k = torch.randn(Hkv, hd, ctx, device="cuda", generator=g)
    v = torch.randn(Hkv, ctx, hd, device="cuda", generator=g)
    k[:, :, kl:] = float("nan")
    v[:, kl:] = float("nan")
    got = attention_prefill(q, k, v, H, Hkv, hd, ctx, p0, n).reshape(n, H, hd).double()
    seen = torch.arange(kl, device="cuda")[None] <= p0 + torch.arange(n, device="cuda")[:, None]
    for h in range(H):
        kv = h // (H // Hkv)
        s = (q[:, h].double() @ k[kv, :, :kl].double() / 8.0).masked_fill(~seen, -float("inf"))
        x = (s - s.amax(1, keepdim=True)).clamp(-87.3, 88.7)
        e = torch.where(seen, (1 + x * 0.5 + x * x * 0.08333333) / (1 - x * 0.5 + x * x * 0.08333333), 0.0)
        ref = e @ v[kv, :kl].double() / e.sum(1, keepdim=True)
        assert torch.isfinite(got[:, h]).all()
        assert float((got[:, h] - ref).abs().max() / ref.abs().max()) < 2e-5


def test_silu_mul_gelu(gpu):
    from smallmind_amd.quantization import gelu, silu_mul
    rng = np.random.default_rng(1)
    g = rng.normal(0, 4, 10001).astype(np.float32)
    u = rng.normal(0, 1, 10001).astype(np.float32)
    assert np.allclose(silu_mul(_dev(g), _dev(u)).cpu().numpy(), O.silu_mul(g, u), rtol=2e-6, atol=1e-7)
    x = rng.normal(0, 3, 10001).astype(np.float32)
    assert np.allclose(gelu(_dev(x)).cpu().numpy(), O.gelu(x), rtol=1e-6, atol=1e-7)


def test_argmax_lowest_index_on_ties(gpu):
    from smallmind_amd.quantization import argmax
    rng = np.random.default_rng(2)
    for n in (1, 63, 32000, 50257):
        v = rng.normal(0, 1, n).astype(np.float32)
        assert argmax(_dev(v)) == int(np.argmax(v))
        if n > 10:
            v[n // 3] = v[n - 2] = v.max() + 1
            assert argmax(_dev(v)) == n // 3


SAMPLING = [dict(), dict(temperature=0.8, top_k=40, top_p=0.95), dict(temperature=0.7, min_p=0.05),
            dict(top_k=1), dict(top_p=0.1), dict(temperature=1.3, top_p=0.5, min_p=0.01),
            dict(repetition_penalty=1.3, presence_penalty=0.4, frequency_penalty=0.2, top_k=100),
            dict(repetition_penalty=1.1, repetition_window=20, temperature=0.5)]


@pytest.mark.parametrize("n", [1000, 32000, 50257])
@pytest.mark.parametrize("opts", range(len(SAMPLING)))
def test_sample_vs_oracle(gpu, n, opts):
    """smx_sample against the oracle pipeline: the final distributions agree to the rounding of
    the normalising sums (the reference adds up to 50K probabilities one by one in fp32, about
    3e-5 relative at this size; the kernel sums in a tree), and the drawn ids are identical
    except where u falls within that rounding of a CDF step."""
    import torch
    from smallmind_amd.quantization import sample
    kw = SAMPLING[opts]
    rng = np.random.default_rng(n + opts)
    logits = rng.normal(0, 3, n).astype(np.float32)
    ctx = rng.integers(0, n, 300).astype(np.int32)
    ctx[-40:] = ctx[-60:-20]   # repeats inside the window
    okw = dict(kw)
    if "repetition_window" in okw:
        okw["window"] = okw.pop("repetition_window")
    for u in rng.random(6):
        tok, p = sample(_dev(logits), u, context=_dev(ctx), **kw)
        otok, op = O.sample(logits, u, context=ctx, **okw)
        p = p.cpu().numpy()
        # kept sets: equal unless the top-p cumulative sum sits within rounding of the cutoff
        if not np.array_equal(p > 0, op > 0):
            base = O.sample(logits, 0.5, context=ctx, **{k: v for k, v in okw.items() if k not in ("top_p", "min_p")})[1]
            c = np.cumsum(np.sort(base[op > 0])[::-1].astype(np.float64))
            assert abs(c[-1] - kw.get("top_p", 1.0)) < 2e-4 or abs(c[-2] - kw.get("top_p", 1.0)) < 2e-4
            continue
        assert np.abs(p - op).max() <= 2e-4 * max(op.max(), 1e-30), (u, np.abs(p - op).max())
        cdf = np.cumsum(op.astype(np.float64))
        if np.min(np.abs(cdf - u)) > 2e-4:
            assert tok == otok, (u, tok, otok)


def test_attention_prefill_many_rows_infinities(gpu):
    """Infinite and nearly overflowing cache entries, which have no finite bf16 parts, give what the
    fp32 kernel of short runs gives for the same tokens (the op bound of this file)."""
    import torch
    from smallmind_amd.quantization import attention_prefill
    H, Hkv, hd, n, ctx = 32, 4, 64, 416, 420
    g = torch.Generator("cuda").manual_seed(5)
    q = torch.randn(n, H, hd, device="cuda", generator=g)
    k = torch.randn(Hkv, hd, ctx, device="cuda", generator=g)
    v = torch.randn(Hkv, ctx, hd, device="cuda", generator=g)
    v[0, 5, 3] = float("inf")
    v[1, 40, 7] = 3.4e38
    k[2, 11, 9] = float("inf")
    k[:, :, n:] = float("inf")    # not written: read by no token
    v[:, n:] = float("inf")
    got = attention_prefill(q, k, v, H, Hkv, hd, ctx, 0, n).reshape(n, H, hd)
    few = attention_prefill(q[n - 16:].contiguous(), k, v, H, Hkv, hd, ctx, n - 16, 16).reshape(16, H, hd)
    got = got[n - 16:]
    assert torch.isinf(few[:, :8, 3]).all() and torch.isfinite(few[:, 24:]).all()
    fin = torch.isfinite(few)
    assert torch.equal(fin, torch.isfinite(got)) and torch.equal(got.isnan(), few.isnan())
    assert torch.equal(got[few.isinf()], few[few.isinf()])
    err = (got - few).abs().double() / few.abs().double().clamp(min=1.0)
    assert float(err[fin].max()) < 2e-5


def _sample64(l, ctx, temperature=1.0, top_k=0, top_p=1.0, min_p=0.0, repetition_penalty=1.0, frequency_penalty=0.0,
              repetition_window=0):
    """Float32 logits stages, float64 probabilities: one array for every cutoff that rounding allows.  The
    fp32 sum behind top-p is within 1e-5 of the exact one (of about 1: a tree of depth 16 over expf's 2 ulp and
    a division), and so is a probability of the min-p threshold; between them they may fall either way."""
    l, f = l.copy(), np.float32
    w = ctx[len(ctx) - min(len(ctx), repetition_window or 256):]
    for t in np.unique(w):
        if repetition_penalty != 1.0:
            l[t] = l[t] / f(repetition_penalty) if l[t] > 0 else l[t] * f(repetition_penalty)
        l[t] -= f(np.sum(w == t)) * f(frequency_penalty)
    l = l * (f(1) / f(temperature))
    if 0 < top_k < len(l):
        l = np.where(l >= np.sort(l)[len(l) - top_k], l, f(-np.inf))
    e = np.exp(l.astype(np.float64) - l.max())
    out = [e / e.sum()]
    if top_p < 1.0:
        v, c = np.unique(out[0], return_counts=True)
        v, cum = v[::-1], np.cumsum((v * c)[::-1])
        lo, hi = (int(np.argmax(cum >= top_p + d)) if cum[-1] >= top_p + d else len(v) - 1 for d in (-1e-5, 1e-5))
        out = [np.where(out[0] >= v[i], out[0], 0.0) for i in range(lo, hi + 1)]
        out = [p / p.sum() for p in out]
    if min_p > 0.0:
        out = [np.where(p < p.max() * min_p * d, 0.0, p) for p in out for d in (1 - 1e-5, 1, 1 + 1e-5)]
        out = [p / p.sum() for p in out]
    return out


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 4097, 32000, 32768, 32769, 50257, 65536, 65537])
@pytest.mark.parametrize("data", ["spread", "flat", "ties", "zeros", "masked"])
def test_sample_paths_vs_float64(gpu, n, data):
    """Values in LDS, in LDS and registers, and in memory; cutoffs found in the list of candidates and
    outside of it (flat: more candidates than it holds; ties across the cutoff; fewer finite logits than
    top-k; +0 and -0 at the cutoff).  Bound: sums of up to 65537 fp32 terms in a tree of depth 16 and
    expf, 32 roundings of 2^-24 and the 2 ulp of expf on each side."""
    from smallmind_amd.quantization import sample
    rng = np.random.default_rng(n + len(data))
    l = rng.normal(0, {"flat": 0.05}.get(data, 3.0), n).astype(np.float32)
    if data == "ties":
        l = np.round(l)
    if data == "zeros":
        l = np.where(rng.random(n) < 0.5, np.float32(0.0), np.float32(-0.0)) - (l > 1) * np.float32(1.0)
        l[: n // 2] = -np.float32(0.0)
    if data == "masked":
        l[rng.permutation(n)[20:]] = -np.inf
    ctx = rng.integers(0, n, 2500).astype(np.int32)
    for kw in [dict(top_k=40, top_p=0.9, min_p=0.02, temperature=0.8, repetition_penalty=1.1),
               dict(top_k=192), dict(top_k=193, top_p=0.5), dict(top_p=0.3), dict(top_p=0.95, frequency_penalty=0.1),
               dict(min_p=0.1, repetition_penalty=1.2, repetition_window=2400), dict(top_k=1)]:
        for u in (0.0, float(rng.random()), 1.0 - 2.0 ** -40):
            tok, p = sample(_dev(l), u, context=_dev(ctx), **kw)
            p = p.cpu().numpy().astype(np.float64)
            allowed = _sample64(l, ctx, **kw) if u == 0.0 else allowed
            same = [ref for ref in allowed if np.array_equal(p > 0, ref > 0)]
            assert same, (kw, (p > 0).sum(), [(ref > 0).sum() for ref in allowed])
            ref = same[0]
            assert np.abs(p - ref).max() <= 2 ** -18 * ref.max(), kw
            cdf = np.cumsum(p)
            if u == 0.0:
                assert tok == 0
            elif u > cdf[-1]:
                assert tok == n - 1
            else:
                assert p[tok] > 0 and cdf[tok] >= u - 1e-12 and cdf[tok] - p[tok] < u + 1e-12, (kw, u, tok)


def test_sample_infinite_logit(gpu):
    """+infinity at the top: its exponential is not a number, no probability is kept and the draw falls
    back to the last token."""
    from smallmind_amd.quantization import sample
    l = np.random.default_rng(1).normal(0, 3, 32000).astype(np.float32)
    l[77] = np.inf
    for kw in (dict(top_k=40, top_p=0.9), dict(top_p=0.9)):
        tok, p = sample(_dev(l), 0.5, **kw)
        assert tok == 31999 and not bool((p != 0).any())


@pytest.mark.parametrize("n", [1000, 40000, 65536, 65537, 90001])
def test_sample_in_place(gpu, n):
    """probs may be the logits' own buffer: the same token and the same bits as in one of its own, with
    the values on the compute unit and, above 65536, in that buffer."""
    import ctypes

    import torch

    from smallmind_amd._lib import SamplingC, call
    rng = np.random.default_rng(n)
    l = _dev(rng.normal(0, 3, n).astype(np.float32))
    ctx = _dev(rng.integers(0, n, 300).astype(np.int32))
    for temp, top_k, top_p, rep in ((0.7, 40, 0.9, 1.3), (0.7, 0, 1.0, 1.3), (1.0, 0, 0.8, 1.3), (0.7, 0, 0.8, 1.0)):
        p = SamplingC(temp, top_k, top_p, 0.0, rep, 0.0, 0.1 * (rep != 1.0), 0)
        got = []
        for own in (False, True):
            src = l.clone()
            dst = src if own else torch.empty_like(src)
            tok = torch.empty(1, dtype=torch.int32, device="cuda")
            call("smx_sample", src.data_ptr(), n, ctx.data_ptr(), ctx.numel(), ctypes.byref(p), 0.37, dst.data_ptr(),
                 tok.data_ptr(), torch.cuda.current_stream().cuda_stream)
            got.append((int(tok.item()), dst))
        assert got[0][0] == got[1][0], (temp, top_k, top_p, rep)
        assert torch.equal(got[0][1], got[1][1]), (temp, top_k, top_p, rep)


def test_stream_read_runs_and_checks_its_size(gpu):
    """smx_stream_read (the bench's streaming-read ceiling) reads device memory without writing
    it, and refuses sizes that are not a positive multiple of 16 bytes."""
    import torch

    from smallmind_amd._lib import SmxError, call
    buf = torch.arange(1 << 18, dtype=torch.int32, device="cuda")
    before = buf.clone()
    s = torch.cuda.current_stream().cuda_stream
    for n in (16, 4096, buf.numel() * 4):
        call("smx_stream_read", buf.data_ptr(), n, s)
    torch.cuda.synchronize()
    assert torch.equal(buf, before)
    for n in (0, 24, 4095):
        with pytest.raises(SmxError):
            call("smx_stream_read", buf.data_ptr(), n, s)
