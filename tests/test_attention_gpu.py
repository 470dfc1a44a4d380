"""The HIP attention layer core (``kernels/fused_attention.py``) against the torch
form it stands in for (``kernels/_eager.py``).

QK-norm, RoPE and the cache rows are the same bf16 roundings of the same
values: the only freedom is the fp32 sum of squares, whose order may move the
scale by an ulp of fp32 and so flip a bf16 rounding (an ulp, 2^-8 of the value)
now and then; a flipped q moves a score, and so a row (``_check``). Where q is
exact (the C entry point without norm weights, RoPE by 0) the output is rounded
once from fp32, so against the fp64 softmax over the kernel's own cache rows it
is within half a bf16 ulp plus fp32 evaluation error: |y - t| <= 2^-8 |t| + 1e-5
max|v|, the bound of ``test_attend_cpu.py``.
"""

from __future__ import annotations

import pytest
import torch

from llms_amd.kernels import _eager
from llms_amd.kernels.fused_attention import attention_core

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _inputs(seed, B, T, Hq, Hk, D, S, pos, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    n = (Hq + 2 * Hk) * D
    y = (r(B, T, n) * scale).bfloat16()
    q, k, v = y.split([Hq * D, Hk * D, Hk * D], dim=-1)
    qn, kn = _eager.RMSNorm(D).to(DEV, torch.bfloat16), _eager.RMSNorm(D).to(DEV, torch.bfloat16)
    with torch.no_grad():
        qn.weight.copy_(1 + 0.1 * r(D))
        kn.weight.copy_(1 + 0.1 * r(D))
    cos, sin = (t.to(DEV, torch.bfloat16) for t in _eager.build_rope_tables(D, S, 1e4))
    ck, cv = (r(B + 1, Hk, S, D).bfloat16() for _ in range(2))
    ck[:, :, pos:] = float("nan")  # slots not written yet may hold anything
    cv[:, :, pos:] = float("nan")
    return dict(q=q, k=k, v=v, q_norm=qn, k_norm=kn, num_heads=Hq, cache_k=ck, cache_v=cv,
                cos=cos[pos:pos + T], sin=sin[pos:pos + T], start_pos=pos)


def _eager_rows(c, B, T, Hq, Hk, D):
    """q, k, v [B, H, T, D] as the torch form rotates and normalises them."""
    q = c["q_norm"](c["q"].view(B, T, Hq, D)).transpose(1, 2)
    k = c["k_norm"](c["k"].view(B, T, Hk, D)).transpose(1, 2)
    q, k = _eager.apply_rope(q, k, c["cos"], c["sin"])
    return q, k, c["v"].view(B, T, Hk, D).transpose(1, 2)


def _near_bf16(a, b, share=0.01):
    """Equal in all but `share` of the elements. Where a flipped rounding of a
    normalised value (its own and its weight product's, 2^-8 of it each) is
    carried through RoPE's two products and their sum (2^-8 each), the element
    moves by at most 2^-6 of the size of its rotate-half pair, also where the
    two products cancel."""
    d = (a.float() - b.float()).abs()
    h = b.shape[-1] // 2
    pair = torch.hypot(b[..., :h].float(), b[..., h:].float())
    assert bool((d <= 2.0 ** -6 * torch.cat([pair, pair], dim=-1)).all())
    assert (d > 0).float().mean().item() <= share


def _check(c, B, T, Hq, Hk, D, y):
    """y, and the cache after the call, against the torch form's values."""
    pos, end = c["start_pos"], c["start_pos"] + T
    q, k, v = _eager_rows(c, B, T, Hq, Hk, D)
    _near_bf16(c["cache_k"][:B, :, pos:end], k)
    assert torch.equal(c["cache_v"][:B, :, pos:end], v)
    full_k, full_v = (t[:B, :, :end].double().repeat_interleave(Hq // Hk, dim=1)
                      for t in (c["cache_k"], c["cache_v"]))
    s = torch.matmul(q.double(), full_k.transpose(-2, -1).contiguous()) * D ** -0.5
    hide = torch.arange(end, device=DEV)[None] > torch.arange(pos, end, device=DEV)[:, None]
    t = torch.matmul(torch.softmax(s.masked_fill(hide, float("-inf")), -1), full_v)
    t = t.transpose(1, 2).reshape(B, T, Hq * D)
    d = (y.double() - t).abs()
    rel = (d.norm() / t.norm()).item()
    print(f"rel {rel:.2e} max {d.max().item():.2e}")
    # a flipped bf16 rounding of q moves a score, and so a row, by up to 2^-8
    # of its size: the bound of one rounding in the 2-norm, twice that per value
    assert rel <= 2.0 ** -8
    assert bool((d <= 2.0 ** -7 * t.abs() + 2.0 ** -8 * full_v.abs().max()).all())


# (B, T, Hq, Hk, D, S, pos): one token and verify steps (1-64 query rows per kv
# head), the first row count past them, ragged prompts, later chunks; chunk and
# tile edges of 32, 64 and 128 keys; group sizes 1, 2, 4, 5; a full cache
CASES = [
    (1, 1, 32, 8, 128, 64, 0), (1, 1, 32, 8, 128, 4096, 31), (2, 1, 16, 8, 128, 300, 128),
    (1, 1, 8, 8, 64, 129, 128), (3, 1, 10, 2, 64, 513, 511), (1, 1, 32, 8, 128, 4096, 4095),
    (1, 4, 32, 8, 128, 2048, 1000), (2, 9, 16, 8, 64, 700, 33), (1, 5, 32, 8, 128, 200, 60),
    (1, 16, 32, 8, 128, 256, 0), (1, 17, 32, 8, 128, 256, 0), (1, 33, 4, 4, 64, 100, 30),
    (1, 65, 8, 8, 128, 200, 127), (1, 100, 32, 8, 128, 100, 0), (2, 129, 10, 2, 64, 300, 5),
    (1, 1000, 32, 8, 128, 1024, 0), (1, 70, 16, 8, 128, 3000, 2900), (1, 2048, 8, 2, 128, 2048, 0),
]


@pytest.mark.parametrize("B,T,Hq,Hk,D,S,pos", CASES)
def test_matches_fp64_attention(B, T, Hq, Hk, D, S, pos):
    print(B, T, Hq, Hk, D, S, pos, flush=True)
    c = _inputs(T + pos, B, T, Hq, Hk, D, S, pos)
    before = c["cache_v"][B].clone().view(torch.int16)
    with torch.inference_mode():
        y = attention_core(**c)
        _check(c, B, T, Hq, Hk, D, y)
        # the spare sequence and the slots past the tokens are untouched
        assert torch.equal(c["cache_v"][B].view(torch.int16), before)
        assert bool(c["cache_k"][:, :, pos + T:].isnan().all())
        # a device position: the same values over the whole cache
        yd = attention_core(**dict(c, start_pos=torch.tensor(pos, device=DEV)))
        assert (yd.float() - y.float()).abs().max() <= 2.0 ** -7 * y.float().abs().max()
        assert torch.equal(attention_core(**c), y)


@pytest.mark.parametrize("T,pos", [(1, 200), (4, 77), (200, 40)])
def test_infinities_and_nan_like_the_torch_form(T, pos):
    """inf and NaN among the keys and values of visible positions reach the
    output as in fp32: an infinite value stays infinite, a NaN or an infinite
    score makes its row NaN."""
    B, Hq, Hk, D, S = 1, 8, 2, 128, 512
    for what in ("v inf", "v nan", "k nan", "k inf"):
        print(T, pos, what, flush=True)
        c = _inputs(3, B, T, Hq, Hk, D, S, pos)
        t = c["cache_v" if what[0] == "v" else "cache_k"]
        t[0, 1, pos - 9, 5] = float(what[2:])
        with torch.inference_mode():
            y = attention_core(**c).view(T, Hq, D)
            q, k, v = _eager_rows(c, B, T, Hq, Hk, D)
            fk, fv = (u[:B, :, :pos + T].repeat_interleave(Hq // Hk, dim=1)
                      for u in (c["cache_k"], c["cache_v"]))
            r = _eager.attend(q, fk, fv, pos)[0].transpose(0, 1)
        for f in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(f(y), f(r)), (what, f)
        ok = torch.isfinite(r)
        assert (y[ok].float() - r[ok].float()).abs().max() <= 2.0 ** -6 * r[ok].float().abs().max()


def test_calls_left_to_the_torch_form():
    """Nothing is launched or written for a call the kernels do not take."""
    B, T, Hq, Hk, D, S, pos = 1, 2, 4, 2, 64, 40, 7
    c = _inputs(1, B, T, Hq, Hk, D, S, pos)
    k0 = c["cache_k"].clone().view(torch.int16)

    class Other(_eager.RMSNorm):
        pass

    odd = c["cache_k"].transpose(-1, -2).contiguous().transpose(-1, -2)  # D not innermost
    with torch.no_grad():
        for change in (dict(start_pos=S - 1), dict(start_pos=-1), dict(q_norm=Other(D).to(DEV)),
                       dict(cos=c["cos"].float()), dict(cos=c["cos"][:1]), dict(cache_k=odd),
                       dict(cache_v=c["cache_v"].float()), dict(k=c["k"].float()),
                       dict(start_pos=torch.tensor(7)), dict(num_heads=3),
                       dict(start_pos=torch.tensor(7, device=DEV, dtype=torch.int32))):
            print(list(change), flush=True)
            assert attention_core(**dict(c, **change)) is None, change
    with torch.enable_grad():  # the norm weights are parameters
        assert attention_core(**c) is None
    h = c["q_norm"].register_forward_hook(lambda *a: None)
    with torch.no_grad():
        assert attention_core(**c) is None
    h.remove()
    assert torch.equal(c["cache_k"].view(torch.int16), k0)
    with torch.no_grad():
        assert attention_core(**c) is not None


def test_cache_layouts_and_strided_rows():
    """A cache laid out [B, S, H, D], a padded one, and projections in a wider
    buffer give the contiguous call's bits."""
    B, T, Hq, Hk, D, S, pos = 2, 3, 8, 2, 128, 96, 50
    c = _inputs(9, B, T, Hq, Hk, D, S, pos)
    with torch.inference_mode():
        want = attention_core(**c)
        for f in (lambda t: t.transpose(1, 2).contiguous().transpose(1, 2),
                  lambda t: torch.nn.functional.pad(t, (0, 8))[..., :D],
                  lambda t: t[:B].clone()):
            d = dict(c, cache_k=f(c["cache_k"]), cache_v=f(c["cache_v"]))
            assert torch.equal(attention_core(**d), want)
            assert torch.equal(d["cache_k"][:B, :, :pos + T], c["cache_k"][:B, :, :pos + T])
        wide = torch.nn.functional.pad(torch.cat([c["q"], c["k"], c["v"]], -1), (4, 12))
        n = Hq * D
        d = dict(c, q=wide[..., 4:4 + n], k=wide[..., 4 + n:4 + n + Hk * D],
                 v=wide[..., 4 + n + Hk * D:4 + n + 2 * Hk * D])
        assert torch.equal(attention_core(**d), want)


@pytest.mark.parametrize("B,T,Hq,Hk,D,S,pos", [(1, 100, 8, 2, 128, 100, 0), (2, 65, 8, 8, 64, 201, 136),
                                               (1, 1, 8, 2, 128, 97, 96), (1, 9, 16, 2, 128, 70, 61)])
def test_full_cache_at_the_end_of_its_memory(B, T, Hq, Hk, D, S, pos):
    """The last tile's rows past the last key are not read: with NaN right behind
    a full cache that is no whole number of tiles, the same bits as without."""
    c = _inputs(11, B, T, Hq, Hk, D, S, pos)
    with torch.inference_mode():
        n = B * Hk * S * D
        for name in ("cache_k", "cache_v"):
            flat = torch.full((n + 64 * D,), float("nan"), dtype=torch.bfloat16, device=DEV)
            flat[:n] = c[name][:B].reshape(-1)
            c[name] = flat[:n].view(B, Hk, S, D)
        y = attention_core(**c)
        _check(c, B, T, Hq, Hk, D, y)
        d = dict(c, cache_k=c["cache_k"].clone(), cache_v=c["cache_v"].clone())
        assert torch.equal(attention_core(**d), y)


def test_overlapping_caches_stay_with_the_torch_form():
    """A cache whose sequences or heads share memory (an expanded one), and keys
    and values in one memory: nothing is launched or written (the torch form
    refuses the first two). Keys and values interleaved in one buffer are taken."""
    B, T, Hq, Hk, D, S, pos = 2, 2, 8, 4, 64, 40, 7
    c = _inputs(2, B, T, Hq, Hk, D, S, pos)
    ck, cv = c["cache_k"][:B].clone(), c["cache_v"][:B].clone()
    with torch.inference_mode():
        want = attention_core(**dict(c, cache_k=ck.clone(), cache_v=cv.clone()))
        for change in (dict(cache_k=ck[:1].clone().expand(B, -1, -1, -1)),
                       dict(cache_v=cv[:, :1].clone().expand(-1, Hk, -1, -1)),
                       dict(cache_k=ck, cache_v=ck), dict(cache_k=c["k"].as_strided(ck.shape, (0, 0, 0, 1)))):
            before = [t.clone().view(torch.int16) for t in (ck, cv)]
            assert attention_core(**dict(c, cache_k=ck, cache_v=cv) | change) is None, list(change)
            assert all(torch.equal(a, b.view(torch.int16)) for a, b in zip(before, (ck, cv)))
        both = torch.stack([ck, cv], dim=2).permute(0, 3, 2, 1, 4).contiguous()  # [B, S, 2, H, D]
        d = dict(c, cache_k=both[:, :, 0].transpose(1, 2), cache_v=both[:, :, 1].transpose(1, 2))
        assert torch.equal(attention_core(**d), want)


def _module(**swap):
    """The swapped attention layer of a one-layer model with heads of 64, its
    cache, an input and the arguments of a step at position 5."""
    from llms_amd import harness
    from llms_amd.kernels import apply_triton_kernels

    cfg = harness.Cfg(vocab_size=64, hidden_size=256, num_hidden_layers=1, num_attention_heads=4,
                      num_key_value_heads=2, head_dim=64, intermediate_size=256,
                      max_position_embeddings=64)
    m = apply_triton_kernels(harness.tiny_model(cfg, device=DEV), **swap)
    g = torch.Generator(device=DEV).manual_seed(6)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()  # noqa: E731
    cache = harness.KVCache([r(1, 2, 32, 64)], [r(1, 2, 32, 64)])
    kw = dict(layer_idx=0, cos=m.rope_cos[5:8], sin=m.rope_sin[5:8], start_pos=5)
    return m, cache, r(1, 3, 256), kw


def test_vmap_over_the_module():
    """torch.func.vmap over the layer with a cache per example runs as it does
    over the torch form: each example's output and cache."""
    from llms_amd.harness import KVCache

    m, cache, x, kw = _module()
    xs, ks, vs = (torch.stack([t, t.flip(-1)]) for t in (x, cache.k[0], cache.v[0]))

    def f(x, k, v):
        return m.layers[0].attn(x, kv_cache=KVCache([k], [v]), **kw), k, v

    with torch.no_grad():
        want = [f(x, k.clone(), v.clone()) for x, k, v in zip(xs, ks, vs)]
        got = torch.func.vmap(f)(xs, ks.clone(), vs.clone())
    for i in range(2):
        for a, b in zip(got, want[i]):
            assert (a[i].float() - b.float()).abs().max() <= 2.0 ** -6 * b.float().abs().max()


def test_autocast_keeps_its_types():
    """Under autocast the layer's core and the head are torch's, with the type
    that autocast gives a matmul (the model's blocks return theirs in bf16)."""
    m, cache, x, kw = _module(linear_down_o=True)
    c = _inputs(4, 1, 2, 4, 2, 64, 32, 5)
    ids = torch.tensor([[3, 1, 4]], device=DEV)
    with torch.inference_mode():
        assert m(ids, m.alloc_cache(32)).dtype == torch.bfloat16
        with torch.autocast("cuda", dtype=torch.float16):
            assert m(ids, m.alloc_cache(32)).dtype == torch.float16
            assert attention_core(**c) is None
        assert attention_core(**c) is not None


def test_inference_cache_is_written_in_inference_mode_only():
    """torch refuses in-place updates of an inference tensor outside inference
    mode; so does the layer. Other caches are written in either mode, and their
    version counts the write."""
    m, cache, x, kw = _module()
    run = lambda c: m.layers[0].attn(x, kv_cache=c, **kw)  # noqa: E731
    with torch.inference_mode():
        inf = type(cache)([cache.k[0].clone()], [cache.v[0].clone()])
    with torch.no_grad():
        with pytest.raises(RuntimeError, match="[Ii]nference"):
            run(inf)
        version = cache.k[0]._version
        want = run(cache)
        assert cache.k[0]._version > version
    with torch.inference_mode():
        assert torch.equal(run(inf), want)


def _direct(q, k, v, ck, cv, pos, pos_dev=None, short=0):
    """fp_attention_bf16 without norm weights and with cos = 1, sin = 0: its
    status and y [B, T, Hq, D]. short: bytes the workspace lacks."""
    import ctypes

    from llms_amd import _lib
    from tests.test_capi import _AttentionArgs

    lib = _lib.capi()
    (B, T, Hq, D), Hk, S = q.shape, k.shape[2], ck.shape[2]
    cos, sin = torch.ones(T, D, device=DEV).bfloat16(), torch.zeros(T, D, device=DEV).bfloat16()
    y = torch.zeros(B, T, Hq, D, device=DEV, dtype=torch.bfloat16)
    need = lib.fp_attention_workspace_bytes(B, T, Hq, Hk, D, S if pos_dev is not None else pos + T)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    P = lambda t: t.data_ptr()  # noqa: E731
    a = _AttentionArgs(q=P(q), k=P(k), v=P(v), ldq=Hq * D, ldk=Hk * D, ldv=Hk * D, cos=P(cos),
                       sin=P(sin), ld_cos=D, ld_sin=D, cache_k=P(ck), cache_v=P(cv),
                       k_s_b=ck.stride(0), k_s_h=ck.stride(1), k_s_p=ck.stride(2), v_s_b=cv.stride(0),
                       v_s_h=cv.stride(1), v_s_p=cv.stride(2), y=P(y), B=B, T=T, n_heads=Hq,
                       n_kv_heads=Hk, head_dim=D, cache_len=S, pos=pos,
                       pos_dev=None if pos_dev is None else P(pos_dev))
    st = lib.fp_attention_bf16(ctypes.byref(a), P(ws), need - short,
                               torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return st, y


def _rows(B, T, Hq, Hk, D, S, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(B + T + D)
    r = lambda *s: (torch.randn(*s, generator=g, device=DEV) * scale).bfloat16()  # noqa: E731
    return r(B, T, Hq, D), r(B, T, Hk, D), r(B, T, Hk, D), r(B, Hk, S, D), r(B, Hk, S, D)


def _fp64(q, ck, cv, pos):
    """Causal softmax attention of q [B, T, Hq, D] at pos .. in 64 bits; rows
    that see no key are NaN."""
    B, T, Hq, D = q.shape
    end = max(0, min(pos + T, ck.shape[2]))
    fk, fv = (t[:, :, :end].double().repeat_interleave(Hq // ck.shape[1], dim=1) for t in (ck, cv))
    s = torch.matmul(q.transpose(1, 2).double(), fk.transpose(-2, -1).contiguous()) * D ** -0.5
    hide = torch.arange(end, device=DEV)[None] > torch.arange(pos, pos + T, device=DEV)[:, None]
    return torch.matmul(torch.softmax(s.masked_fill(hide, float("-inf")), -1), fv).transpose(1, 2)


@pytest.mark.parametrize("B,T,Hq,Hk,D,S,pos", [(1, 1, 32, 8, 128, 2048, 2000), (2, 4, 8, 2, 64, 600, 500),
                                               (1, 200, 8, 2, 128, 500, 300), (1, 700, 16, 8, 64, 700, 0)])
@pytest.mark.parametrize("scale", [0.25, 1.0, 2.0])
def test_probabilities_keep_fp32_precision(B, T, Hq, Hk, D, S, pos, scale):
    """q and the keys enter exactly, so nothing but fp32 evaluation and the one
    rounding of the output is between y and 64 bits: p.V in fewer than 24 bits of
    p would show (one bf16 part exceeds the bound: ``test_attend_cpu.py``). Flat to peaked
    softmax; both kernels, with and without a key split."""
    q, k, v, ck, cv = _rows(B, T, Hq, Hk, D, S, scale)
    st, y = _direct(q, k, v, ck, cv, pos)
    assert st == 0
    for c, n in ((ck, k), (cv, v)):
        assert torch.equal(c[:, :, pos:pos + T], n.transpose(1, 2))
    t = _fp64(q, ck, cv, pos)
    d = (y.double() - t).abs()
    print(B, T, D, scale, "max excess", (d - 2.0 ** -8 * t.abs()).max().item())
    assert bool((d <= 2.0 ** -8 * t.abs() + 1e-5 * cv.double().abs().max()).all())


@pytest.mark.parametrize("T", [2, 100])
def test_workspace_and_device_positions_outside_the_cache(T):
    """A workspace one byte short is refused. Device positions outside the cache
    are neither written nor attended; inside, the int position's values."""
    B, Hq, Hk, D, S = 1, 8, 2, 64, 150
    q, k, v, ck0, cv0 = _rows(B, T, Hq, Hk, D, S)
    assert _direct(q, k, v, ck0.clone(), cv0.clone(), 5, short=1)[0] == 6
    for pos in (40, S - 1, S + 3, -1, -T, 2 ** 40, -2 ** 40):
        print(T, pos, flush=True)
        ck, cv = ck0.clone(), cv0.clone()
        st, y = _direct(q, k, v, ck, cv, 0, pos_dev=torch.tensor(pos, device=DEV))
        assert st == 0
        for c, c0, n in ((ck, ck0, k), (cv, cv0, v)):
            want = c0.clone()
            lo, hi = max(pos, 0), min(pos + T, S)
            if lo < hi:
                want[:, :, lo:hi] = n[:, lo - pos:hi - pos].transpose(1, 2)
            assert torch.equal(c, want), pos
        t = _fp64(q, ck, cv, max(min(pos, S + T), -2 * T))
        seen = pos + torch.arange(T, device=DEV) >= 0
        d = (y.double() - t).abs()[:, seen]
        assert bool((d <= 2.0 ** -8 * t[:, seen].abs() + 1e-5 * cv.double().abs().max()).all()), pos
        assert bool(y[:, ~seen].isnan().all()), pos
