"""The RMSNorm prologue fused into QKV and gate-up-SiLU (one launch in the
row-streaming regime, a prologue kernel plus the usual kernels above it)
against the oracle: reference RMSNorm (``src/engine/attention.py:28-33``)
followed by the reference's unfused projection, with the projection hull
widened by the norm's admissible rounding spread."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import ref
from tests._util import bits, ffn_inputs, gen, qkv_inputs, randn_bf16

DEV = "cuda"
EPS = 1e-6


def _norm_weight(seed: int, K: int) -> torch.Tensor:
    return (1.0 + 0.3 * torch.randn(K, generator=gen(seed))).to(torch.bfloat16)


def _x(seed: int, M: int, K: int, std: float = 3.0) -> torch.Tensor:
    return randn_bf16(gen(seed), M, K, std=std)


def _rows(M: int, limit: int = 96) -> np.ndarray:
    if M <= limit:
        return np.arange(M)
    return np.unique(np.concatenate([np.linspace(0, M - 1, limit).astype(int), [M - 1]]))


def _check(y: torch.Tensor, out: ref.OracleOut, label: str) -> None:
    p = ref.check_parity(bits(y), out)
    print(f"{label}: {p}")
    assert p.ok, f"{label}: {p}"


def _kern():
    from llms_amd import kernels

    return kernels


def check_norm_qkv(M, K, n_q, n_k, seed=0, std=3.0, eps=EPS, gamma=None):
    x = _x(seed + 1, M, K, std)
    _, w = qkv_inputs(seed + 2, 1, K, n_q, n_k)
    g = _norm_weight(seed + 3, K) if gamma is None else gamma
    q, k, v = _kern().fused_rmsnorm_qkv(x.to(DEV), g.to(DEV), eps, w.to(DEV), n_q=n_q, n_k=n_k)
    y = torch.cat([q, k, v], dim=-1).cpu()
    rows = _rows(M)
    out = ref.ref_rmsnorm_qkv_full(bits(x)[rows], bits(g), eps, bits(w), n_q, n_k)
    _check(y[rows], out, f"norm+qkv M={M} K={K}")


def check_norm_gate_up(M, K, N, seed=0, std=3.0, eps=EPS):
    x = _x(seed + 1, M, K, std)
    _, wg, wu = ffn_inputs(seed + 2, 1, K, N)
    g = _norm_weight(seed + 3, K)
    y = _kern().fused_rmsnorm_gate_up_silu(x.to(DEV), g.to(DEV), eps, wg.to(DEV), wu.to(DEV)).cpu()
    rows = _rows(M)
    out = ref.ref_rmsnorm_gate_up_silu_full(bits(x)[rows], bits(g), eps, bits(wg), bits(wu))
    _check(y[rows], out, f"norm+gate-up M={M} K={K} N={N}")


# ------------------------------------------------------------------ CPU


def test_workspace_bytes_and_errors():
    """The workspace query always leaves room for the normalised rows:
    decode-sized calls usually run as one launch and leave it unused, but
    fall back to the two-launch path when a pointer or stride is not 16-byte
    aligned; larger calls add split partials. Argument errors come back
    before any launch."""
    from llms_amd import _lib

    lib = _lib.capi()
    wb = lib.fp_rmsnorm_workspace_bytes
    rows = lambda M, K: (M * K * 2 + 255) // 256 * 256  # noqa: E731
    assert wb(1, 6144, 2560, 0, 0) == rows(1, 2560) and wb(2, 9728, 2560, 1, 0) == rows(2, 2560)
    assert wb(4, 9728, 2560, 1, 1) == rows(4, 2560)   # int8 rows kernel to 4 rows
    assert wb(3, 6144, 2560, 0, 0) == rows(3, 2560)   # bf16 from 3 rows
    assert wb(1, 6144, 2541, 0, 0) == (2541 * 2 + 255) // 256 * 256  # K % 8 != 0
    assert wb(512, 2560, 9728, 0, 0) > 512 * 9728 * 2  # rows + split partials
    P = ctypes.c_void_p(16)
    # fp_rmsnorm_qkv_bf16(x, ldx, gamma, eps, w, ldw, y, ldy, M, n_q, n_k, K, ws, ws_bytes, stream)
    assert lib.fp_rmsnorm_qkv_bf16(P, 64, None, 1e-6, P, 64, P, 96, 2, 64, 16, 64, None, 0, None) == 1
    assert lib.fp_rmsnorm_qkv_bf16(P, 64, P, -1.0, P, 64, P, 96, 2, 64, 16, 64, None, 0, None) == 2
    assert lib.fp_rmsnorm_qkv_bf16(P, 64, P, float("nan"), P, 64, P, 96, 2, 64, 16, 64, None, 0,
                                   None) == 2
    assert lib.fp_rmsnorm_qkv_bf16(P, 64, P, 1e-6, P, 64, P, 96, 2, 64, 16, 64, ctypes.c_void_p(8),
                                   64, None) == 6
    assert lib.fp_rmsnorm_gate_up_silu_bf16(P, 64, P, 1e-6, P, 64, P, 60, P, 32, 2, 32, 64, None, 0,
                                            None) == 3
    assert lib.fp_rmsnorm_qkv_w8(P, 64, P, 1e-6, P, 64, None, P, 96, 2, 64, 16, 64, None, 0,
                                 None) == 1
    assert lib.fp_rmsnorm_gate_up_silu_w8(None, 64, None, 1e-6, None, 64, None, None, 64, None, None,
                                          32, 0, 32, 64, None, 0, None) == 0  # M == 0


def test_python_argument_errors():
    kern = _kern()
    x = torch.randn(2, 64).bfloat16()
    w = torch.randn(96, 64).bfloat16()
    with pytest.raises(ValueError, match="norm weight shape"):
        kern.fused_rmsnorm_qkv(x, torch.ones(63).bfloat16(), EPS, w, n_q=64, n_k=16)
    with pytest.raises(ValueError, match="eps"):
        kern.fused_rmsnorm_qkv(x, torch.ones(64).bfloat16(), -1.0, w, n_q=64, n_k=16)
    with pytest.raises(ValueError, match="HIP"):
        kern.fused_rmsnorm_qkv(x, torch.ones(64).bfloat16(), EPS, w, n_q=64, n_k=16)
    with pytest.raises(ValueError, match="Wg shape"):
        kern.fused_rmsnorm_gate_up_silu(x, torch.ones(64).bfloat16(), EPS, w, w[:10])


# ------------------------------------------------------------------ GPU


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 3, 4, 8, 64, 300])
def test_norm_qkv_qwen3_4b(M):
    check_norm_qkv(M, 2560, 4096, 1024, seed=M)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 5, 64, 300])
def test_norm_gate_up_qwen3_4b(M):
    check_norm_gate_up(M, 2560, 9728, seed=10 + M)


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", [(1, 1024), (2, 16384), (1, 2541), (3, 2541), (1, 32768),
                                 (2, 8), (70, 1032)])
def test_norm_shapes_and_paths(M, K):
    """Small and large K, K % 8 != 0 (the element-wise prologue), the rows
    kernel's LDS limit, tiny K."""
    check_norm_qkv(M, K, 96, 16, seed=20 + K + M)
    check_norm_gate_up(M, K, 100, seed=21 + K + M)


@pytest.mark.gpu
def test_norm_edge_values():
    """An all-zero row (r = 1/sqrt(eps), output 0), a large eps, tiny and
    large row scales, and a norm weight that is not 16-byte aligned (a view at
    offset 1: the one-launch path is refused, the prologue runs)."""
    K, n_q, n_k = 2560, 256, 64
    for std in (1e-3, 40.0):
        check_norm_qkv(2, K, n_q, n_k, seed=31, std=std)
    check_norm_qkv(2, K, n_q, n_k, seed=32, eps=0.5)
    x = _x(33, 2, K)
    x[0] = 0
    _, w = qkv_inputs(34, 1, K, n_q, n_k)
    g = _norm_weight(35, K)
    q, k, v = _kern().fused_rmsnorm_qkv(x.to(DEV), g.to(DEV), EPS, w.to(DEV), n_q=n_q, n_k=n_k)
    y = torch.cat([q, k, v], dim=-1).cpu()
    assert torch.all(y[0] == 0)
    _check(y, ref.ref_rmsnorm_qkv_full(bits(x), bits(g), EPS, bits(w), n_q, n_k), "zero row")
    gbig = torch.empty(K + 1, dtype=torch.bfloat16, device=DEV)
    gbig[1:] = g.to(DEV)
    q, k, v = _kern().fused_rmsnorm_qkv(x.to(DEV), gbig[1:], EPS, w.to(DEV), n_q=n_q, n_k=n_k)
    _check(torch.cat([q, k, v], dim=-1).cpu(),
           ref.ref_rmsnorm_qkv_full(bits(x), bits(g), EPS, bits(w), n_q, n_k), "misaligned gamma")


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 4, 100])
def test_norm_int8(M):
    kern = _kern()
    K, n_q, n_k, I = 2560, 4096, 1024, 9728
    x = _x(40 + M, M, K)
    g = _norm_weight(41, K)
    _, w = qkv_inputs(42, 1, K, n_q, n_k)
    q8, s8 = kern.quantize_w8_per_row(w.to(DEV))
    q, k, v = kern.fused_rmsnorm_qkv_w8(x.to(DEV), g.to(DEV), EPS, q8, s8, n_q=n_q, n_k=n_k)
    rows = _rows(M)
    wd = ref.dequant_w8(q8.cpu().numpy(), s8.cpu().numpy())
    _check(torch.cat([q, k, v], dim=-1).cpu()[rows],
           ref.ref_rmsnorm_qkv_full(bits(x)[rows], bits(g), EPS, wd, n_q, n_k), f"int8 norm+qkv M={M}")
    _, wg, wu = ffn_inputs(43, 1, K, I)
    qg, sg = kern.quantize_w8_per_row(wg.to(DEV))
    qu, su = kern.quantize_w8_per_row(wu.to(DEV))
    y = kern.fused_rmsnorm_gate_up_silu_w8(x.to(DEV), g.to(DEV), EPS, qg, sg, qu, su).cpu()
    _check(y[rows], ref.ref_rmsnorm_gate_up_silu_full(
        bits(x)[rows], bits(g), EPS, ref.dequant_w8(qg.cpu().numpy(), sg.cpu().numpy()),
        ref.dequant_w8(qu.cpu().numpy(), su.cpu().numpy())), f"int8 norm+gate-up M={M}")


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 64])
def test_norm_deterministic_and_raw_abi(M):
    """Repeated calls are bit-identical; through the raw C ABI a call that
    needs the prologue and gets no workspace returns FP_ERR_WORKSPACE and
    launches nothing (y keeps its sentinel)."""
    from llms_amd import _lib

    kern = _kern()
    K, n_q, n_k = 2560, 4096, 1024
    x = _x(50 + M, M, K).to(DEV)
    g = _norm_weight(51, K).to(DEV)
    _, w = qkv_inputs(52, 1, K, n_q, n_k)
    w = w.to(DEV)
    a = torch.cat(kern.fused_rmsnorm_qkv(x, g, EPS, w, n_q=n_q, n_k=n_k), dim=-1)
    b = torch.cat(kern.fused_rmsnorm_qkv(x, g, EPS, w, n_q=n_q, n_k=n_k), dim=-1)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    lib = _lib.capi()
    N = n_q + 2 * n_k
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    need = lib.fp_rmsnorm_workspace_bytes(M, N, K, 0, 0)
    assert need >= (M * K * 2 + 255) // 256 * 256
    st = lib.fp_rmsnorm_qkv_bf16(P(x), K, P(g), EPS, P(w), K, P(y), N, M, n_q, n_k, K, None, 0, stream)
    if M > 2:  # past the one-launch decode path: the normalised rows need room
        assert st == 6
        torch.cuda.synchronize()
        assert torch.all(y == 7.0)
    else:
        assert st == 0
    if M <= 2:
        # an odd row stride keeps x off the one-launch path: the queried
        # workspace is enough for the two-launch path
        xs = torch.zeros(M, K + 1, dtype=torch.bfloat16, device=DEV)
        xs[:, :K] = x
        ws = torch.empty(need, dtype=torch.uint8, device=DEV)
        y2 = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
        assert lib.fp_rmsnorm_qkv_bf16(P(xs), K + 1, P(g), EPS, P(w), K, P(y2), N, M, n_q, n_k, K,
                                       None, 0, stream) == 6
        assert lib.fp_rmsnorm_qkv_bf16(P(xs), K + 1, P(g), EPS, P(w), K, P(y2), N, M, n_q, n_k, K,
                                       P(ws), need, stream) == 0
        torch.cuda.synchronize()
        _check(y2.cpu(), ref.ref_rmsnorm_qkv_full(bits(x), bits(g), EPS, bits(w), n_q, n_k),
               f"norm+qkv strided x M={M}")
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
    assert lib.fp_rmsnorm_qkv_bf16(P(x), K, P(g), EPS, P(w), K, P(y), N, M, n_q, n_k, K, P(ws),
                                   need, stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), a.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("M,K", [(1, 2048), (1, 2064), (1, 2560), (1, 2576), (2, 1024), (2, 1032),
                                 (2, 1280), (2, 1296), (3, 512), (4, 2560)])
def test_norm_in_rows_or_apart(M, K):
    """Row counts and sizes on both sides of the rule that leaves the norm to
    the row kernel or to a launch of its own, and the call without a workspace
    (always the row kernel): both are the oracle's result."""
    from llms_amd import _lib

    kern = _kern()
    check_norm_qkv(M, K, 96, 16, seed=60 + K + M)
    check_norm_gate_up(M, K, 100, seed=61 + K + M)
    x, g = _x(62, M, K), _norm_weight(63, K)
    _, wg, wu = ffn_inputs(64, 1, K, 100)
    qg, sg = kern.quantize_w8_per_row(wg.to(DEV))
    qu, su = kern.quantize_w8_per_row(wu.to(DEV))
    if K % 16:
        return
    y = kern.fused_rmsnorm_gate_up_silu_w8(x.to(DEV), g.to(DEV), EPS, qg, sg, qu, su).cpu()
    xd, gd = x.to(DEV), g.to(DEV)
    y0 = torch.empty(M, 100, dtype=torch.bfloat16, device=DEV)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert _lib.capi().fp_rmsnorm_gate_up_silu_w8(
        P(xd), K, P(gd), EPS, P(qg), K, P(sg), P(qu), K, P(su), P(y0), 100, M, 100, K, None, 0,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    out = ref.ref_rmsnorm_gate_up_silu_full(
        bits(x), bits(g), EPS, ref.dequant_w8(qg.cpu().numpy(), sg.cpu().numpy()),
        ref.dequant_w8(qu.cpu().numpy(), su.cpu().numpy()))
    _check(y, out, f"int8 norm+gate-up M={M} K={K}")
    _check(y0.cpu(), out, f"int8 norm+gate-up M={M} K={K}, no workspace")


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(2, 2560, 2048), (2, 2560, 2056), (2, 3072, 1024), (2, 3072, 1032),
                                   (2, 1536, 4096), (2, 1536, 4104), (1, 4096, 4096), (1, 4096, 4104),
                                   (3, 1024, 2048), (4, 2048, 2048), (1, 4096, 32800)])
def test_norm_in_rows_or_apart_by_width(M, K, N):
    """The same at the widths where the rule changes, bf16 and int8."""
    kern = _kern()
    check_norm_qkv(M, K, N - 32, 16, seed=90 + K + M)
    if N <= 4104:
        check_norm_gate_up(M, K, N // 2, seed=91 + K + M)
    x, g = _x(92, M, K), _norm_weight(93, K)
    _, w = qkv_inputs(94, 1, K, N, 0)
    q, s = kern.quantize_w8_per_row(w.to(DEV))
    wq = ref.dequant_w8(q.cpu().numpy(), s.cpu().numpy())
    y = kern.fused_rmsnorm_qkv_w8(x.to(DEV), g.to(DEV), EPS, q, s, n_q=N, n_k=0)[0]
    _check(y.cpu(), ref.ref_rmsnorm_qkv_full(bits(x), bits(g), EPS, wq, N, 0), f"int8 norm+qkv {M} {K} {N}")
    h = N // 2
    y = kern.fused_rmsnorm_gate_up_silu_w8(x.to(DEV), g.to(DEV), EPS, q[:h], s[:h], q[h:], s[h:])
    _check(y.cpu(), ref.ref_rmsnorm_gate_up_silu_full(bits(x), bits(g), EPS, wq[:h], wq[h:]),
           f"int8 norm+gate-up {M} {K} {h}")


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,V", [(1, 256, 40000), (2, 1024, 33000), (3, 2560, 8200), (8, 2560, 8201),
                                   (9, 4096, 8320), (16, 1024, 10000), (17, 256, 9000),
                                   (33, 256, 8300), (16, 1024, 12300), (5, 512, 16380), (9, 1024, 28680),
                                   (12, 4096, 28680), (8, 1024, 48001), (20, 512, 16390), (32, 512, 24580)])
def test_norm_and_wide_head(M, K, V):
    """The final norm and head of a model: wide outputs at the row counts where
    their tile changes, against the oracle; past 16 rows, with gradients or a
    hooked norm the helper leaves the call to torch."""
    from llms_amd.kernels._eager import RMSNorm
    from llms_amd.kernels.fused_norm import fused_rmsnorm_head

    x, g = _x(70 + M, M, K), _norm_weight(71, K)
    _, w = qkv_inputs(72, 1, K, V, 0)
    norm = RMSNorm(K, eps=EPS).to(DEV, torch.bfloat16)
    with torch.no_grad():
        norm.weight.copy_(g)
        xd, wd = x.to(DEV), w.to(DEV)
        y = fused_rmsnorm_head(xd[None], norm, wd)
        if M > 16:
            assert y is None
            y = _kern().fused_rmsnorm_qkv(xd, norm.weight, EPS, wd, n_q=V, n_k=0)[0][None]
        assert y.shape == (1, M, V)
        _check(y[0].cpu(), ref.ref_rmsnorm_qkv_full(bits(x), bits(g), EPS, bits(w), V, 0),
               f"head M={M} K={K} V={V}")
        h = norm.register_forward_hook(lambda *a: None)
        assert fused_rmsnorm_head(xd[None], norm, wd) is None
        h.remove()
    assert fused_rmsnorm_head(xd[None], norm, wd) is None  # the weight is a parameter


@pytest.mark.gpu
def test_head_calls_left_to_torch():
    """What ``F.linear(norm(h), W)`` takes and the kernels do not: a weight that
    broadcasts, a negative eps, a column-major head; and its own shape error."""
    from llms_amd.kernels._eager import RMSNorm
    from llms_amd.kernels.fused_norm import fused_rmsnorm_head

    K, V = 256, 512
    h, w = (t.to(DEV) for t in (_x(80, 2, K)[None], _x(81, V, K)))
    norm = lambda n, eps: RMSNorm(n, eps=eps).to(DEV, torch.bfloat16)  # noqa: E731
    with torch.no_grad():
        assert fused_rmsnorm_head(h, norm(K, EPS), w) is not None
        for n, t in ((norm(1, EPS), w), (norm(K, -1e-3), w), (norm(K, float("inf")), w),
                     (norm(K, EPS), w.T.contiguous().T), (norm(K, EPS), w[:, :-8]),
                     (norm(K, EPS), w[0])):
            assert fused_rmsnorm_head(h, n, t) is None


def test_head_where_the_library_is_faster():
    """Wide heads whose rows 16-byte loads do not divide (by length, stride or
    address) from two rows of h, and very wide ones of short rows at two to four,
    are left to torch."""
    from llms_amd.kernels.fused_norm import _library_head

    def left(rows, K, N=20000, off=0, pad=0):
        w = torch.empty(N * (K + pad) + 64, dtype=torch.bfloat16)
        off += -(w.data_ptr() // 2) % 8
        return _library_head(rows, w[off:off + N * (K + pad)].view(N, K + pad)[:, :K])

    assert left(2, 541) and left(16, 541) and not left(1, 541) and not left(2, 541, N=16384)
    assert not left(2, 544) and left(2, 544, off=1) and left(2, 544, pad=4) and not left(2, 544, pad=8)
    assert left(4, 64, N=40000) and not left(5, 64, N=40000) and not left(1, 64, N=40000)
    assert not left(2, 256, N=40000) and not left(2, 64, N=32768)
