"""The dense prefill GEMM (weights dequantized once per call into a workspace) against the
fp64 product of the dequantized weights.

Both round every weight to bf16(s q + b) alike, so an output differs from the reference by
its own bf16 rounding (2^-8 of it, 2^-7 with the bias added and rounded again) and by the
fp32 accumulation: at most K 2^-23 of sum |x w|, of which the bound takes the square root of
K steps' worth times 8 (random signs)."""
import ctypes
import math

import pytest
import torch

from shardcompute_amd import _lib

pytestmark = pytest.mark.gpu


def _inputs(M, N, K, bits, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    wq, s, b = _lib.quantize(torch.randn((N, K), generator=g, device="cuda").mul_(0.02), bits=bits)
    x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    w = _lib.dequantize(wq, s, b, bits=bits)
    ref = x.double() @ w.double().T
    acc = 8 * math.sqrt(K) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    return x, wq, s, b, bias, ref, acc


# (256 CUs) the smallest products taken at each line of the size rule, ragged rows and columns,
# stages of odd number, narrow tiles alone, wide ones alone (two rounds), a round of wide ones
# and the last columns narrow, weights in two column chunks (N K above 2^27), many row tiles
SHAPES = [(1280, 6560, 2048, 4), (1024, 11232, 2048, 8), (1600, 12504, 1536, 4), (1300, 20008, 1024, 8),
          (1281, 15880, 1024 + 576, 8), (2048, 4096, 4096, 4), (2049, 4104, 2048, 8), (2815, 11008, 2112, 4),
          (2041, 11272, 2112, 4), (2048, 28672, 1024, 8), (1030, 34000, 4096, 8), (51000, 512, 1024, 4)]


@pytest.mark.parametrize("M,N,K,bits", SHAPES)
def test_dense_against_reference(device, M, N, K, bits):
    assert _lib.load().sc_qmm_workspace_bytes(M, N, K) > 0
    print(f"dense M={M} N={N} K={K} bits={bits}", flush=True)
    x, wq, s, b, bias, ref, acc = _inputs(M, N, K, bits, M + N)
    y = _lib.qmm(x, wq, s, b, bits=bits)
    bad = (y.double() - ref).abs() > 2.0 ** -8 * ref.abs() + acc
    assert not bad.any(), bad.nonzero()[:3]
    yb = _lib.qmm(x, wq, s, b, bias=bias, bits=bits)
    r = y.double() + bias.double()
    bad = (yb.double() - r).abs() > 2.0 ** -8 * r.abs() + 1e-30
    assert not bad.any(), bad.nonzero()[:3]


@pytest.mark.parametrize("M,I,K,bits", [(2048, 4096, 2048, 4), (1281, 5624, 2112, 8), (1030, 17000, 4096, 4)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_dense_swiglu_equals_product_then_gate(device, M, I, K, bits, with_bias):
    assert _lib.load().sc_qmm_workspace_bytes(M, 2 * I, K) > 0
    x, wq, s, b, bias, _, _ = _inputs(M, 2 * I, K, bits, I)
    bias = bias if with_bias else None
    act, _ = _lib.qmm_swiglu(x, wq, s, b, bias=bias, bits=bits)
    assert torch.equal(act, _lib.silu_mul(_lib.qmm(x, wq, s, b, bias=bias, bits=bits)))


def test_workspace_forms(device):
    """A misaligned output and a small, null or misaligned workspace take the fused GEMM; every
    form agrees with the reference."""
    M, N, K, bits = 2048, 4096, 1024 * 2, 4
    x, wq, s, b, _, ref, acc = _inputs(M, N, K, bits, 7)
    lib, P = _lib.load(), ctypes.c_void_p
    need = lib.sc_qmm_workspace_bytes(M, N, K)
    assert need == N * K * 2
    ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
    flat = torch.empty(M * N + 8, dtype=torch.bfloat16, device="cuda")
    for y_off, ws_off, ws_bytes in ((0, 0, need), (1, 0, need), (0, 8, need), (0, 0, need - 1), (0, None, 0)):
        y = flat[y_off:y_off + M * N]
        y.fill_(float("nan"))
        rc = lib.sc_qmm_bf16_ws(P(x.data_ptr()), P(wq.data_ptr()), P(s.data_ptr()), P(b.data_ptr()), None,
                                P(y.data_ptr()), M, N, K, bits, 64,
                                None if ws_off is None else P(ws.data_ptr() + ws_off), ws_bytes,
                                P(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.sc_last_error()
        bad = (y.view(M, N).double() - ref).abs() > 2.0 ** -8 * ref.abs() + acc
        assert not bad.any(), (y_off, ws_off, ws_bytes)


@pytest.mark.parametrize("M,N,K", [(1279, 6560, 2048), (1280, 6552, 2048), (1023, 32768, 4096), (1024, 11224, 2048),
                                   (1279, 16384, 8256), (1600, 12496, 1536), (1300, 19992, 1024), (4096, 4096, 960)])
def test_below_the_size_rule_no_workspace(device, M, N, K):
    assert _lib.load().sc_qmm_workspace_bytes(M, N, K) == 0


def test_rows_of_element_stores_take_the_fused_gemm(device):
    """Widths that are no multiple of 8 want no workspace (2-byte stores cost the dense kernel
    more than it gains on most of them) and give the fused GEMM's bits."""
    M, N, K, bits = 1300, 16001, 1600, 4
    assert _lib.load().sc_qmm_workspace_bytes(M, N, K) == 0 < _lib.load().sc_qmm_workspace_bytes(M, N - 1, K)
    x, wq, s, b, bias, _, _ = _inputs(M, N, K, bits, 3)
    assert torch.equal(_lib.qmm(x, wq, s, b, bias=bias, bits=bits),
                       _lib.qmm(x, wq, s, b, bias=bias, bits=bits, path=_lib.PATH_GEMM))


def test_dense_under_graph_capture(device):
    M, N, K, bits = 2048, 4096, 2048, 4
    x, wq, s, b, _, _, _ = _inputs(M, N, K, bits, 9)
    y = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    _lib.qmm(x, wq, s, b, bits=bits, out=y)
    eager = y.clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _lib.qmm(x, wq, s, b, bits=bits, out=y)
    for _ in range(3):
        y.zero_()
        _lib.qmm(x[:1300], wq, s, b, bits=bits)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager)
