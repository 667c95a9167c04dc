"""The 128 x 128-tile GEMM (161 rows and more, few tiles) against the fp64 product of the
dequantized weights, with the dense GEMM's bound: the output's bf16 rounding (2^-8 of it) and
8 sqrt(K) 2^-24 sum |x w| for the fp32 sums."""
import math

import pytest
import torch

from shardcompute_amd import _lib

pytestmark = pytest.mark.gpu


def _inputs(M, N, K, bits):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    wq, s, b = _lib.quantize(torch.randn((N, K), generator=g, device="cuda").mul_(0.02), bits=bits)
    x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
    return x, wq, s, b, torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)


# one row and one column past a tile, ragged widths and odd ones (which run on the fused GEMM), one scale block, the largest tile
# count and one past it, K split with and without enough blocks for its splits
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [(161, 128, 512), (257, 129, 1024), (300, 1001, 512), (170, 77, 2048), (170, 1000, 1024), (201, 72, 5120),
                                   (2048, 2048, 512), (2049, 2048, 512), (333, 2048, 5632), (200, 300, 4096)])
def test_mid_against_reference(device, M, N, K, bits):
    print(f"mid M={M} N={N} K={K} W{bits}", flush=True)
    x, wq, s, b, bias = _inputs(M, N, K, bits)
    w = _lib.dequantize(wq, s, b, bits=bits).double()
    ref = x.double() @ w.T
    acc = 8 * math.sqrt(K) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    y = _lib.qmm(x, wq, s, b, bits=bits)
    bad = (y.double() - ref).abs() > 2.0 ** -8 * ref.abs() + acc
    assert not bad.any(), bad.nonzero()[:3]
    yb = _lib.qmm(x, wq, s, b, bias=bias, bits=bits)
    r = y.double() + bias.double()
    assert not ((yb.double() - r).abs() > 2.0 ** -8 * r.abs() + 1e-30).any()


@pytest.mark.parametrize("M,I,K,bits", [(161, 512, 1024, 4), (333, 1000, 2048, 8), (200, 136, 5632, 4)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_mid_swiglu_equals_product_then_gate(device, M, I, K, bits, with_bias):
    x, wq, s, b, bias = _inputs(M, 2 * I, K, bits)
    bias = bias if with_bias else None
    act, _ = _lib.qmm_swiglu(x, wq, s, b, bias=bias, bits=bits)
    assert torch.equal(act, _lib.silu_mul(_lib.qmm(x, wq, s, b, bias=bias, bits=bits)))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,equal", [(200, 304, 4096, True), (333, 2048, 5632, False), (300, 1000, 2048, True)])
def test_mid_without_allocation(device, bits, M, N, K, equal):
    """Split-K partials that fit the allocation-free array (4 MiB): sc_qmm_bf16's bits; partials
    that do not (4 x 333 x 2048 floats): K whole, against the reference."""
    print(f"mid noalloc M={M} N={N} K={K} W{bits}", flush=True)
    x, wq, s, b, bias = _inputs(M, N, K, bits)
    y = _lib.qmm(x, wq, s, b, bias=bias, bits=bits)
    yn = _lib.qmm(x, wq, s, b, bias=bias, bits=bits, no_alloc=True)
    assert torch.equal(y, yn) == equal
    w = _lib.dequantize(wq, s, b, bits=bits).double()
    p = x.double() @ w.T
    ref = p + bias.double()
    acc = 8 * math.sqrt(K) * 2.0 ** -24 * (x.double().abs() @ w.abs().T)
    assert not ((yn.double() - ref).abs() > 2.0 ** -8 * (ref.abs() + p.abs()) + acc).any()
