"""The band kernel at up to 16 rows (16-row MFMA blocks, the x sums as fp32 MFMAs) and its
stream's tail, against the float64 oracle.

Codes stay exact on MFMA and scale and bias are applied per group in fp32, the decode GEMVs'
rule, so the bound is theirs: 2 bf16 steps of the larger of the result and the product before
the bias, plus 1e-5 of the largest result for the fp32 sums."""
import numpy as np
import pytest
import torch

from oracle.bf16 import bf16_to_f32, f32_to_bf16
from oracle.mlx_affine import quantize_bf16, quantized_matmul_f64
from shardcompute_amd import _lib
from tests.gpu_util import dev_bf16, dev_u32, host_u16, host_u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M", [1, 8, 15, 16])
def test_band_up_to_16_rows(device, bits, M):
    rng = np.random.default_rng(1600 + M + bits)
    # one scale block (the tail alone), one weight row, ragged widths, several blocks
    for K, N in [(512, 1), (512, 300), (1024, 257), (3584, 130), (8192, 96)]:
        x = f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
        wq, s, b = quantize_bf16((rng.standard_normal((N, K)) * 0.02).astype(np.float32), 64, bits)
        bias = f32_to_bf16(rng.standard_normal(N).astype(np.float32) * 0.1) if N % 2 == 0 else None
        prod = quantized_matmul_f64(x, wq, s, b, 64, bits)
        ref = prod
        if bias is not None:
            ref = bf16_to_f32(f32_to_bf16(prod.astype(np.float32))).astype(np.float64) + bf16_to_f32(bias)[None, :]
        for plan in [(0, 0), (8, 1), (4, 1), (8, 3), (4, 16)]:
            print(f"band16 M={M} K={K} N={N} W{bits} plan={plan}", flush=True)
            y = _lib.qmm(dev_bf16(x), dev_u32(wq), dev_bf16(s), dev_bf16(b),
                         None if bias is None else dev_bf16(bias), bits=bits, band_plan=plan)
            torch.cuda.synchronize()
            got = bf16_to_f32(host_u16(y)).astype(np.float64)
            _, e = np.frexp(np.maximum(np.abs(ref), np.abs(prod)))
            bad = np.argwhere(np.abs(got - ref) > 2 * np.ldexp(1.0, e - 8) + 1e-5 * np.max(np.abs(ref)))
            assert bad.size == 0, (plan, bad[0], got[tuple(bad[0])], ref[tuple(bad[0])])


@pytest.mark.parametrize("bits,M,N,K", [
    (4, 16, 8192, 1024), (4, 16, 11264, 2048), (4, 16, 14000, 4096), (4, 9, 16384, 512),  # the band's would: fit / fit / exceed / be none
    (8, 16, 32752, 1024), (8, 9, 32768, 1024), (8, 16, 22000, 4096), (8, 9, 43528, 1024)])
def test_wide_products_of_9_to_16_rows_need_no_more_scratch(device, bits, M, N, K):
    """The allocation-free entry gives sc_qmm_bf16's bits on either side of the 9-16-row rule's
    line (8192 weight rows) and for wider products, whose partials on the band kernel would
    exceed its scratch or be scratch that the GEMV, unsplit, does not take."""
    rng = np.random.default_rng(N + K)
    x = dev_bf16(f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32)))
    per = 8 if bits == 4 else 4
    wq = dev_u32(rng.integers(0, 2**32, (N, K // per), dtype=np.uint32))
    s = dev_bf16(f32_to_bf16(rng.uniform(0.001, 0.01, (N, K // 64)).astype(np.float32)))
    b = dev_bf16(f32_to_bf16(rng.uniform(-0.05, 0.05, (N, K // 64)).astype(np.float32)))
    y = _lib.qmm(x, wq, s, b, None, bits=bits)
    y2 = _lib.qmm(x, wq, s, b, None, bits=bits, no_alloc=True)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    cols = np.r_[0:16, N // 2:N // 2 + 16, N - 16:N]
    ref = quantized_matmul_f64(host_u16(x), host_u32(wq)[cols], host_u16(s)[cols],
                               host_u16(b)[cols], 64, bits)
    got = bf16_to_f32(host_u16(y)).astype(np.float64)[:, cols]
    _, e = np.frexp(np.abs(ref))
    assert np.all(np.abs(got - ref) <= 2 * np.ldexp(1.0, e - 8) + 1e-5 * np.max(np.abs(ref)))


@pytest.mark.parametrize("bits,M,N,K", [(8, 11, 24560, 3072), (8, 9, 44752, 4096), (4, 13, 14648, 3072)])
def test_wide_products_of_9_to_16_rows_run_on_the_gemv(device, bits, M, N, K):
    """The band kernel's tiles and splits miss one round of the CUs here by a little (1.1-1.5
    times the GEMV's time); its sums run in another order, so the bits tell the two apart."""
    g = torch.Generator(device="cuda")
    g.manual_seed(N)
    x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
    w = _lib.quantize(torch.randn((N, K), generator=g, device="cuda").mul_(0.02), bits=bits)
    y, yg, yb = (_lib.qmm(x, *w, bits=bits, path=p) for p in (_lib.PATH_AUTO, _lib.PATH_GEMV, _lib.PATH_BAND))
    assert not torch.equal(yg, yb)
    assert torch.equal(y, yg)
