"""ParallelMLP.intermediate against the gate|up product followed by the activation.

From 9 rows on the two are equal bit for bit.  Up to 8 rows the fused product pairs gate and
up columns in its tiles, so its fp32 sums run in another order and a rare element moves by a
bf16 step of gate or up: as for the fused entry itself, under 2 % of the elements, by at most
2e-3 of the largest."""
import pytest
import torch

from shardcompute_amd import _lib
from shardcompute_amd.parallel.mlp import ParallelMLP

pytestmark = pytest.mark.gpu


def _mlp(hidden, inter, bits):
    g = torch.Generator(device="cuda")
    g.manual_seed(hidden + inter)

    def w(n, k):
        return (*_lib.quantize(torch.randn((n, k), generator=g, device="cuda").mul_(0.02), bits=bits), None)

    mlp = ParallelMLP(hidden, inter, 1, 0, use_quantized=True, quantization_bits=bits)
    mlp.load_quantized_shards(*w(inter, hidden), *w(hidden, inter), *w(inter, hidden))
    return mlp, g


def _product(mlp, x):
    gu = mlp.gate_up(x)
    return gu, _lib.act(gu, mlp.activation_name, gated=True)


@pytest.mark.parametrize("hidden,inter,bits", [(4096, 1024, 4), (8192, 512, 8), (512, 512, 4)])
@pytest.mark.parametrize("rows", [1, 6, 8, 9, 33, 100, 200, 1100])
def test_intermediate_matches_product_then_activation(device, hidden, inter, bits, rows):
    print(f"intermediate {hidden} -> {inter} W{bits} rows={rows}", flush=True)
    mlp, g = _mlp(hidden, inter, bits)
    x = torch.randn((rows, hidden), generator=g, device="cuda").to(torch.bfloat16)
    _, ref = _product(mlp, x)
    a = mlp.intermediate(x)
    if rows > 8:
        assert torch.equal(a, ref)
    else:
        assert (a.float() - ref.float()).abs().max() <= 2e-3 * ref.float().abs().max()
        assert (a != ref).double().mean() < 0.02


def test_intermediate_into_buffers(device):
    """``gu_out`` holds the product afterwards, ``out`` may be the input's own buffer (the
    product has read it by then)."""
    mlp, g = _mlp(512, 512, 4)
    for rows in (1, 8, 40, 300):
        x = torch.randn((rows, 512), generator=g, device="cuda").to(torch.bfloat16)
        gu_ref, ref = _product(mlp, x)
        gu = torch.full((rows, 1024), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert torch.equal(mlp.intermediate(x, gu_out=gu), ref) and torch.equal(gu, gu_ref)
        assert mlp.intermediate(x, out=x) is x and torch.equal(x, ref)
