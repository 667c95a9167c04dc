"""The SwiGLU product takes the library's split-K scratch only where the plain product does: a
K in one piece (one scale block, or tiles enough for one split) runs as a process's first
product under graph capture, which the scratch's allocation would break, and gives the bits
of the plain product and its activation."""
import os
import subprocess
import sys

import pytest
import torch

from shardcompute_amd import _lib

pytestmark = pytest.mark.gpu

_FIRST_CALL = r"""
import sys, torch
sys.path.insert(0, sys.argv[1])
from shardcompute_amd import _lib
M, I, K, bits = (int(v) for v in sys.argv[2:6])
g = torch.Generator(device="cuda"); g.manual_seed(M + I)
x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
w = _lib.quantize(torch.randn((2 * I, K), generator=g, device="cuda").mul_(0.02), bits=bits)
bias = torch.randn(2 * I, generator=g, device="cuda").to(torch.bfloat16)
act = torch.empty((M, I), dtype=torch.bfloat16, device="cuda")
gu = torch.empty((M, 2 * I), dtype=torch.bfloat16, device="cuda")
torch.cuda.synchronize()
graph = torch.cuda.CUDAGraph()
with torch.cuda.graph(graph):
    _lib.qmm_swiglu(x, *w, bias=bias, bits=bits, act_out=act, gate_up_scratch=gu)
ref = _lib.silu_mul(_lib.qmm(x, *w, bias=bias, bits=bits))
for r in range(3):
    act.fill_(float("nan"))
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(act, ref), f"replay {r}"
print("captured ok", flush=True)
"""


# band kernel: one scale block; 224 tiles of 128 rows; 16-column GEMV: 2048 tiles of 16 rows
@pytest.mark.parametrize("M,I,K,bits", [(24, 512, 512, 4), (100, 14336, 1024, 8), (12, 24576, 1024, 4)])
def test_unsplit_swiglu_takes_no_scratch(device, M, I, K, bits):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    print(f"fresh process: swiglu M={M} I={I} K={K} W{bits} first under capture", flush=True)
    p = subprocess.run([sys.executable, "-c", _FIRST_CALL, root, str(M), str(I), str(K), str(bits)],
                       capture_output=True, text=True, timeout=100, cwd=root)
    assert p.returncode == 0, p.stdout[-2000:] + p.stderr[-4000:]
    assert "captured ok" in p.stdout


def test_scratch_of_fewer_rows_is_left_alone(device):
    """gate_up_scratch is [rows, 2 I]; one of fewer rows is not written past its end (nor
    before it): the binding takes its own."""
    M, I, K, bits = 24, 512, 512, 4
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x = torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16)
    w = _lib.quantize(torch.randn((2 * I, K), generator=g, device="cuda").mul_(0.02), bits=bits)
    whole = torch.full((M, 2 * I), 7.0, dtype=torch.bfloat16, device="cuda")
    act, _ = _lib.qmm_swiglu(x, *w, bits=bits, gate_up_scratch=whole[:3])
    assert torch.equal(act, _lib.silu_mul(_lib.qmm(x, *w, bits=bits)))
    assert (whole == 7.0).all()
