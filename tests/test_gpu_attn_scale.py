"""Prefill attention for scales outside the usual 1 / sqrt(head_dim): zero (uniform weights),
negative, and very small and large ones, at sizes that the 128-column kernel takes otherwise.

Bound: bf16 probabilities and outputs, per query row |y - ref| <= 1e-2 of the row's 2-norm."""
import math

import pytest
import torch

from shardcompute_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [0.0, -0.125, -1.0, 1e-38, -1e-38, 2.0])
@pytest.mark.parametrize("masked", [False, True])
def test_prefill_attention_any_scale(device, D, scale, masked):
    B, S, H, Hkv, past, cap = 4, 520, 8, 1, 20, 544
    print(f"attention scale={scale} D={D} masked={masked}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    T = past + S
    q = torch.randn((B * S, H * D), generator=g, device="cuda").to(torch.bfloat16)
    kc = torch.randn((B, Hkv, cap, D), generator=g, device="cuda").to(torch.bfloat16)
    vt = torch.randn((B, Hkv, D, cap), generator=g, device="cuda").to(torch.bfloat16)
    mask = torch.randn((B, 1, 1, T), generator=g, device="cuda") if masked else None
    if masked:
        mask[1, :, :, :3] = -math.inf
    cnt = torch.tensor([past, 0], dtype=torch.int32, device="cuda")
    out = _lib.attention(q, B, S, H, Hkv, D, kc, vt, cnt, scale, mask=mask, n_keys=T)
    torch.cuda.synchronize()
    hidden = torch.arange(T, device="cuda")[None] > torch.arange(past, T, device="cuda")[:, None]
    for b in range(B):
        v = vt[b, 0, :, :T].double().T.contiguous()
        for h in range(H):
            s = (q.view(B, S, H, D)[b, :, h].double() @ kc[b, 0, :T].double().T.contiguous()) * scale
            if masked:
                s = s + mask[b, 0].double()
            ref = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v
            got = out.view(B, S, H, D)[b, :, h].double()
            assert torch.isfinite(got).all(), (b, h)
            assert ((got - ref).abs().amax(-1) <= 1e-2 * ref.norm(dim=-1)).all(), (b, h)
