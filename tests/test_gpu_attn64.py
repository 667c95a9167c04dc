"""Prefill attention at head_dim 64 against float64, on the 128-column kernel and on either
side of the rule that keeps the key-splitting kernel where its workgroups are few: positions
at the edges of a workgroup's columns (128 / R positions), GQA ratios 1 to 32, cached
prefixes, several 64-key blocks, garbage past the length, an additive mask.

The bound is the attention's, bf16 probabilities and outputs, for each row by itself:
|y - ref| <= 1e-2 |ref| in the 2-norm (probabilities and outputs each rounded by 2^-9 rms)."""
import math

import pytest
import torch

from shardcompute_amd import _lib

pytestmark = pytest.mark.gpu

D = 64


def _reference(q, k, v, past, mask):
    """q [B, H, S, D], k and v [B, Hkv, T, D] in float64."""
    B, H, S, _ = q.shape
    T, R = k.shape[2], H // k.shape[1]
    hidden = torch.arange(T, device=q.device)[None] > torch.arange(past, past + S, device=q.device)[:, None]
    out = torch.empty_like(q)
    for b in range(B):
        for h in range(H):
            s = q[b, h] @ k[b, h // R].T.contiguous() / math.sqrt(D)
            if mask is not None:
                s = s + mask[b].double()
            out[b, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[b, h // R]
    return out


# (B, S, H, Hkv, past, T_cap).  The first block runs on the key-splitting kernel (256 CUs: at
# most 528 workgroups of 16 columns there, with a mask 1024, or 512 for up to 256 positions or
# 128 slots, 256 more for a kv head per q head), the others on the 128-column one, those marked
# so without a mask only (the last two of them: few workgroups there, which would split the
# keys of a short cache)
CASES = [(1, 16, 32, 4, 0, 32), (2, 17, 32, 4, 47, 96), (1, 33, 16, 4, 0, 64), (2, 129, 4, 4, 5, 160),
         (1, 100, 8, 1, 300, 512), (1, 264, 32, 4, 400, 1024), (3, 150, 8, 8, 100, 352),
         (1, 265, 32, 4, 400, 1024), (1, 385, 32, 4, 400, 1024), (2, 129, 32, 32, 5, 160),       # no mask
         (3, 150, 8, 8, 0, 320), (2, 97, 16, 2, 60, 192),                                        # no mask
         (17, 16, 32, 4, 0, 32), (16, 17, 32, 4, 47, 96), (3, 200, 32, 4, 0, 224), (1, 517, 32, 4, 0, 544),
         (1, 515, 32, 4, 133, 672), (4, 129, 32, 32, 5, 160), (8, 70, 32, 8, 7, 96), (2, 530, 16, 1, 3, 544),
         (1, 520, 32, 1, 0, 544)]


@pytest.mark.parametrize("B,S,H,Hkv,past,T_cap", CASES)
@pytest.mark.parametrize("masked", [False, True])
def test_prefill_attention_head_dim_64(device, B, S, H, Hkv, past, T_cap, masked):
    print(f"attention64 B={B} S={S} H={H} Hkv={Hkv} past={past} T_cap={T_cap} masked={masked}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(S + past)
    T = past + S
    q = torch.randn((B * S, H * D), generator=g, device="cuda").to(torch.bfloat16)
    kc = torch.randn((B, Hkv, T_cap, D), generator=g, device="cuda").to(torch.bfloat16)
    vt = torch.randn((B, Hkv, D, T_cap), generator=g, device="cuda").to(torch.bfloat16)
    mask = None
    if masked:
        # left padding of the first key of odd rows and a random bias elsewhere
        mask = torch.randn((B, 1, 1, T), generator=g, device="cuda")
        if T > 1:
            mask[1::2, :, :, :1] = torch.finfo(torch.float32).min
    kd, vd = kc[:, :, :T].double(), vt[:, :, :, :T].double().transpose(2, 3).contiguous()
    kc[:, :, T:] = float("nan")
    vt[:, :, :, T:] = float("nan")
    cnt = torch.tensor([past, 0], dtype=torch.int32, device="cuda")
    out = _lib.attention(q, B, S, H, Hkv, D, kc, vt, cnt, 1 / math.sqrt(D), mask=mask, n_keys=T)
    torch.cuda.synchronize()
    ref = _reference(q.view(B, S, H, D).transpose(1, 2).double(), kd, vd, past,
                     None if mask is None else mask[:, 0])
    got = out.view(B, S, H, D).transpose(1, 2).double()
    assert torch.isfinite(got).all()
    assert ((got - ref).norm(dim=-1) <= 1e-2 * ref.norm(dim=-1)).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("masked", [False, True])
def test_prefill_softmax_sum_is_fp32(device, D, masked):
    """The probabilities meet V in bf16, their sum is that of the fp32 values.  One key block
    (no running maximum), so the result is known to its last bit but for the few elements
    whose probabilities lie within the scores' fp32 error (~2^-20) of a bf16 rounding
    boundary, ~1e-3 of them; a sum of the rounded values moves 4-5 % of them."""
    B, S, H, past = 30, 40, 8, 24
    T = past + S
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    q = torch.randn((B * S, H * D), generator=g, device="cuda").to(torch.bfloat16)
    kc = torch.randn((B, 1, T, D), generator=g, device="cuda").to(torch.bfloat16)
    vt = torch.randn((B, 1, D, T), generator=g, device="cuda").to(torch.bfloat16)
    mask = torch.randn((1, 1, 1, T), generator=g, device="cuda") if masked else None
    cnt = torch.tensor([past, 0], dtype=torch.int32, device="cuda")
    out = _lib.attention(q, B, S, H, 1, D, kc, vt, cnt, 1 / math.sqrt(D), mask=mask, n_keys=T).view(B, S * H, D)
    limit = torch.arange(past, T, device="cuda").repeat_interleave(H)
    s = torch.bmm(q.view(B, S * H, D).double(), kc[:, 0].double().transpose(1, 2).contiguous()) / math.sqrt(D)
    if masked:
        s = s + mask[0, 0].double()
    s = s.masked_fill(torch.arange(T, device="cuda") > limit[:, None], -math.inf)
    p = torch.exp(s - s.amax(-1, keepdim=True))
    o = torch.bmm(p.float().to(torch.bfloat16).double(), vt[:, 0].double().transpose(1, 2).contiguous())
    exact = (o / p.sum(-1, keepdim=True)).float().to(torch.bfloat16)
    assert (out != exact).double().mean() <= 0.01
