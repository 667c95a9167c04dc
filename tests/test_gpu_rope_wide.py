"""The one-launch rotation and cache append of many positions against the wave-per-head kernel.

A call whose rows are not 16-byte aligned takes the latter, whose arithmetic the wide kernel
repeats element by element: the rotated q, the keys and the values are equal bit for bit."""
import pytest
import torch

from shardcompute_amd import _lib

pytestmark = pytest.mark.gpu


# S at the edges of the 64-token v tile and of the four-token workgroups, more heads than a
# wave takes at once and fewer, cached positions, a rotary offset
@pytest.mark.parametrize("B,S,H,Hkv,D,past,offset", [(1, 16, 32, 8, 128, 0, 0), (2, 65, 32, 4, 64, 31, 0),
                                                     (3, 63, 8, 1, 128, 5, 7), (1, 129, 2, 2, 64, 3, 0),
                                                     (1, 257, 20, 4, 128, 0, 0)])
def test_wide_equals_wave_per_head(device, B, S, H, Hkv, D, past, offset):
    print(f"rope wide B={B} S={S} H={H} Hkv={Hkv} D={D} past={past}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(S)
    T, W = (past + S + 31) // 32 * 32, (H + 2 * Hkv) * D
    rows = torch.randn((B * S, W), generator=g, device="cuda").to(torch.bfloat16)
    ang = torch.rand((T + offset, D // 2), generator=g, device="cuda") * 6
    cnt = torch.tensor([past, 0], dtype=torch.int32, device="cuda")
    out = []
    for shift in (0, 1):       # the tables 16-byte aligned, and 4 bytes off
        cos, sin = (torch.empty(ang.numel() + 4, device="cuda")[shift:shift + ang.numel()].view_as(ang).copy_(f)
                    for f in (ang.cos(), ang.sin()))
        qkv = rows.clone()
        kc = torch.zeros((B, Hkv, T, D), dtype=torch.bfloat16, device="cuda")
        vt = torch.zeros((B, Hkv, D, T), dtype=torch.bfloat16, device="cuda")
        _lib.rope_append_kv(qkv, B, S, H, Hkv, D, cos, sin, kc, vt, cnt, pos_offset=offset)
        out.append((qkv, kc, vt))
    for a, b in zip(*out):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert torch.equal(out[0][2][:, :, :, past:past + S],
                       rows.view(B, S, H + 2 * Hkv, D)[:, :, H + Hkv:].permute(0, 2, 3, 1))
    assert not out[0][1][:, :, past + S:].any() and not out[0][2][..., past + S:].any()
