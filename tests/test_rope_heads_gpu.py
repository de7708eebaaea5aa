"""Prompt RoPE + append where a workgroup takes several whole heads (csrc/hip/attn_prefill.hip): token counts around its 64-token
blocks, head counts that its share does not divide, earlier tokens, explicit positions, both cache types."""
import pytest
import torch

from bigdl_amd.ops import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("b,s,hq,hkv,d,past,ids", [(3, 1101, 13, 7, 128, 0, False), (1, 4096, 32, 8, 64, 5, False), (2, 1665, 30, 11, 128, 3, True),
                                                   (1, 8191, 17, 1, 64, 0, False), (5, 1, 210, 3, 128, 9, False), (5, 65, 100, 10, 64, 0, False),
                                                   (1, 6000, 41, 6, 128, 1, False)])
def test_whole_heads(fp8, b, s, hq, hkv, d, past, ids):
    torch.manual_seed(s)
    lmax = (past + s + 300) // 256 * 256
    qkv = torch.randn(b, s, (hq + 2 * hkv) * d, device="cuda").half()
    was = qkv.clone()
    half = d // 2
    ang = torch.arange(lmax, device="cuda").float()[:, None] / (10000 ** (torch.arange(half, device="cuda").float() / half))
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    dt = torch.uint8 if fp8 else torch.float16
    kc, vc = (torch.zeros(b, hkv, *shape, dtype=dt, device="cuda") for shape in ((lmax, d), (d, lmax)))
    pos = torch.arange(past, past + s, device="cuda").expand(b, s)
    pos = (pos * 7 % lmax).contiguous() if ids else pos
    hip.prefill_rope_append(qkv, kc, vc, table, n_heads=hq, n_kv_heads=hkv, head_dim=d, past=past, position_ids=pos if ids else None)
    x = was.view(b, s, hq + 2 * hkv, d)[:, :, : hq + hkv].double()
    c, n = table[pos, :, 0].double()[:, :, None], table[pos, :, 1].double()[:, :, None]
    x0, x1 = x[..., :half], x[..., half:]
    ref = torch.cat([x0 * c - x1 * n, x1 * c + x0 * n], -1)
    got = qkv.view(b, s, hq + 2 * hkv, d)
    # two products and a sum in fp32 (3 x 2^-24 of their size, below 16 here), then fp16: 2^-11, or 2^-25 below its normal numbers
    assert ((got[:, :, : hq + hkv].double() - ref).abs() <= ref.abs() * 2.0 ** -11 + 48 * 2.0 ** -24).all()
    v = got[:, :, hq + hkv:].permute(0, 2, 3, 1)
    assert torch.equal(got[:, :, hq + hkv:], was.view(b, s, hq + 2 * hkv, d)[:, :, hq + hkv:])
    k = got[:, :, hq: hq + hkv].permute(0, 2, 1, 3)
    to = (lambda t: t.to(torch.float8_e5m2).view(torch.uint8)) if fp8 else (lambda t: t)
    assert torch.equal(kc[:, :, past:past + s], to(k)) and torch.equal(vc[..., past:past + s], to(v))
    assert not kc[:, :, :past].any() and not kc[:, :, past + s:].any() and not vc[..., :past].any() and not vc[..., past + s:].any()
