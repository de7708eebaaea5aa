"""Where the decode attention puts a new key's values: a step's V^T column, its neighbours, and the block edges of the fp16 cache."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,hkv,group", [(64, 2, 4), (128, 2, 1), (96, 1, 2)])
@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("past", [0, 1, 31, 32, 255, 256, 300, 511])
def test_a_new_value_row_lands_in_its_column_only(d, hkv, group, splits, past):
    from bigdl_amd.ops import hip
    g = torch.Generator().manual_seed(past + d)
    b, cap, hq = 2, 512, hkv * group
    qkv = torch.randn(b, (hq + 2 * hkv) * d, generator=g).half()
    k = torch.randn(b, hkv, cap, d, generator=g).half()
    vt = torch.randn(b, hkv, d, cap, generator=g).half()
    kc, vc, q2 = k.cuda(), vt.cuda(), qkv.cuda()
    lens = torch.full((b,), past, dtype=torch.int32, device="cuda")
    table = torch.zeros(cap, d // 2, 2)
    table[..., 0] = 1.0                                     # no rotation: keys and queries as they are
    out = torch.empty(b, hq * d, dtype=torch.float16, device="cuda")
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, 1, d, splits) + 16, device="cuda")
    cnt = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    hip.attn_decode(q2, kc, vc, lens, out, ws, cnt, n_heads=hq, n_kv_heads=hkv, head_dim=d, q_len=1, batch=b, scale=d ** -0.5,
                    splits=splits, rope_table=table.cuda())
    newk = qkv[:, hq * d:(hq + hkv) * d].view(b, hkv, d)
    newv = qkv[:, (hq + hkv) * d:].view(b, hkv, d)
    k[:, :, past], vt[:, :, :, past] = newk, newv
    assert torch.equal(vc.cpu(), vt) and torch.equal(kc.cpu(), k)
    q = qkv[:, :hq * d].view(b, hkv, group, d).double()
    p = torch.softmax(q @ k[:, :, :past + 1].double().transpose(-1, -2) * d ** -0.5, -1)
    ref = (p @ vt[..., :past + 1].double().transpose(-1, -2)).reshape(b, hq * d)
    # probabilities and outputs of 2^-11 on values up to about 4
    torch.testing.assert_close(out.cpu().double(), ref, rtol=2e-3, atol=4e-3)


# the most query heads a kv head that one row tile holds, one more (two tiles), heads of 256, and more heads a kv head than a
# workgroup takes (two workgroups a kv head append the same row)
@pytest.mark.parametrize("d,hkv,group", [(128, 2, 16), (96, 1, 17), (128, 1, 32), (128, 1, 40), (256, 2, 2)])
@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("past", [0, 31, 256, 511])
def test_groups_of_many_heads_and_wide_heads(d, hkv, group, splits, past):
    test_a_new_value_row_lands_in_its_column_only(d, hkv, group, splits, past)
