"""Rotation and append of a short prompt (16 tokens a workgroup) against the same sequence inside a batch that takes 64 a workgroup: the
same bits in q, k, both caches and the unquantized values, and nothing else touched."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("s,past", [(1, 0), (15, 3), (16, 0), (17, 8), (63, 1), (77, 0), (130, 21)])
@pytest.mark.parametrize("d,rot,interleaved", [(64, 64, False), (96, 96, False), (128, 128, True), (128, 64, False), (256, 256, False), (80, 32, True)])
def test_short_prompt_like_a_batch(d, rot, interleaved, s, past, fp8):
    from bigdl_amd.ops import hip
    hq, hkv, lmax = 4, 2, 192
    # more workgroups than the rule's limit, but not so many that whole heads are taken (they round otherwise)
    batch = 6 * 128 // ((hq + 2 * hkv) * -(-s // 64)) + 1
    g = torch.Generator(device="cuda").manual_seed(s + d)
    qkv = torch.randn(batch, s, (hq + 2 * hkv) * d, device="cuda", generator=g).half()
    table = torch.randn(256, rot // 2, 2, device="cuda", generator=g)
    kind = torch.uint8 if fp8 else torch.float16

    def run(x):
        n = x.shape[0]
        kc, vc = torch.full((n, hkv, lmax, d), 7, dtype=kind, device="cuda"), torch.full((n, hkv, d, lmax), 7, dtype=kind, device="cuda")
        vt = torch.full((n, hkv, d, (s + 7) // 8 * 8), 7.0, dtype=torch.float16, device="cuda")
        x = x.clone()
        hip.prefill_rope_append(x, kc, vc, table, n_heads=hq, n_kv_heads=hkv, head_dim=d, past=past, rot_dim=rot, interleaved=interleaved,
                                vt_scratch=vt)
        return x, kc, vc, vt

    many = run(qkv)
    for b in (0, batch - 1):
        for one, all_ in zip(run(qkv[b:b + 1]), many):
            assert torch.equal(one[0], all_[b])
