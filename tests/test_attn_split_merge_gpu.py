"""Ranges of keys whose partial results meet in the workgroup that arrives last: launch after launch on one workspace, so that a read
of an earlier launch's numbers shows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("d,hq,hkv,batch", [(64, 8, 2, 9), (128, 32, 8, 12), (128, 40, 8, 3), (256, 8, 4, 5)])
def test_launch_after_launch(d, hq, hkv, batch, fp8):
    from bigdl_amd.ops import hip
    lmax, past, rounds = 2304, 2200, 6
    g = torch.Generator(device="cuda").manual_seed(d + hq)
    dev = dict(device="cuda", generator=g)
    past_len = torch.full((batch,), past, dtype=torch.int32, device="cuda")
    for splits in (2, 5, 17):
        ws = torch.full((hip.attn_decode_ws_floats(batch, hq, hkv, 1, d, splits),), 3e4, device="cuda")
        counters = torch.zeros(hip.attn_decode_counters(batch, hq, hkv), dtype=torch.int32, device="cuda")
        data, outs = [], []
        for i in range(rounds):
            k = torch.randn(batch, hkv, lmax, d, **dev).half()
            v = (torch.randn(batch, hkv, d, lmax, **dev) + (-1) ** i * 4).half()      # each launch's results are far from the last one's
            if fp8:
                k8, v8 = torch.empty_like(k, dtype=torch.uint8), torch.empty_like(v, dtype=torch.uint8)
                hip.to_e5m2(k, k8)
                hip.to_e5m2(v, v8)
                k, v = k8, v8
            data.append((torch.randn(batch, (hq + 2 * hkv) * d, **dev).half(), k, v))
            outs.append([torch.empty(batch, hq * d, dtype=torch.float16, device="cuda") for _ in range(2)])

        def launch(i, n, out):
            qkv, k, v = data[i]
            hip.attn_decode(qkv, k, v, past_len, out, ws, counters, n_heads=hq, n_kv_heads=hkv, head_dim=d, q_len=1, batch=batch,
                            scale=d ** -0.5, splits=n)

        for i in range(rounds):
            launch(i, splits, outs[i][0])
        for i in range(rounds):
            launch(i, 1, outs[i][1])
        assert int(counters.abs().sum()) == 0
        # both are sums of values with weights rounded to fp16 (e5m2: two e4m3 terms, 2^-8) and a result in fp16
        vmax = 4 + 6.0
        bound = 2 * vmax * ((2.0 ** -8 if fp8 else 2.0 ** -11) + 2.0 ** -11)
        for got, one in outs:
            assert (got.float() - one.float()).abs().max().item() <= bound, splits
