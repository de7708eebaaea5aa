"""A single routed slot (one token, one expert) on either side of the 16-wavefront form: 32 k-tiles, 256 column tiles."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "nf4", "sym_int8"])
@pytest.mark.parametrize("n,k", [(32, 3968), (32, 4096), (32, 4160), (4096, 4096), (4112, 4096), (48, 8192)])
def test_single_slot(name, n, k):
    from bigdl_amd.ops import hip
    qt, e = Q.ggml_tensor_qtype[name], 3
    k = k if name != "nf4" else (k + 127) // 128 * 128
    w = torch.randn(e * n, k, generator=torch.Generator().manual_seed(1)) * 0.05
    raw = host.quantize(w, qt).view(torch.uint8)
    dev = host.relayout_to_device(raw, qt, e * n, k).cuda()
    w = host.dequantize(raw, qt, w.shape).double().view(e, n, k)
    x = torch.randn(1, k, generator=torch.Generator().manual_seed(2)).half()
    gamma = (1 + 0.1 * torch.randn(k, generator=torch.Generator().manual_seed(3))).half()
    scale = torch.tensor([0.75])
    xn = (x * gamma).double() * torch.rsqrt(x.double().pow(2).mean() + 1e-5)     # (x * gamma is rounded to fp16 first)
    for expert in (0, 2, -1):
        ids = torch.tensor([expert], dtype=torch.int32).cuda()
        plain = hip.gemv_lowbit_moe(x.cuda(), dev, qt, e, n, k, ids)
        full = hip.gemv_lowbit_moe(x.cuda(), dev, qt, e, n, k, ids, slot_scale=scale.cuda(), gamma=gamma.cuda(), eps=1e-5, act="silu")
        if expert < 0:
            assert not plain.any() and not full.any()
            continue
        y, z = x.double() @ w[expert].t(), torch.nn.functional.silu(xn @ w[expert].t()) * 0.75
        # fp32 sums, nf4's code table in fp16 (2^-11 each), results in fp16 (2^-11)
        for got, ref, rows in ((plain, y, x.double()), (full, z, xn)):
            bound = (2.0 ** -10 if name == "nf4" else 2.0 ** -15) * (rows.abs() @ w[expert].abs().t()) + 2.0 ** -11 * ref.abs() + 1e-5
            assert ((got.cpu().double() - ref).abs() <= bound).all()
