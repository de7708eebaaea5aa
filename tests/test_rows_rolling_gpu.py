"""Gate / up pairs of six and eight weight tiles on the few-row product (csrc/hip/gemm_rows_kernel.h), whose tiles are requested again one
by one, against a float64 product of the dequantized weights."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu


def _weight(n, k, qt, seed):
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.05
    raw = host.quantize(w, qt).view(torch.uint8)
    return host.relayout_to_device(raw, qt, n, k).cuda(), host.dequantize(raw, qt, w.shape).double()


# K: fewer k-tiles than wavefronts, one less, a cut last one, wavefronts with one and two, with two and three; N: a cut tile, a cut workgroup
@pytest.mark.parametrize("name", ["asym_int4", "woq_int4", "asym_int5", "sym_int8", "fp8_e4m3", "fp8_e5m2"])
@pytest.mark.parametrize("n,k", [(40, 128), (136, 896), (136, 1184), (72, 2304), (264, 4096)])
@pytest.mark.parametrize("m,norm", [(1, False), (3, True), (16, True), (16, False)])
def test_pair_matches_float64(name, n, k, m, norm):
    from bigdl_amd.ops import hip
    k = k if name != "woq_int4" else (k + 127) // 128 * 128
    eps, qt = 1e-5, Q.ggml_tensor_qtype[name]
    (dg, wg), (du, wu) = _weight(n, k, qt, 1), _weight(n, k, qt, 2)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(m, k, generator=g).half()
    gamma = (1 + 0.1 * torch.randn(k, generator=g)).half()
    xs, rs = x.double(), 1.0
    if norm:
        xs, rs = (x * gamma).double(), torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + eps)      # (rounded before the product)
    y, u = xs @ wg.t() * rs, xs @ wu.t() * rs
    ty, tu = (2.0 ** -16 * (xs.abs() @ w.abs().t()) * rs + 1e-5 for w in (wg, wu))          # exact codes, fp32 sums and scales
    silu = torch.nn.functional.silu
    for nt in (3, 4):
        out = hip.gemm_rows(x.cuda(), dg, qt, n, k, w2=du, act="silu", gamma=gamma.cuda() if norm else None, eps=eps,
                            out_dtype=torch.float32, nt=nt).double().cpu()
        assert ((out - silu(y) * u).abs() <= 1.2 * ty * u.abs() + tu * y.abs() + 1e-5).all(), nt
