"""The skinny product (csrc/hip/gemv_kernel.h) of one to five rows, whose partial sums meet by lane groups up to four rows, against a
float64 product of the dequantized weight."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu


def _weight(n, k, qt, seed):
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.05
    raw = host.quantize(w, qt).view(torch.uint8)
    return host.relayout_to_device(raw, qt, n, k).cuda(), host.dequantize(raw, qt, w.shape).double()


# K of the lean form, of 8 wavefronts with a staging loop, of 16 wavefronts, of x that is not staged (four rows and more); N with a last tile that
# is cut; rows of one lane group (up to four) and of all
@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "sym_int8", "fp4", "asym_int5"])
@pytest.mark.parametrize("n,k", [(72, 1024), (40, 4096), (24, 9216), (24, 20480)])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 16])
def test_rows_norm_bias_residual_pair(name, n, k, m):
    from bigdl_amd.ops import hip
    eps, qt = 1e-5, Q.ggml_tensor_qtype[name]
    (dg, wg), (du, wu) = _weight(n, k, qt, 1), _weight(n, k, qt, 2)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(m, k, generator=g).half()
    gamma = (1 + 0.1 * torch.randn(k, generator=g)).half()
    b1, b2, res = torch.randn(n, generator=g).half(), torch.randn(n, generator=g).half(), torch.randn(m, n, generator=g).half()
    # x * gamma is rounded to fp16 before the product
    xs, rs = (x * gamma).double(), torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + eps)
    y = xs @ wg.t() * rs + b1.double()
    u = xs @ wu.t() * rs + b2.double()
    kw = dict(gamma=gamma.cuda(), eps=eps, out_dtype=torch.float32)
    one = hip.gemv_lowbit(x.cuda(), dg, qt, n, k, bias=b1.cuda(), residual=res.float().cuda(), **kw).double().cpu()
    two = hip.gemv_lowbit(x.cuda(), dg, qt, n, k, w2=du, bias=b1.cuda(), bias2=b2.cuda(), act="silu", **kw).double().cpu()
    half = hip.gemv_lowbit(x.cuda(), dg, qt, n, k, residual=res.cuda()).double().cpu()
    # exact codes, scales in fp32: fp32 sums (k 2^-24 of the absolute sum, bounded loosely), for the pair times the factor's size
    tol = 2.0 ** -16 * (xs.abs() @ wg.abs().t()) * rs + 1e-5
    tol_u = 2.0 ** -16 * (xs.abs() @ wu.abs().t()) * rs + 1e-5
    assert ((one - y - res.double()).abs() <= tol).all()
    silu = torch.nn.functional.silu
    assert ((two - silu(y) * u).abs() <= 1.2 * tol * u.abs() + tol_u * y.abs() + 1e-5).all()
    ref = x.double() @ wg.t() + res.double()
    assert ((half - ref).abs() <= 2.0 ** -10 * ref.abs() + 2.0 ** -16 * (x.double().abs() @ wg.abs().t()) + 1e-5).all()
