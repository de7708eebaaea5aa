"""The loop of the prompt product (csrc/hip/gemm_prompt_kernel.h) where its look-ahead is longer than K, and every tile
configuration around its edges, against float64."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu

TILES = [(256, 256), (256, 192), (128, 128), (256, 128), (192, 256), (192, 128)]


@pytest.fixture()
def hip():
    from bigdl_amd.ops import hip as h
    h.lib()
    yield h
    h.gemm_prompt_force()


def _weight(n, k, qt, seed):
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.05
    raw = host.quantize(w, qt)
    return host.relayout_to_device(raw, qt, n, k).cuda(), host.dequantize(raw, qt, w.shape).double()


def _x(m, k):
    """rows k + 8 apart, NaN behind each and behind the last one"""
    buf = torch.full((m + 1, k + 8), float("nan"), dtype=torch.float16)
    buf[:m, :k] = torch.randn(m, k, generator=torch.Generator().manual_seed(3)).half()
    return buf.cuda()[:m, :k], buf[:m, :k].double()


# one k tile of 128 a split, two, three (odd), seven: shorter than, as long as and longer than what is requested ahead
@pytest.mark.parametrize("k,splitk", [(256, 2), (256, 1), (384, 1), (896, 1), (896, 3)])
@pytest.mark.parametrize("cfg", range(6))
def test_short_and_odd_k(hip, cfg, k, splitk):
    bm, bn = TILES[cfg]
    m, n, qt = bm + 1, bn + 24, Q.SYM_INT4               # a second row block of one row, a column block with half a weight tile
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k)
    hip.gemm_prompt_force(cfg, splitk)
    ref = xd @ w.t()
    # fp16 weight (2^-11 of each term) and output
    bound = 2.0 ** -10 * (xd.abs() @ w.abs().t()) + 2.0 ** -10 * ref.abs()
    for _ in range(3):
        out = hip.gemm_prompt(x, dev, qt, n, k)
        assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("qname", ["asym_int4", "fp4", "nf4", "sym_int5", "asym_int5", "fp6", "sym_int8", "fp8_e4m3", "fp8_e5m2"])
@pytest.mark.parametrize("cfg", range(6))
def test_every_format_in_every_tile(hip, cfg, qname):
    bm, bn = TILES[cfg]
    m, n, k, qt = bm - 1, bn - 8, 640, Q.ggml_tensor_qtype[qname]
    dev, w = _weight(n, k, qt, 2)
    x, xd = _x(m, k)
    hip.gemm_prompt_force(cfg, 1)
    out = hip.gemm_prompt(x, dev, qt, n, k)
    ref = xd @ w.t()
    # codes times scale (and minimum) in fp16: 2^-11 of each weight, and of its minimum, which is at most the largest of its block of 32
    top = w.abs().view(n, k // 32, 32).amax(-1, keepdim=True).expand(n, k // 32, 32).reshape(n, k)
    assert ((out.double().cpu() - ref).abs() <= 2.0 ** -10 * (xd.abs() @ top.t()) + 2.0 ** -10 * ref.abs()).all()


@pytest.mark.parametrize("act", ["silu", "gelu", None])
@pytest.mark.parametrize("cfg", range(6))
def test_pairs(hip, cfg, act):
    bm, bn = TILES[cfg]
    m, n, k, qt = bm + 17, bn // 2 + 16, 384, Q.SYM_INT4
    (dg, wg), (du, wu) = _weight(n, k, qt, 4), _weight(n, k, qt, 5)
    x, xd = _x(m, k)
    hip.gemm_prompt_force(cfg, 1)
    out = hip.gemm_prompt_pair(x, dg, du, qt, n, k, act=act)
    g, u = xd @ wg.t(), xd @ wu.t()
    f = {"silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu, None: lambda t: t}[act]
    ref = f(g) * u
    # both factors round to fp16 (|f'| <= 1.13), the weights too, then the product rounds
    e = 2.0 ** -11
    eg = e * g.abs() + 2.0 ** -10 * (xd.abs() @ wg.abs().t())
    eu = e * u.abs() + 2.0 ** -10 * (xd.abs() @ wu.abs().t())
    bound = 1.13 * eg * u.abs() + f(g).abs() * eu + 1.13 * eg * eu + e * ref.abs() + 1e-4
    assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gate_where_the_exponential_is_largest(hip, dtype):
    """silu(g) u for g down to where 1 + e^-g overflows: the products of zero rows are the biases"""
    n, k, qt = 256, 256, Q.SYM_INT4
    dev, _ = _weight(n, k, qt, 3)
    g = torch.linspace(-100, 100, n - 64).bfloat16().half()
    g = torch.cat([torch.arange(-96, -80, 0.25).bfloat16().half(), g])
    u = torch.full((n,), 2.0 ** 15).half()
    out = hip.gemm_prompt_pair(torch.zeros(300, k, dtype=torch.float16, device="cuda"), dev, dev, qt, n, k, bias=g.cuda(), bias2=u.cuda(),
                               act="silu", out_dtype=dtype)
    ref = g.double() / (1 + torch.exp(-g.double())) * 2.0 ** 15
    # e^-g overflows fp32 below -88.72, which leaves zero; else the result's rounding, e^x to 2^-17 at 2^7, fp16's smallest steps
    ref = torch.where(g.double() < -88.72, 0.0, ref).clamp(-torch.finfo(dtype).max, torch.finfo(dtype).max)
    bound = (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7) * ref.abs() + (2.0 ** -24 if dtype == torch.float16 else 1e-38)
    ok = (out.double().cpu() - ref).abs() <= bound
    big = ref.abs() >= torch.finfo(dtype).max                 # (beyond fp16: infinite)
    assert (ok | big).all(), (g[~(ok | big).all(0)], out[0].cpu()[~(ok | big).all(0)])
