"""The few-row low-bit product (csrc/hip/gemm_rows_kernel.h) against a float64 product of the dequantized weight."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu
FORMATS = ["sym_int4", "asym_int4", "woq_int4", "fp4", "nf4", "sym_int5", "asym_int5", "fp6", "sym_int8", "fp8_e4m3", "fp8_e5m2"]


@pytest.fixture(scope="module")
def hip():
    from bigdl_amd.ops import hip as h
    h.lib()
    return h


def _weight(n, k, qt, seed):
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.05
    raw = host.quantize(w, qt)
    raw = raw.view(torch.uint8) if raw.dtype != torch.uint8 else raw
    return host.relayout_to_device(raw, qt, n, k).cuda(), host.dequantize(raw, qt, w.shape).double()


def _x(m, k, seed):
    """[m, k] rows inside a buffer of NaN: what lies behind a row or below the last one must not be read as data"""
    buf = torch.full((m + 2, k + 24), float("nan"), dtype=torch.float16)
    buf[:m, :k] = torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).half()
    return buf.cuda()[:m, :k], buf[:m, :k].double()


def _close(out, x, w, ref, m, extra=0.0, nf4=False):
    # up to 16 rows the codes are exact in fp16 and the scale is applied in fp32: fp32 sums only (k * 2^-24 of the absolute
    # sum, bounded loosely), but for nf4, whose code values are a table in fp16 (2^-11 each).  More rows round
    # code * scale (+ min) to fp16: 2^-11 of a weight's larger term, on top of the table's, times two.
    bound = (2.0 ** -9 if m > 16 else 2.0 ** -11 if nf4 else 2.0 ** -16) * (x.abs() @ w.abs().t()) + 1e-5 + extra
    assert torch.isfinite(out).all()
    assert ((out.double().cpu() - ref).abs() <= bound).all()


# (rows, N, K): tile edges of rows and columns, a last k-tile that is cut, fewer k-tiles than wavefronts, one more than
# the tiles in flight
SHAPES = [(1, 16, 32), (6, 37, 2080), (16, 200, 1024), (17, 48, 96), (32, 65, 2304), (33, 130, 3232), (64, 80, 1184), (70, 33, 1024)]


@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("shape", SHAPES)
def test_every_tiling_matches_float64(hip, name, shape):
    m, n, k = shape
    k = k if name not in ("nf4", "woq_int4") else (k + 127) // 128 * 128
    qt = Q.ggml_tensor_qtype[name]
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k, 2)
    ref = xd @ w.t()
    mt = 1 if m <= 16 else 2 if m <= 32 else 4
    for nt in (0, 1, 2, 3) + ((4,) if mt < 4 else ()):
        _close(hip.gemm_rows(x, dev, qt, n, k, out_dtype=torch.float32, nt=nt), xd, w, ref, m, nf4=name == "nf4")
    parts = hip.gemm_rows(x, dev, qt, n, k, out_dtype=torch.float32, nt=2, splitk=3)
    if parts.dim() == 3:
        _close(parts.sum(0), xd, w, ref, m, nf4=name == "nf4")


@pytest.mark.parametrize("name", ["sym_int4", "asym_int5", "nf4", "sym_int8"])
@pytest.mark.parametrize("m", [3, 16, 24, 61])
def test_pairs_norm_bias_residual(hip, name, m):
    n, k, eps = 104, 1280, 1e-5
    qt = Q.ggml_tensor_qtype[name]
    (dg, wg), (du, wu) = _weight(n, k, qt, 3), _weight(n, k, qt, 4)
    x, xd = _x(m, k, 5)
    b1, b2 = torch.randn(n).half(), torch.randn(n).half()
    res = torch.randn(m, n).half()
    gamma = (1 + 0.1 * torch.randn(k)).half()
    silu = torch.nn.functional.silu
    for nt in (0, 1, 2):
        xn, kw = xd, {}
        if m <= 16:
            # x * gamma is rounded to fp16 before the product, so the reference multiplies those values
            xn = (xd.half() * gamma).double() * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + eps)
            kw = dict(gamma=gamma.cuda(), eps=eps)
        got = hip.gemm_rows(x, dg, qt, n, k, w2=du, bias=b1.cuda(), bias2=b2.cuda(), act="silu", out_dtype=torch.float32, nt=nt, **kw)
        ref = silu(xn @ wg.t() + b1.double()) * (xn @ wu.t() + b2.double())
        torch.testing.assert_close(got.cpu().double(), ref, rtol=4e-3, atol=8e-3)      # two products of 2^-9 and 2^-10 each, silu's slope 1.1
        out = res.cuda()
        hip.gemm_rows(x, dg, qt, n, k, bias=b1.cuda(), residual=out, out=out, nt=nt)    # in place, as on the residual stream
        torch.testing.assert_close(out.cpu().double(), xd @ wg.t() + b1.double() + res.double(), rtol=2e-3, atol=8e-3)


@pytest.mark.parametrize("name", ["sym_int4", "q4_k", "nf4", "sym_int8"])
@pytest.mark.parametrize("m", [4, 8, 13, 16, 17, 40, 64, 65, 192, 193])
def test_public_products_at_their_row_limits(hip, name, m):
    """gemv_lowbit / gemm_lowbit / gemm_lowbit_ex on either side of each change of kernel, K split included"""
    qt = Q.ggml_tensor_qtype[name]
    n, k = 272, 11008
    dev, w = _weight(n, k, qt, 6)
    x, xd = _x(m, k, 7)
    f = hip.gemv_lowbit if m <= 16 else hip.gemm_lowbit
    out = f(x, dev, qt, n, k, out_dtype=torch.float32)
    # (q4_k: the tiled scale d * sc6 and min dmin * m6 are fp16, 2^-11 of terms up to the block's range, taken as 0.4)
    _close(out, xd, w, xd @ w.t(), m if name != "q4_k" else 64, extra=0.0 if name != "q4_k" else 2.0 ** -11 * 0.4 * xd.abs().sum(-1, keepdim=True), nf4=name == "nf4")
    if m > 16:
        both = hip.gemm_lowbit_ex(x, dev, qt, n, k, w2=dev, act="silu")
        y = xd @ w.t()
        torch.testing.assert_close(both.cpu().double(), torch.nn.functional.silu(y) * y, rtol=1e-2, atol=0.15)     # y reaches 30: 2^-9 of y^2


@pytest.mark.parametrize("m,n,k", [(1, 16, 256), (5, 37, 512), (16, 130, 2304), (17, 48, 4096), (40, 33, 2816), (64, 80, 1024), (70, 20, 512)])
def test_q6k_blocks_without_expansion(hip, m, n, k):
    w0 = torch.randn(n, k, generator=torch.Generator().manual_seed(8)) * 0.05
    raw = host.quantize(w0, Q.Q6_K)
    w = host.dequantize(raw, Q.Q6_K, w0.shape).double()
    x, xd = _x(m, k, 9)
    ref = xd @ w.t()
    # code * sub-scale reaches 32 * 128: above 2048 it is rounded to 2^-11
    for nt in (0, 1, 2, 3):
        out = hip.gemm_rows(x, raw.cuda(), Q.Q6_K, n, k, out_dtype=torch.float32, nt=nt)
        bound = 2.0 ** -11 * (xd.abs() @ w.abs().t()) + 1e-5
        assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("m", [4, 16, 17, 32, 33, 64, 100, 128])
def test_q6k_weights_are_no_coarser_than_expanded_ones(hip, m):
    """One-hot rows read the weights as the product uses them: d * code * sub-scale with nothing rounded while code * sub-scale is
    at most 2048 (exact in fp16), rounded once to fp16 above; in the mean closer than weights expanded to fp16."""
    n, k = 64, 256
    raw = host.quantize(torch.randn(n, k, generator=torch.Generator().manual_seed(16)) * 0.05, Q.Q6_K)
    w = host.dequantize(raw, Q.Q6_K, (n, k)).double()                     # (exact: fp32 holds d * code * sub-scale)
    d = raw.view(torch.uint8).reshape(n, 210)[:, 208:].contiguous().view(torch.float16).double()
    exact = (w / d).abs() <= 2048
    assert 0.5 < exact.double().mean() < 0.99
    used = torch.zeros(n, k, dtype=torch.float64)
    for first in range(0, k, m):
        rows = min(m, k - first)
        x = torch.zeros(m, k, dtype=torch.float16)
        x[torch.arange(rows), first + torch.arange(rows)] = 1
        out = hip.gemm_q6k(x.cuda(), raw.view(torch.uint8).cuda(), n, k, out_dtype=torch.float32)
        used[:, first:first + rows] = out[:rows].t().cpu().double()
    off = (used - w).abs()
    assert (off <= torch.where(exact, 2.0 ** -22, 2.0 ** -11) * w.abs()).all()
    assert off.pow(2).mean() <= (w.half().double() - w).pow(2).mean()


# fewer rows than wavefronts, more than the grid holds at once, one block, a quad of blocks and one more, a full request
# group and one more, an LDS image of x that is too large (the last: the tile kernel)
@pytest.mark.parametrize("n,k", [(5, 256), (16, 1024), (9000, 1280), (33, 4096), (40, 4352), (64, 11008), (24, 28672)])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
def test_q6k_one_wavefront_a_row(hip, m, n, k):
    w0 = torch.randn(n, k, generator=torch.Generator().manual_seed(12)) * 0.05
    w0[0, :256] = 0                                                      # a block of scale 0
    raw = host.quantize(w0, Q.Q6_K)
    w = host.dequantize(raw, Q.Q6_K, w0.shape).double()
    x, xd = _x(m, k, 13)
    bias, res = torch.randn(n).half(), torch.randn(m, n).half()
    ref = torch.relu(xd @ w.t() + bias.double()) + res.double()
    # codes, scales and x exact in fp32: products and sums round (a lane's chain is k / 64 long).  Through the tile kernel
    # code * sub-scale rounds to 2^-11.
    bound = (2.0 ** -11 if m * k > 40960 else 2.0 ** -17) * (xd.abs() @ w.abs().t()) + 1e-5
    out = hip.gemm_rows(x, raw.cuda(), Q.Q6_K, n, k, out_dtype=torch.float32, bias=bias.cuda(), act="relu", residual=res.float().cuda())
    assert ((out.double().cpu() - ref).abs() <= bound).all()
    for dt, eps in ((torch.float16, 2.0 ** -10), (torch.bfloat16, 2.0 ** -7)):
        out = hip.gemm_rows(x, raw.cuda(), Q.Q6_K, n, k, out_dtype=dt)
        ref2 = xd @ w.t()
        assert ((out.double().cpu() - ref2).abs() <= bound + eps * ref2.abs() + 1e-7).all()


def test_q6k_linear_takes_the_blocks_for_few_rows(hip):
    from bigdl_amd.transformers.low_bit_linear import FP4Params, Q6K_MAX_ROWS, lowbit_matmul
    n, k = 96, 1024
    w0 = torch.randn(n, k, generator=torch.Generator().manual_seed(10)) * 0.05
    p = FP4Params(host.quantize(w0, Q.Q6_K), quantized=True, _shape=(n, k), qtype=Q.Q6_K).to("cuda")
    w = host.dequantize(p.data.cpu(), Q.Q6_K, (n, k)).double()
    for m in (1, Q6K_MAX_ROWS, Q6K_MAX_ROWS + 1):
        for dt, tol in ((torch.float16, 2e-3), (torch.float32, 2e-3), (torch.bfloat16, 1e-2)):
            x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dt)
            got = lowbit_matmul(x.cuda(), p, n)
            ref = x.double() @ w.t()
            assert got.dtype == dt
            # inputs and outputs of 2^-11 (2^-9 in bf16) on values of about 1.6
            torch.testing.assert_close(got.cpu().double(), ref, rtol=tol, atol=4 * tol)
    # strides and an offset that the kernel's 16-byte loads do not take
    x = torch.randn(3, k + 3, generator=torch.Generator().manual_seed(11)).half()[:, 3:]
    torch.testing.assert_close(lowbit_matmul(x.cuda(), p, n).cpu().double(), x.double() @ w.t(), rtol=2e-3, atol=8e-3)


@pytest.mark.parametrize("m", [1, 3, 40, 256, 300])
def test_nf4_table_is_exact_in_every_position(hip, m):
    """Every nf4 code in every position of a fragment, block scale 1 and one-hot rows: the products are the table, in fp16."""
    n, k, qt = 32, 512, Q.ggml_tensor_qtype["nf4"]
    grid = torch.linspace(-1, 1, 4096).reshape(64, 64).clone()
    grid[:, 0] = 1                                        # every block's scale
    table = host.dequantize(host.quantize(grid, qt), qt, (64, 64)).unique()
    assert len(table) == 16
    codes = torch.randint(0, 16, (n, k), generator=torch.Generator().manual_seed(7))
    codes[:, ::64] = 15                                   # 1.0: the block's largest value
    w = table[codes]
    dev = host.relayout_to_device(host.quantize(w, qt).view(torch.uint8), qt, n, k).cuda()
    want = w.half()
    assert torch.equal(hip.dequant_t16(dev, qt, n, k).cpu(), want)
    for first in range(0, k, m):
        x = torch.zeros(m, k, dtype=torch.float16)
        rows = min(m, k - first)
        x[torch.arange(rows), first + torch.arange(rows)] = 1
        product = hip.gemv_lowbit if m <= 16 else hip.gemm_lowbit
        if m <= 3 and first > 24:                         # (the other rows of a fragment come with the larger m)
            break
        assert torch.equal(product(x.cuda(), dev, qt, n, k).cpu()[:rows], want[:, first:first + rows].t())


@pytest.mark.parametrize("shape", [(16, 4096), (17, 4544), (300, 256), (1024, 64), (1024, 72), (511, 137)])
def test_half_of_bf16_matches_torch(hip, shape):
    """both sides of the 64 Ki line, an odd size; values beyond fp16's range, infinities, NaN and denormal results"""
    from bigdl_amd.transformers.low_bit_linear import _half
    x = torch.randn(shape, generator=torch.Generator().manual_seed(14)) * 10.0 ** torch.randint(-7, 6, shape, generator=torch.Generator().manual_seed(15))
    x.view(-1)[:6] = torch.tensor([float("inf"), -float("inf"), float("nan"), 65504.0, 65520.0, -1e30])
    x = x.bfloat16().cuda()
    # (with and without limits that bf16 rounds to 65536, which is infinite in fp16)
    for want in (x.to(torch.float16), x.clamp(-65504.0, 65504.0).to(torch.float16)):
        torch.testing.assert_close(_half(x), want, rtol=0, atol=0, equal_nan=True)
    sat = hip.bf16_to_f16(x)
    torch.testing.assert_close(sat, x.float().clamp(-65504.0, 65504.0).half() if x.numel() % 8 == 0 else x.half(), rtol=0, atol=0, equal_nan=True)
    xs = x[:, 1:]                                        # not contiguous
    torch.testing.assert_close(_half(xs), xs.to(torch.float16), rtol=0, atol=0, equal_nan=True)
