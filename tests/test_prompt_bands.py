"""Tile order of the prompt product in bands of four row blocks and its shared gate / up epilogue, against float64."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu


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
    buf = torch.full((m + 1, k + 8), float("nan"), dtype=torch.float16)
    buf[:m, :k] = torch.randn(m, k, generator=torch.Generator().manual_seed(3)).half()
    return buf.cuda()[:m, :k], buf[:m, :k].double()


# row blocks: one, a whole band, a band and one block (cut), two bands and three; configuration 2 has 128-row tiles, 0 and 1 256
@pytest.mark.parametrize("cfg,m", [(2, 1), (2, 512), (2, 513), (2, 1400), (0, 1030), (1, 1300)])
@pytest.mark.parametrize("splitk", [1, 2])
def test_every_tile_of_every_band(hip, cfg, m, splitk):
    n, k, qt = 440, 512, Q.SYM_INT4
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k)
    hip.gemm_prompt_force(cfg, splitk)
    out = hip.gemm_prompt(x, dev, qt, n, k)
    ref = xd @ w.t()
    # fp16 weight (2^-11 of each term) and output
    assert ((out.double().cpu() - ref).abs() <= 2.0 ** -10 * (xd.abs() @ w.abs().t()) + 2.0 ** -10 * ref.abs()).all()


# either side of 256 tiles, where the order changes from whole columns to bands: 4 x 64 and 4 x 65 tiles, 11 x 24 (the last band
# three blocks high), 5 x 52 of 256 columns; as a pair 9 x 29 tiles of 64 columns
@pytest.mark.parametrize("cfg,m,n,pair", [(2, 500, 8192, False), (2, 500, 8200, False), (2, 1400, 3072, False), (0, 1030, 13312, False),
                                          (2, 1100, 1856, True)])
def test_more_tiles_than_compute_units(hip, cfg, m, n, pair):
    k, qt = 256, Q.SYM_INT4
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k)
    hip.gemm_prompt_force(cfg, 1)
    ref = xd @ w.t()
    bound = 2.0 ** -10 * (xd.abs() @ w.abs().t()) + 2.0 ** -10 * ref.abs()
    if pair:
        out = hip.gemm_prompt_pair(x, dev, dev, qt, n, k, act="relu")
        # the same product twice, so f(y) = max(y, 0) * y: twice the product's error times |y|, and one more rounding
        bound, ref = 2 * bound * (ref.abs() + bound) + 2.0 ** -10 * ref * ref, ref.relu() * ref
    else:
        out = hip.gemm_prompt(x, dev, qt, n, k)
    assert ((out.double().cpu() - ref).abs() <= bound + 1e-6).all()


@pytest.mark.parametrize("cfg,m", [(2, 130), (2, 700), (0, 1030), (1, 257)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_both_halves_of_a_pair_write_their_rows(hip, cfg, m, dtype):
    n, k, qt = 304, 512, Q.SYM_INT4
    (dg, wg), (du, wu) = _weight(n, k, qt, 4), _weight(n, k, qt, 5)
    x, xd = _x(m, k)
    hip.gemm_prompt_force(cfg, 1)
    out = hip.gemm_prompt_pair(x, dg, du, qt, n, k, act="silu", out_dtype=dtype)
    g, u = xd @ wg.t(), xd @ wu.t()
    ref = torch.nn.functional.silu(g) * u
    # both factors round to the output type (|silu'| <= 1.1), the weights to fp16, then the product rounds
    e = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    eg = e * g.abs() + 2.0 ** -10 * (xd.abs() @ wg.abs().t())
    eu = e * u.abs() + 2.0 ** -10 * (xd.abs() @ wu.abs().t())
    bound = 1.1 * eg * u.abs() + torch.nn.functional.silu(g).abs() * eu + 1.1 * eg * eu + e * ref.abs() + 1e-4
    assert ((out.double().cpu() - ref).abs() <= bound).all()
