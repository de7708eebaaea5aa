"""The low-bit product on x in fragment order (csrc/hip/gemm_frag_kernel.h) against a float64 product of the dequantized weight."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu
FORMATS = ["sym_int4", "asym_int4", "woq_int4", "fp4", "nf4", "sym_int5", "asym_int5", "fp6", "sym_int8", "fp8_e4m3", "fp8_e5m2"]
TILINGS = [(3, 2), (3, 3), (3, 4), (3, 6), (4, 2), (4, 3), (4, 4), (4, 6), (4, 8), (5, 3), (5, 4), (5, 6), (5, 8), (6, 2), (6, 4), (6, 6),
           (7, 3), (7, 4), (8, 3), (8, 4)]


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


def _x(m, k, seed, dtype=torch.float16):
    """[m, k] rows inside a buffer of NaN: what lies behind a row or below the last one must not be read as data"""
    buf = torch.full((m + 2, k + 24), float("nan"), dtype=dtype)
    buf[:m, :k] = torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).to(dtype)
    return buf.cuda()[:m, :k], buf[:m, :k].half().double()


def _close(out, x, w, ref):
    # code * scale (+ min) is rounded to fp16: 2^-11 of a weight's larger term, on top of the table's of nf4, times two
    bound = 2.0 ** -9 * (x.abs() @ w.abs().t()) + 1e-5
    assert torch.isfinite(out).all()
    assert ((out.double().cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("m,k", [(1, 32), (16, 128), (77, 2080), (130, 1184)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fragment_order(hip, m, k, dtype):
    x, xd = _x(m, k, 1, dtype)
    kt, mt = (k + 127) // 128, (m + 15) // 16
    want = torch.zeros(mt * 16, kt * 128, dtype=torch.float64)
    want[:m, :k] = xd
    # [k step][row tile][k group][row][8]
    want = want.view(mt, 16, kt * 4, 4, 8).permute(2, 0, 3, 1, 4).reshape(-1)
    assert torch.equal(hip.frag_pack(x).cpu().double(), want)


# (rows, N, K): cut row and column tiles, a cut last k-tile, fewer k-tiles than wavefronts, one more than those in flight
@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (33, 130, 3232), (77, 37, 2080), (113, 200, 1024), (203, 80, 1184)])
def test_every_tiling_matches_float64(hip, name, m, n, k):
    k = k if name not in ("nf4", "woq_int4") else (k + 127) // 128 * 128
    qt = Q.ggml_tensor_qtype[name]
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k, 2)
    xp = hip.frag_pack(x)
    ref = xd @ w.t()
    for mt, ns in TILINGS:
        _close(hip.gemm_frag(xp, m, dev, qt, n, k, out_dtype=torch.float32, mt=mt, ns=ns), xd, w, ref)
    parts = hip.gemm_frag(xp, m, dev, qt, n, k, out_dtype=torch.float32, mt=4, ns=3, splitk=3)
    if parts.dim() == 3:
        _close(parts.sum(0), xd, w, ref)


@pytest.mark.parametrize("name", ["sym_int4", "asym_int5", "nf4", "sym_int8"])
@pytest.mark.parametrize("m,n", [(24, 104), (77, 70), (130, 33)])
def test_pairs_bias_residual(hip, name, m, n):
    k = 1280
    qt = Q.ggml_tensor_qtype[name]
    (dg, wg), (du, wu) = _weight(n, k, qt, 3), _weight(n, k, qt, 4)
    x, xd = _x(m, k, 5)
    xp = hip.frag_pack(x)
    g = torch.Generator().manual_seed(8)
    b1, b2 = torch.randn(n, generator=g).half(), torch.randn(n, generator=g).half()
    silu = torch.nn.functional.silu
    # each product is off by _close's bound at most; silu is 1.1 steep at most.  Over all values the errors of the weights' roundings,
    # 2^-11 each and nf4's table again, are independent: 2^-10.5 of a product, twice with that slope of a pair
    first, second = xd @ wg.t() + b1.double(), xd @ wu.t() + b2.double()
    e1, e2 = (2.0 ** -9 * (xd.abs() @ w.abs().t()) + 1e-5 for w in (wg, wu))
    ref, bound = silu(first) * second, 1.1 * e1 * (second.abs() + e2) + e2 * silu(first).abs()
    for mt, ns in [t for t in TILINGS if t[1] % 2 == 0]:
        got = hip.gemm_frag(xp, m, dg, qt, n, k, w2=du, bias=b1.cuda(), bias2=b2.cuda(), act="silu", out_dtype=torch.float32, mt=mt, ns=ns)
        off = got.cpu().double() - ref
        assert (off.abs() <= bound).all() and (off.norm() / ref.norm()).item() < 2.1 * 2.0 ** -10.5
    for dtype in (torch.float16, torch.bfloat16, torch.float32):
        res = torch.randn(m, n, generator=g).to(dtype)
        out = res.cuda()
        hip.gemm_frag(xp, m, dg, qt, n, k, bias=b1.cuda(), residual=out, out=out, mt=5, ns=3)    # in place, as on the residual stream
        tol = dict(rtol=8e-3, atol=2e-2) if dtype == torch.bfloat16 else dict(rtol=2e-3, atol=8e-3)
        torch.testing.assert_close(out.cpu().double(), xd @ wg.t() + b1.double() + res.double(), **tol)


# N odd, a multiple of 4 and of 16; K with and without a cut last k-tile
@pytest.mark.parametrize("name,m,n,k,kind", [("asym_int4", 258, 261, 9440, 0), ("sym_int4", 276, 212, 10784, 0), ("nf4", 283, 208, 8832, 1),
                                             ("nf4", 283, 208, 8832, 2), ("sym_int8", 283, 229, 10560, 1), ("fp6", 266, 210, 6400, 2)])
def test_split_of_k_in_the_public_call(hip, name, m, n, k, kind):
    """partial sums behind the ordered x, added up by the launch that applies bias, activation and the residual: in place, rows apart"""
    qt = Q.ggml_tensor_qtype[name]
    assert hip.lib().bigdl_gemm_frag_workspace(m, n, k, qt, 0, 2) >= 2 * m * n
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k, 2, torch.bfloat16 if kind == 1 else torch.float16)
    assert kind == 2 or hip.gemm_lowbit_frag(m, n, k, qt, x.stride(0), False, kind)
    g = torch.Generator().manual_seed(3)
    bias, res = torch.randn(n, generator=g).half(), torch.randn(m, n, generator=g).half()
    for dtype, step in ((torch.float32, 0.0), (torch.float16, 2.0 ** -11)):
        buf = torch.full((m, n + 8), 7.0, dtype=dtype, device="cuda")
        out = buf[:, :n]
        out.copy_(res)
        hip.gemm_lowbit(hip.Frags(hip.frag_pack(x), m, k) if kind == 2 else x, dev, qt, n, k, bias=bias.cuda(), act="silu", residual=out, out=out)
        first = xd @ w.t() + bias.double()
        ref = torch.nn.functional.silu(first) + res.double()
        off = (out.double().cpu() - ref).abs()
        # _close's bound through silu, 1.1 steep at most, and the result's rounding; all together as for the pairs below
        assert (off <= 1.1 * (2.0 ** -9 * (xd.abs() @ w.abs().t()) + 1e-5) + step * ref.abs()).all()
        assert (off.norm() / ref.norm()).item() < 1.1 * 2.0 ** -10.5 + step and (buf[:, n:] == 7).all()


@pytest.mark.parametrize("name,m,n,k", [("sym_int4", 77, 2048, 2048), ("sym_int8", 203, 1536, 4096), ("asym_int4", 300, 520, 1056)])
def test_bf16_rows_of_a_linear(hip, monkeypatch, name, m, n, k):
    """rounded to fp16 by the pass that orders them; up to fp16's largest and past it, as the conversion of the other kernels does"""
    from bigdl_amd.transformers.low_bit_linear import FP4Params, lowbit_matmul
    qt = Q.ggml_tensor_qtype[name]
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(1)) * 0.05
    raw = host.quantize(w, qt)
    raw = raw.view(torch.uint8) if raw.dtype != torch.uint8 else raw
    par = FP4Params(raw.flatten(), quantized=True, _shape=(n, k), qtype=qt).to("cuda")
    x, xd = _x(m, k, 2, torch.bfloat16)
    kinds = []
    real = hip._gemm_frag_dense
    monkeypatch.setattr(hip, "_gemm_frag_dense", lambda x, kind, *a, **kw: (kinds.append(kind), real(x, kind, *a, **kw))[1])
    out = lowbit_matmul(x, par, n)
    assert kinds == [1] and out.dtype == torch.bfloat16
    wd = host.dequantize(raw, qt, (n, k)).double()
    ref = xd @ wd.t()
    bound = 2.0 ** -9 * (xd.abs() @ wd.abs().t()) + 2.0 ** -8 * ref.abs() + 1e-5
    assert ((out.double().cpu() - ref).abs() <= bound).all()
    big = torch.zeros(m, k, dtype=torch.bfloat16, device="cuda")
    big[0, 0], big[1, 1], big[2, 2] = 3e38, -3e38, float("nan")
    monkeypatch.setattr(hip, "gemm_lowbit_frag", lambda *a, **kw: False)
    other = lowbit_matmul(big, par, n)
    monkeypatch.undo()
    assert torch.equal(lowbit_matmul(big, par, n).isfinite(), other.isfinite()) and not other[:3].isfinite().any()


@pytest.mark.parametrize("splits", [1, 2, 5])
@pytest.mark.parametrize("b,q_len,hq,hkv,d", [(40, 1, 8, 2, 64), (17, 3, 4, 4, 128), (33, 1, 40, 1, 96)])
def test_decode_attention_in_fragment_order(hip, splits, b, q_len, hq, hkv, d):
    """one key range, and several that the last workgroup combines"""
    g = torch.Generator().manual_seed(5)
    cap, past = 512, 300
    qkv = torch.randn(b * q_len, (hq + 2 * hkv) * d, generator=g).half().cuda()
    k, vt = torch.randn(b, hkv, cap, d, generator=g).half().cuda(), torch.randn(b, hkv, d, cap, generator=g).half().cuda()
    lens = torch.full((b,), past, dtype=torch.int32, device="cuda")
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, q_len, d, splits) + 16, device="cuda")
    cnt = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    rows = torch.empty(b * q_len, hq * d, dtype=torch.float16, device="cuda")
    frags = hip.Frags(torch.zeros(hip.frag_halves(b * q_len, hq * d), dtype=torch.float16, device="cuda"), b * q_len, hq * d)
    for out in (rows, frags):
        hip.attn_decode(qkv, k, vt, lens, out, ws, cnt, n_heads=hq, n_kv_heads=hkv, head_dim=d, q_len=q_len, batch=b, scale=d ** -0.5,
                        splits=splits, append=True)
    assert rows.isfinite().all() and torch.equal(frags.data, hip.frag_pack(rows))


@pytest.mark.parametrize("name", ["sym_int4", "fp6"])
@pytest.mark.parametrize("m", [700, 2048, 2100])
def test_many_rows_of_a_ragged_k(hip, name, m):
    """a K that the prompt kernel does not take: one call of up to FRAG_MAX_ROWS rows, more in pieces"""
    from bigdl_amd.transformers.low_bit_linear import lowbit_rows
    n, k = 328, 1184
    qt = Q.ggml_tensor_qtype[name]
    dev, w = _weight(n, k, qt, 1)
    x, xd = _x(m, k, 2)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(3)).half()
    assert hip.gemm_lowbit_frag(min(m, hip.FRAG_MAX_ROWS), n, k, qt, x.stride(0))
    _close(lowbit_rows(x, dev, qt, n, k, bias=bias.cuda(), out_dtype=torch.float32), xd, w, xd @ w.t() + bias.double())


@pytest.mark.parametrize("rows,width", [(33, 128), (77, 2048), (130, 4096 + 128), (64, 9216)])
def test_norm_in_fragment_order(hip, rows, width):
    g = torch.Generator().manual_seed(7)
    x, res = torch.randn(rows, width, generator=g).half().cuda(), torch.randn(rows, width, generator=g).half().cuda()
    w = (1 + 0.1 * torch.randn(width, generator=g)).half().cuda()
    h0, h1 = torch.empty_like(x), torch.empty_like(x)
    want = hip.frag_pack(hip.rms_norm(x, w, 1e-5, residual=res, res_out=h0))
    got = hip.rms_norm(x, w, 1e-5, residual=res, res_out=h1, frags=True)
    assert got.shape == (rows, width) and torch.equal(h0, h1)
    tiles = (rows + 15) // 16
    live = (torch.arange(tiles * 16, device="cuda") < rows).view(tiles, 1, 16, 1)        # rows past the last one are not written
    view = (width // 32, tiles, 4, 16, 8)
    assert torch.equal(torch.where(live, got.data.view(view), 0), torch.where(live, want.view(view), 0))


@pytest.mark.parametrize("name", ["sym_int4", "q4_k"])
@pytest.mark.parametrize("m", [64, 77, 203, 400])
def test_norm_pair_down_without_rows_in_between(hip, name, m):
    """norm -> gate / up -> down with x in fragment order all along, against the same products on rows"""
    n, k = 1536, 1024
    qt = Q.ggml_tensor_qtype[name]
    (dg, _), (du, _), (dd, _) = _weight(n, k, qt, 3), _weight(n, k, qt, 4), _weight(k, n, qt, 5)
    x = _x(m, k, 6)[0].contiguous()
    w = torch.ones(k, dtype=torch.float16, device="cuda")
    y = hip.rms_norm(x, w, 1e-5)
    ref = hip.gemm_lowbit(hip.gemm_lowbit_ex(y, dg, qt, n, k, w2=du, act="silu"), dd, qt, k, n, out_dtype=torch.float32)
    f = hip.rms_norm(x, w, 1e-5, frags=True)
    f = hip.gemm_lowbit_ex(f, dg, qt, n, k, w2=du, act="silu", out_frags=True)
    got = hip.gemm_lowbit(f, dd, qt, k, n, out_dtype=torch.float32)
    # the same fp16 operands; sums in another order move the pair's results by a rounding to fp16 (2^-11) here and there
    assert ((got - ref).norm() / ref.norm()).item() < 2.0 ** -11


@pytest.mark.parametrize("b,sq,hq,d", [(1, 77, 4, 128), (3, 20, 6, 64), (1, 130, 4, 96)])
def test_prompt_attention_in_fragment_order(hip, b, sq, hq, d):
    q, k, v = (torch.randn(b, hq, sq, d, device="cuda").half() for _ in range(3))
    want = hip.frag_pack(hip.attn_prefill(q, k, v, scale=d ** -0.5).view(b * sq, hq * d))
    got = hip.attn_prefill(q, k, v, scale=d ** -0.5, frags=True)
    tiles = (b * sq + 15) // 16
    live = (torch.arange(tiles * 16, device="cuda") < b * sq).view(tiles, 1, 16, 1)
    view = (hq * d // 32, tiles, 4, 16, 8)
    assert torch.equal(torch.where(live, got.data.view(view), 0), torch.where(live, want.view(view), 0))


@pytest.mark.parametrize("batch,past,fp8", [(33, 40, False), (50, 300, True), (1, 90, False)])
def test_engine_with_and_without_fragment_order(hip, monkeypatch, batch, past, fp8):
    """prompt pass and decode steps: every product that takes x in fragment order against the same engine on rows"""
    from bigdl_amd.models import decoder as D
    cfg = D.DecoderConfig(vocab_size=2048, hidden_size=1024, intermediate_size=2048, num_layers=2, num_heads=8, num_kv_heads=4,
                          head_dim=128, max_position=512)
    ids = torch.randint(0, 2048, (batch, past + 2), generator=torch.Generator().manual_seed(3)).cuda()
    taken = []

    def run(frags):
        if not frags:
            monkeypatch.setattr(hip, "gemm_lowbit_frag", lambda *a, **k: False)
        else:
            real = hip._gemm_frag_dense
            monkeypatch.setattr(hip, "_gemm_frag_dense", lambda x, kind, *a, **k: (taken.append(kind), real(x, kind, *a, **k))[1])
        eng = D.build_random_decoder(cfg, Q.SYM_INT4, device="cuda", seed=0)
        eng.ensure_cache(batch, past + 16, fp8=fp8)
        out = [eng.prefill(ids[:, :past]).view(batch, -1)]
        for j in range(2):
            out.append(eng.decode(ids[:, past + j:past + j + 1].contiguous(), 1)[0].clone())
        monkeypatch.undo()
        return out

    with_frags, on_rows = run(True), run(False)
    assert 2 in taken
    for a, b in zip(with_frags, on_rows):
        # the same fp16 operands and fp32 sums in another order: single roundings to fp16 (2^-11) differ and pass through two layers
        assert ((a - b).norm() / b.norm()).item() < 4e-3


def test_only_known_entries_take_fragment_order(hip):
    m, k, n = 48, 256, 128
    w = _weight(n, k, Q.SYM_INT4, 1)[0]
    x = hip.rms_norm(torch.randn(m, k).half().cuda(), torch.ones(k, dtype=torch.float16, device="cuda"), 1e-5, frags=True)
    rows = torch.zeros(m, k, dtype=torch.float16, device="cuda")
    for call in (lambda: hip.gemv_lowbit(x, w, Q.SYM_INT4, n, k), lambda: hip.gemm_prompt(x, w, Q.SYM_INT4, n, k),
                 lambda: hip.gemm_rows(x, w, Q.SYM_INT4, n, k), lambda: hip.frag_pack(x), lambda: hip.bf16_to_f16(x),
                 lambda: hip.gemm_lowbit(rows, w, Q.SYM_INT4, n, k, out=hip.Frags(rows.new_empty(hip.frag_halves(m, n)), m, n))):
        with pytest.raises(ValueError):
            call()


@pytest.mark.parametrize("gemv_max", [16, 64])
def test_engine_with_products_on_gemv(hip, monkeypatch, gemv_max):
    """40 rows: the products run on gemv_lowbit where BIGDL_GEMV_MAX_ROWS says so, and get rows from whatever is in front of them"""
    from bigdl_amd.models import decoder as D
    cfg = D.DecoderConfig(vocab_size=1024, hidden_size=1024, intermediate_size=2048, num_layers=2, num_heads=16, num_kv_heads=4,
                          head_dim=128, max_position=512, norm="layer", gated_mlp=False, act="gelu")     # (a pair is 32 rows at most there)
    assert hip.gemm_lowbit_frag(40, 1024, 2048, Q.SYM_INT4, None, False, 3)
    ids = torch.randint(0, 1024, (40, 9), generator=torch.Generator().manual_seed(3)).cuda()

    def run():
        eng = D.build_random_decoder(cfg, Q.SYM_INT4, device="cuda", seed=0)
        eng.ensure_cache(40, 64, fp8=False)
        return eng.prefill(ids[:, :8]).view(40, -1), eng.decode(ids[:, 8:].contiguous(), 1)[0].clone()

    monkeypatch.setattr(D, "GEMV_MAX_ROWS", gemv_max)
    got = run()
    monkeypatch.setattr(hip, "gemm_lowbit_frag", lambda *a, **k: False)
    for a, b in zip(got, run()):
        # the same fp16 operands and fp32 sums in another order, as above
        assert ((a - b).norm() / b.norm()).item() < 4e-3


@pytest.mark.parametrize("name,n,k", [("sym_int4", 2048, 2048), ("nf4", 1536, 4096)])
def test_rows_of_stride_zero(hip, name, n, k):
    """one row seen 203 times: accepted by the other kernels, so by the pass that orders x too"""
    qt = Q.ggml_tensor_qtype[name]
    dev, w = _weight(n, k, qt, 1)
    row = torch.randn(1, k, generator=torch.Generator().manual_seed(2)).half()
    x = row.cuda().expand(203, k)
    assert torch.equal(hip.frag_pack(x), hip.frag_pack(x.contiguous())) and hip.gemm_lowbit_frag(203, n, k, qt, 0)
    out = hip.gemm_lowbit(x, dev, qt, n, k, out_dtype=torch.float32)
    xd = row.double().expand(203, k)
    _close(out, xd, w, xd @ w.t())
    assert torch.equal(out, out[:1].expand(203, n))
