"""Products whose K is split and whose sums the RMSNorm behind adds up (csrc/hip/gemm_lowbit.hip ``bigdl_gemm_parts``, misc_ops.hip
``rms_norm_parts_kernel``)."""
import random

import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import hip, host

needs_library = pytest.mark.skipif(not hip._LIB_PATH.exists(), reason="the kernel library is not built")


def _weight(n, k, qt, seed):
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * 0.05
    raw = host.quantize(w, qt).view(torch.uint8)
    return host.relayout_to_device(raw, qt, n, k).cuda(), host.dequantize(raw, qt, w.shape).double()


@needs_library
@pytest.mark.parametrize("qt", [Q.SYM_INT4, Q.ASYM_INT4, Q.NF4, Q.SYM_INT8])
def test_rule(qt):
    """no split where nothing takes it; at least eight k-tiles a split"""
    L = hip.lib()
    for m in (1, 16, 32):
        assert L.bigdl_gemm_parts(m, 4096, 14336, 14336, qt, 2) == 0
    assert L.bigdl_gemm_parts(64, 4097, 14336, 14336, qt, 2) == 0         # rows of the slabs a norm cannot read in whole pieces
    assert L.bigdl_gemm_parts(64, 4096, 14340, 14340, qt, 2) == 0
    assert L.bigdl_gemm_parts(64, 4096, 14336, 14336, qt, 0) == 0         # rows, few of them: not this product's
    assert L.bigdl_gemm_parts(1024, 4096, 11000, 11000, qt, 0) == 0       # K the prompt kernel does not take
    for m in (33, 64, 77, 300, 512):
        for n, k in ((2048, 256), (4096, 4096), (2048, 5632), (4096, 14336)):
            s = L.bigdl_gemm_parts(m, n, k, k, qt, 2)
            assert s in (0, 2, 4) and (k + 127) // 128 >= 8 * s, (m, n, k, s)
    assert L.bigdl_gemm_parts(64, 4096, 14336, 14336, qt, 2) > 1          # 128 column tiles of a long K: half the chip without


@needs_library
@pytest.mark.parametrize("m,n,k,name,whole,split", [
    (80, 5120, 2048, "asym_int5", 14.5, 17.5), (54, 4096, 2048, "fp8_e5m2", 10.1, 12.1), (74, 8192, 5632, "sym_int4", 21.9, 25.6),
    (439, 2048, 4096, "asym_int4", 19.0, 21.4), (52, 3072, 4096, "sym_int4", 11.4, 12.8), (193, 5120, 8192, "sym_int8", 36.2, 40.4),
    (118, 5120, 5632, "nf4", 22.8, 25.3), (64, 4096, 11008, "sym_int4", 23.1, 19.7), (77, 4096, 14336, "asym_int4", 29.6, 24.7),
    (36, 4096, 14336, "asym_int4", 23.0, 20.1)])
def test_rule_takes_the_faster_form(m, n, k, name, whole, split):
    """products of rows in fragment order with their norm, us on an MI355X: whole, and with their sums left to it"""
    s = hip.lib().bigdl_gemm_parts(m, n, k, k, Q.ggml_tensor_qtype[name], 2)
    assert (s > 1) == (split < whole) and s != 1


@needs_library
def test_rule_of_rows():
    """a product of rows leaves the sums of the splits that it has without a norm too: six k-tiles a split at least, none where it is whole"""
    L, seen, rng = hip.lib(), set(), random.Random(1)
    sizes = [(300, 4096, 11008), (844, 5120, 4096), (3000, 2048, 5632)]
    sizes += [(rng.randint(257, 8000), 128 * rng.randint(4, 64), 128 * rng.randint(2, 112)) for _ in range(400)]
    for m, n, k in sizes:
        splits, s = hip.gemm_prompt_plan(m, n, k)[1], L.bigdl_gemm_parts(m, n, k, k, Q.SYM_INT4, 0)
        assert s == (splits if splits > 1 else 0) and (s == 0 or k // 128 >= 6 * s), (m, n, k, s)
        seen.add(s)
    assert seen >= {0, 2, 3, 4, 5, 6, 7, 8}


@needs_library
@pytest.mark.parametrize("m,n,k,kind", [(64, 4096, 14336, 2), (1024, 4096, 11008, 0)])
def test_only_the_planned_scratch(m, n, k, kind):
    """a scratch of fewer or more slabs than the plan writes is refused, by the first of the checks (the addresses are odd ones, which the
    next refuses: no launch comes of this)"""
    L = hip.lib()
    s = L.bigdl_gemm_parts(m, n, k, k, Q.SYM_INT4, kind)
    assert s > 1
    for floats in (0, (s - 1) * m * n, s * m * n - 1, s * m * n + 1, (s + 1) * m * n):
        assert L.bigdl_gemm_parts_run(4104, 4104, 4104, floats, m, n, k, k, Q.SYM_INT4, kind, None) == -5
    assert L.bigdl_gemm_parts_run(4104, 4104, 4104, s * m * n, m, n, k, k, Q.SYM_INT4, kind, None) == -1


@pytest.mark.gpu
def test_another_plan_between_two_calls():
    m, n, k = 700, 1024, 14336
    dev, w = _weight(n, k, Q.SYM_INT4, 8)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(9)).half()
    ref, mag = x.double() @ w.t(), x.double().abs() @ w.abs().t()
    xg = x.cuda()
    try:
        for splits in (0, 2, 3, 1, 0):
            hip.gemm_prompt_force(-1, splits)
            torch.full((16 << 20,), float("nan"), device="cuda")               # (what the next allocation holds)
            p = hip.gemm_parts(xg, dev, Q.SYM_INT4, n, k)
            if splits == 1:
                assert p is None
                continue
            assert p.data.shape[0] == (splits or hip.lib().bigdl_gemm_parts(m, n, k, k, Q.SYM_INT4, 0))
            assert ((p.data.double().sum(0).cpu() - ref).abs() <= 2.0 ** -9 * mag + 1e-5).all(), splits
    finally:
        hip.gemm_prompt_force()


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("rows,h", [(1, 8), (5, 128), (33, 2304), (70, 4096), (3, 16384)])
def test_norm_of_parts(parts, rows, h):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(parts, rows, h, generator=g)
    bias, res, w = (torch.randn(*s, generator=g).half() for s in ((h,), (rows, h), (h,)))
    for use_bias, use_res, offset in ((False, False, 0.0), (True, True, 1.0), (False, True, 0.0)):
        p = hip.Parts(x.cuda(), bias.cuda() if use_bias else None)
        r, out = res.cuda(), torch.empty(rows, h, dtype=torch.float16, device="cuda")
        kept = r.clone()
        got = hip.rms_norm(p, w.cuda(), 1e-5, residual=r if use_res else None, res_out=out, offset=offset)
        s = x.double().sum(0) + (bias.double() if use_bias else 0) + (res.double() if use_res else 0)
        ref = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5) * (w.double() + offset)
        # fp32 sums and one rounding to fp16
        assert ((out.double().cpu() - s).abs() <= 2.0 ** -11 * s.abs() + 1e-5).all()
        assert ((got.double().cpu() - ref).abs() <= 2.0 ** -10 * ref.abs() + 2e-5).all()
        assert torch.equal(r, kept)
        if h % 128 == 0:
            f = hip.rms_norm(p, w.cuda(), 1e-5, residual=r if use_res else None, offset=offset, frags=True)
            assert torch.equal(f.data.view(h // 32, -1, 4, 16, 8).permute(1, 3, 0, 2, 4).reshape(-1, h)[:rows], got)
        if use_res:                        # the residual stream in place
            assert torch.equal(hip.rms_norm(p, w.cuda(), 1e-5, residual=r, res_out=r, offset=offset), got) and torch.equal(r, out)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["sym_int4", "asym_int5", "nf4", "sym_int8"])
@pytest.mark.parametrize("m,n,k", [(33, 2048, 5632), (64, 4096, 4096), (77, 2056, 7168), (300, 1024, 14336), (700, 1024, 14336)])
def test_parts_are_the_product(name, m, n, k):
    qt = Q.ggml_tensor_qtype[name]
    dev, w = _weight(n, k, qt, 2)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(3)).half()
    bias = torch.randn(n, generator=torch.Generator().manual_seed(4)).half()
    xg = x.cuda() if m > 512 else hip.Frags(hip.frag_pack(x.cuda()), m, k)
    p = hip.gemm_parts(xg, dev, qt, n, k, bias=bias.cuda())
    if (m, n, k) == (64, 4096, 4096) and name != "asym_int5":
        assert p is None                     # better whole
        return
    ref = x.double() @ w.t()
    # weights rounded to fp16: 2^-11 of a weight's larger term, for a table's value too, times two
    assert ((p.data.double().sum(0).cpu() - ref).abs() <= 2.0 ** -9 * (x.double().abs() @ w.abs().t()) + 1e-5).all()
    assert ((p.sum().double().cpu() - ref - bias.double()).abs() <= 2.0 ** -9 * (x.double().abs() @ w.abs().t()) + 2.0 ** -10 * ref.abs() + 1e-2).all()
    with pytest.raises(ValueError):
        hip.gemm_lowbit(p, dev, qt, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens,bias", [(1, 70, False), (36, 3, False), (2, 300, True)])
def test_engine_with_and_without(monkeypatch, batch, tokens, bias):
    """prompts and steps of an engine whose norms add split sums, and of one whose products add them themselves"""
    from bigdl_amd.models.decoder import DecoderConfig, NativeDecoder, build_random_decoder
    cfg = DecoderConfig(vocab_size=512, hidden_size=1024, intermediate_size=6144, num_layers=3, num_heads=8, num_kv_heads=4, head_dim=128,
                        max_position=1024)
    ids = torch.randint(0, 512, (batch, tokens), generator=torch.Generator().manual_seed(5)).cuda()
    step = torch.randint(0, 512, (batch, 1), generator=torch.Generator().manual_seed(6)).cuda()
    made, outs = [], []
    real = hip.gemm_parts

    def counted(*a, **kw):
        p = real(*a, **kw)
        made.append(p is not None)
        return p

    monkeypatch.setattr(hip, "gemm_parts", counted)
    for adds in (True, False):
        eng = build_random_decoder(cfg, Q.SYM_INT4, device="cuda", seed=0)
        if bias:
            g = torch.Generator().manual_seed(7)
            for lw in eng.layers:
                lw.o.bias, lw.down.bias = (torch.randn(1024, generator=g).half().cuda() * 0.1 for _ in range(2))
        if not adds:
            monkeypatch.setattr(NativeDecoder, "_norm_adds", lambda self: False)
            made.append(None)
        eng.ensure_cache(batch, tokens + 16, fp8=False)
        outs.append([eng.prefill(ids).float(), *(eng.decode(step, 1)[0].float().clone() for _ in range(3))])
    assert any(made[:made.index(None)]) and not any(made[made.index(None):])
    for a, b in zip(*outs):
        assert (a - b).norm() <= 4e-3 * b.norm()            # an fp16 rounding of the products less: 2^-11 of them, three layers


@pytest.mark.gpu
@pytest.mark.parametrize("batch,tokens", [(1, 70), (36, 3), (1, 600)])
@pytest.mark.parametrize("kind", ["ungated", "output norms", "experts", "dense head", "gate and up of two formats"])
def test_engines_of_other_designs(monkeypatch, kind, batch, tokens):
    """the same of engines where only some products stand in front of a norm that adds: o and down of the layers around are split"""
    from dataclasses import replace

    from bigdl_amd.models.decoder import DecoderConfig, NativeDecoder, build_random_decoder
    cfg = DecoderConfig(vocab_size=512, hidden_size=1024, intermediate_size=6144, num_layers=3, num_heads=32, num_kv_heads=4, head_dim=128,
                        max_position=1024, gated_mlp=kind != "ungated")
    eng = build_random_decoder(cfg, Q.SYM_INT4, device="cuda", seed=0, lm_head_qtype=Q.FP16 if kind == "dense head" else None)
    layers = list(eng.layers)
    if kind == "output norms":
        ones = [(1 + 0.1 * torch.randn(1024, generator=torch.Generator().manual_seed(i))).half().cuda() for i in range(3)]
        layers[0].post_ffn_out_norm, layers[1].post_attn_out_norm, layers[2].pre_ffn_norm = ones
    elif kind == "experts":
        # (both experts for every token: a choice between them could fall either way)
        cfg = replace(cfg, num_experts=2, top_k=2, moe_intermediate_size=512)
        layers[1] = build_random_decoder(cfg, Q.SYM_INT4, device="cuda", seed=1).layers[1]
    elif kind == "gate and up of two formats":
        layers[1].up = build_random_decoder(cfg, Q.NF4, device="cuda", seed=1).layers[1].up
    ids = torch.randint(0, 512, (batch, tokens), generator=torch.Generator().manual_seed(5)).cuda()
    step = torch.randint(0, 512, (batch, 1), generator=torch.Generator().manual_seed(6)).cuda()
    real, made, outs = hip.gemm_parts, [], []

    def counted(x, w, qtype, n, k, **kw):
        p = real(x, w, qtype, n, k, **kw)
        made.append((k, p is not None))
        return p

    monkeypatch.setattr(hip, "gemm_parts", counted)
    for adds in (True, False):
        if not adds:
            monkeypatch.setattr(NativeDecoder, "_norm_adds", lambda self: False)
            # o, and down where its x comes in fragment order or is a long prompt's
            assert (4096, True) in made and ((6144, True) in made) == (kind != "ungated" or tokens > 512)
            made.clear()
        e = NativeDecoder(cfg, eng.embed, layers, eng.final_norm, eng.lm_head, device="cuda")
        e.ensure_cache(batch, tokens + 16, fp8=False)
        outs.append([e.prefill(ids).float(), *(e.decode(step, 1)[0].float().clone() for _ in range(3))])
    assert not any(split for _, split in made)
    for a, b in zip(*outs):
        assert (a - b).norm() <= 4e-3 * b.norm()            # (as above)
