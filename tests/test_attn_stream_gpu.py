"""Decode attention with K / V^T through LDS in whole lines (csrc/hip/attn_decode_stream.h) against float64: lengths
around its blocks (64 keys a wavefront in e5m2 caches, 32 in fp16; two or four wavefronts), several lengths in a batch, ranges without
keys, groups of 1 to 32 query heads, and what changes a score.  The cache behind the last piece that holds a key is NaN: nothing of it
may reach a result."""
import math

import pytest
import torch

from bigdl_amd.ops import hip

pytestmark = pytest.mark.gpu

LMAX = 1024


def _f64(q, k, v, scale, softcap=0.0, window=0, slopes=None, mask=None):
    """q [Hq, D], k / v [Hkv, n, D] (the newest key last), all float64"""
    hq, n = q.shape[0], k.shape[1]
    g = hq // k.shape[0]
    s = torch.einsum("hd,hnd->hn", q, k.repeat_interleave(g, 0)) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    pos = torch.arange(n)
    if slopes is not None:
        s = s + slopes.double()[:, None] * (pos - (n - 1))
    if mask is not None:
        s = s + mask.double()[:n]
    if window:
        s = s.masked_fill(pos <= n - 1 - window, -math.inf)
    return torch.einsum("hn,hnd->hd", torch.softmax(s, -1), v.repeat_interleave(g, 0))


def _rotate(x, pos, table, interleaved):
    """x [H, D] float64; table [max_pos, rot / 2, 2]"""
    rot = 2 * table.shape[1]
    c, s = table[pos, :, 0].double(), table[pos, :, 1].double()
    y = x.clone()
    if interleaved:
        a, b = x[:, 0:rot:2], x[:, 1:rot:2]
        y[:, 0:rot:2], y[:, 1:rot:2] = a * c - b * s, b * c + a * s
    else:
        h = rot // 2
        a, b = x[:, :h], x[:, h:rot]
        y[:, :h], y[:, h:rot] = a * c - b * s, b * c + a * s
    return y


def _case(d, fp8, hq, hkv, pasts, splits, defer=False, interleaved=False, rot=None, rope=True, **opt):
    torch.manual_seed(hash((d, fp8, hq, hkv, len(pasts), splits)) % 1000)
    b = len(pasts)
    piece = 64 if fp8 else 32
    k = torch.randn(b, hkv, LMAX, d).half()
    v = torch.randn(b, hkv, d, LMAX).half()
    if fp8:
        k, v = k.to(torch.float8_e5m2), v.to(torch.float8_e5m2)
    kf, vf = k.double(), v.double()
    raw = torch.uint8 if fp8 else torch.int16
    kd, vd = k.view(raw).clone(), v.view(raw).clone()
    for i, p in enumerate(pasts):
        end = (p + 1 + piece - 1) // piece * piece
        kd[i, :, end:] = 0x7F if fp8 else 0x7FFF
        vd[i, :, :, end:] = 0x7F if fp8 else 0x7FFF
        kd[i, :, p] = 0x7F if fp8 else 0x7FFF          # the new token's place: written by the call
        vd[i, :, :, p] = 0x7F if fp8 else 0x7FFF
    dt = torch.uint8 if fp8 else torch.float16
    kd, vd = kd.view(dt).cuda(), vd.view(dt).cuda()
    before_k, before_v = kd.clone(), vd.clone()
    qkv = torch.randn(b, (hq + 2 * hkv) * d).half()
    half = (rot or d) // 2
    ang = torch.arange(LMAX).float()[:, None] / (10000 ** (torch.arange(half).float() / half))
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    out = torch.full((b, hq * d), float("nan"), dtype=torch.float16, device="cuda")
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, 1, d, splits), dtype=torch.float32, device="cuda")
    counters = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    scale = 1.0 / math.sqrt(d)
    slopes = torch.rand(hq) * 0.05 if opt.pop("alibi", False) else None
    mask = (torch.randn(b, 1, LMAX) * 2).half() if opt.pop("mask", False) else None
    hip.attn_decode(qkv.cuda(), kd, vd, torch.tensor(pasts, dtype=torch.int32, device="cuda"), out, ws, counters, n_heads=hq, n_kv_heads=hkv,
                    head_dim=d, q_len=1, batch=b, scale=scale, splits=splits, rope_table=table.cuda() if rope else None, append=not rope,
                    interleaved=interleaved, defer_combine=defer, alibi=None if slopes is None else slopes.cuda(),
                    mask=None if mask is None else mask.cuda(), **opt)
    torch.cuda.synchronize()
    if defer and splits > 1:
        # [b * hkv][splits][16][d + 4]: O row, maximum (log2), sum
        w = ws[: b * hkv * splits * 16 * (d + 4)].view(b, hkv, splits, 16, d + 4)[:, :, :, : hq // hkv].cpu().double()
        f = torch.exp2(w[..., d] - w[..., d].amax(2, keepdim=True))
        got = ((w[..., :d] * f[..., None]).sum(2) / (w[..., d + 1] * f).sum(2)[..., None]).reshape(b, hq, d)
    else:
        got = out.cpu().double().view(b, hq, d)
    x = qkv.double().view(b, hq + 2 * hkv, d)
    worst = 0.0
    kc, vc = kd.cpu(), vd.cpu()
    for i, p in enumerate(pasts):
        q, kn, vn = x[i, :hq], x[i, hq:hq + hkv], x[i, hq + hkv:]
        if rope:
            q, kn = _rotate(q, p, table, interleaved), _rotate(kn, p, table, interleaved)
        # what the call wrote: the value exactly, the key to a rounding of its rotation
        wk, wv = kc[i, :, p], vc[i, :, :, p]
        if fp8:
            wk, wv = wk.view(torch.float8_e5m2).double(), wv.view(torch.float8_e5m2).double()
            assert torch.equal(wv, vn.half().to(torch.float8_e5m2).double())
            assert ((wk - kn).abs() <= 0.13 * kn.abs() + 1e-4).all()
        else:
            assert torch.equal(wv.double(), vn)
            assert ((wk.double() - kn).abs() <= 1e-3 * kn.abs() + 1e-4).all()
        kk = torch.cat([kf[i, :, :p], wk.double()[:, None]], 1)
        vv = torch.cat([vf[i, :, :, :p].transpose(1, 2), vn.half().to(torch.float8_e5m2).double()[:, None] if fp8 else vn[:, None]], 1)
        ref = _f64(q, kk, vv, scale, slopes=slopes, mask=None if mask is None else mask[i, 0], **opt)
        worst = max(worst, ((got[i] - ref).norm() / ref.norm()).item())
    # nothing else of the caches has changed
    before_k, before_v = before_k.cpu(), before_v.cpu()
    for i, p in enumerate(pasts):
        before_k[i, :, p], before_v[i, :, :, p] = kc[i, :, p], vc[i, :, :, p]
    assert torch.equal(before_k.view(raw), kc.view(raw)) and torch.equal(before_v.view(raw), vc.view(raw))
    assert int(counters.abs().sum()) == 0
    # fp16 operands: q, the weights and the result round to 2^-11 each; an error e of a score (|score| < 8 in these cases, mask included)
    # changes its weight by a factor 1 + e: 8 x 2^-11 + 2 x 2^-11 < 5e-3.  Two e4m3 terms hold q and the weights to 2^-8 each, of q
    # averaged over the channels of a score (a quarter of it): 8 / 4 x 2^-8 + 2^-8 < 1.2e-2
    assert worst < (1.2e-2 if fp8 and d == 128 else 5e-3), worst


EDGES = [0, 1, 30, 31, 32, 33, 63, 64, 65, 126, 127, 128, 129, 191, 255, 256, 257, 300, 511, 512, 700, 1022, 1023]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv,splits", [(2, 2, 2), (8, 2, 3), (7, 1, 1), (16, 1, 2), (40, 40, 1), (32, 16, 2), (32, 1, 2), (50, 2, 1)])
def test_lengths(d, fp8, hq, hkv, splits):
    _case(d, fp8, hq, hkv, EDGES, splits)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("hq,hkv", [(8, 2), (24, 1)])
@pytest.mark.parametrize("splits", [4, 5, 16, 17, 33])
def test_merges_any_number_of_ranges(d, fp8, hq, hkv, splits):
    _case(d, fp8, hq, hkv, [0, 31, 256, 700, 1023], splits)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("opt", [dict(softcap=20.0), dict(window=100), dict(alibi=True), dict(mask=True), dict(interleaved=True),
                                 dict(interleaved=True, rot=32), dict(rope=False), dict(defer=True)], ids=lambda o: next(iter(o)) + str(len(o)))
def test_options(d, fp8, opt):
    _case(d, fp8, 6, 2, [5, 127, 128, 400, 1000], 3, **opt)
    _case(d, fp8, 96, 96, [0, 63, 64, 200, 256, 777, 1023], 1, **{**opt, "defer": False})


SEVERAL = [(4, 4, 9), (8, 2, 4), (1, 1, 3), (2, 2, 16), (8, 2, 7), (16, 1, 2), (60, 60, 5), (240, 60, 6), (24, 1, 3)]


# (two row tiles of e5m2 with heads of 128 take the form that widens them: more exact than one token's)
@pytest.mark.parametrize("d,fp8,hq,hkv,n", [(d, fp8, *c) for d in (64, 128) for fp8 in (False, True) for c in SEVERAL
                                            if not (fp8 and d == 128 and c[0] // c[1] * c[2] > 16)])
@pytest.mark.parametrize("interleaved", [False, True])
def test_several_tokens_round_as_one_after_the_other(d, fp8, hq, hkv, n, interleaved):
    """a draft's check in one call and the decode steps it stands for: the same bits, in the output and in both caches"""
    torch.manual_seed(n)
    pasts = [0, 29, 60, 63, 120, 250, 255, 500, 1000]
    b = len(pasts)
    dt = torch.float8_e5m2 if fp8 else torch.float16
    raw = torch.uint8 if fp8 else torch.int16
    k, v = torch.randn(b, hkv, LMAX, d).half().to(dt).cuda(), torch.randn(b, hkv, d, LMAX).half().to(dt).cuda()
    qkv = torch.randn(b, n, (hq + 2 * hkv) * d, device="cuda").half()
    ang = torch.arange(LMAX, device="cuda").float()[:, None] / (10000 ** (torch.arange(d // 2, device="cuda").float() / (d // 2)))
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    counters = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, n, d, 1), dtype=torch.float32, device="cuda")

    def call(x, kc, vc, first, m):
        out = torch.empty(b * m, hq * d, dtype=torch.float16, device="cuda")
        past = torch.tensor(pasts, dtype=torch.int32, device="cuda") + first
        c = (lambda t: t.view(torch.uint8)) if fp8 else (lambda t: t)
        hip.attn_decode(x.reshape(b * m, -1), c(kc), c(vc), past, out, ws, counters, n_heads=hq, n_kv_heads=hkv, head_dim=d, q_len=m,
                        batch=b, scale=d ** -0.5, splits=1, rope_table=table, interleaved=interleaved)
        return out.view(b, m, hq * d)

    k1, v1 = k.clone(), v.clone()
    many = call(qkv, k1, v1, 0, n)
    steps = torch.cat([call(qkv[:, t:t + 1].contiguous(), k, v, t, 1) for t in range(n)], 1)
    assert torch.equal(k1.view(raw), k.view(raw)) and torch.equal(v1.view(raw), v.view(raw))
    assert torch.equal(many, steps)


@pytest.mark.parametrize("d,fp8", [(64, False), (64, True), (128, False), (128, True)])
@pytest.mark.parametrize("hq,hkv,b,n", [(8, 2, 3, 3), (12, 4, 130, 5)])
@pytest.mark.parametrize("opt", ["window", "softcap", "alibi", "mask", "append"])
@pytest.mark.parametrize("splits", [1, 3])
def test_several_tokens_with_what_changes_a_score(d, fp8, hq, hkv, b, n, opt, splits):
    """the same bits as one after the other with one range; with several, whose bounds depend on the length, the same result"""
    torch.manual_seed(b + n)
    pasts = [(37 * i) % 900 for i in range(b)]
    k, v = torch.randn(b, hkv, LMAX, d, device="cuda").half(), torch.randn(b, hkv, d, LMAX, device="cuda").half()
    if fp8:
        k, v = (t.to(torch.float8_e5m2).view(torch.uint8) for t in (k, v))
    qkv = torch.randn(b, n, (hq + 2 * hkv) * d, device="cuda").half()
    ang = torch.rand(LMAX, d // 2, device="cuda")
    table = None if opt == "append" else torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    mask = (2 * torch.randn(b, n, LMAX, device="cuda")).half()
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, n, d, splits), dtype=torch.float32, device="cuda")
    counters = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    extra = {"window": dict(window=100), "softcap": dict(softcap=20.0), "alibi": dict(alibi=torch.rand(hq, device="cuda") * 0.05)}.get(opt, {})

    def call(kc, vc, first, m):
        out = torch.empty(b * m, hq * d, dtype=torch.float16, device="cuda")
        more = dict(extra, mask=mask[:, first:first + m].contiguous()) if opt == "mask" else extra
        hip.attn_decode(qkv[:, first:first + m].reshape(b * m, -1), kc, vc, torch.tensor(pasts, dtype=torch.int32, device="cuda") + first, out, ws,
                        counters, n_heads=hq, n_kv_heads=hkv, head_dim=d, q_len=m, batch=b, scale=d ** -0.5, splits=splits, rope_table=table,
                        append=table is None, **more)
        return out.view(b, m, hq * d)

    k1, v1 = k.clone(), v.clone()
    many, steps = call(k1, v1, 0, n), torch.cat([call(k, v, t, 1) for t in range(n)], 1)
    assert torch.equal(k1, k) and torch.equal(v1, v)
    if splits == 1:
        assert torch.equal(many, steps)
    # (each within the bound of _case of the exact result)
    assert ((many.double() - steps.double()).norm() / steps.double().norm()).item() < 2 * (1.2e-2 if fp8 and d == 128 else 5e-3)


# (heads of 64 in an e5m2 cache of one range come here from 512 pairs on)
@pytest.mark.parametrize("d,fp8,hq,hkv,b,splits", [
    (d, fp8, *c, splits) for d in (64, 128) for fp8 in (False, True) for c in [(8, 2, 2), (40, 40, 2), (40, 40, 16), (40, 2, 3)]
    for splits in (1, 2) if not (fp8 and d == 64 and splits == 1 and c[1] * c[2] < 512)])
def test_weights_far_below_the_largest_keep_their_bits(d, fp8, hq, hkv, b, splits):
    """The first key takes nearly all of the weight, and the values of the first 64 keys are zero: the result is the sum over all the
    others, whose weights are e^-16 of the largest"""
    torch.manual_seed(d + hq)
    n, gap = 1000, 16.0
    dt, raw = (torch.float8_e5m2, torch.uint8) if fp8 else (torch.float16, torch.float16)
    k, v = torch.randn(b, hkv, LMAX, d).half(), (1024 * torch.randn(b, hkv, d, LMAX)).half()
    u = torch.nn.functional.normalize(torch.randn(b, hkv, d), dim=-1)
    # (every query's score of key 0 is close to gap, those of the others are normal)
    q = u.repeat_interleave(hq // hkv, 1) * d ** 0.5 + 0.3 * torch.randn(b, hq, d)
    k[:, :, 0] = (gap * u).half()
    v[..., :64] = 0
    k, v = k.to(dt), v.to(dt)
    qkv = torch.cat([q, torch.randn(b, 2 * hkv, d)], 1).reshape(b, -1).half()
    kd, vd = k.view(raw).cuda(), v.view(raw).cuda()
    out = torch.empty(b, hq * d, dtype=torch.float16, device="cuda")
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, 1, d, splits), dtype=torch.float32, device="cuda")
    counters = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    hip.attn_decode(qkv.cuda(), kd, vd, torch.full((b,), n - 1, dtype=torch.int32, device="cuda"), out, ws, counters, n_heads=hq,
                    n_kv_heads=hkv, head_dim=d, q_len=1, batch=b, scale=d ** -0.5, splits=splits, append=True)
    kk, vv = kd.cpu().view(dt)[:, :, :n].double(), vd.cpu().view(dt)[..., :n].double().transpose(2, 3)
    worst = 0.0
    for i in range(b):
        ref = _f64(qkv.double().view(b, -1, d)[i, :hq], kk[i], vv[i], d ** -0.5)
        worst = max(worst, ((out[i].cpu().double().view(hq, d) - ref).norm() / ref.norm()).item())
    # as in _case; the error of the largest score, 16, is in all of the result: 16 x 2^-11 + 2 x 2^-11, or 16 / 4 x 2^-8 + 2^-8
    assert worst < (2e-2 if fp8 and d == 128 else 9e-3), worst


def _plain(d, fp8, qkv, kd, vd, past, table, hq, hkv):
    b = qkv.shape[0]
    out = torch.empty(b, hq * d, dtype=torch.float16, device="cuda")
    ws = torch.empty(hip.attn_decode_ws_floats(b, hq, hkv, 1, d, 1), dtype=torch.float32, device="cuda")
    counters = torch.zeros(hip.attn_decode_counters(b, hq, hkv), dtype=torch.int32, device="cuda")
    hip.attn_decode(qkv, kd, vd, torch.full((b,), past, dtype=torch.int32, device="cuda"), out, ws, counters, n_heads=hq, n_kv_heads=hkv,
                    head_dim=d, q_len=1, batch=b, scale=d ** -0.5, splits=1, rope_table=table)
    return out


def _small_cache(d, fp8, hkv, lmax):
    k, v = torch.randn(1, hkv, lmax, d, device="cuda").half(), torch.randn(1, hkv, d, lmax, device="cuda").half()
    return (t.to(torch.float8_e5m2).view(torch.uint8) if fp8 else t for t in (k, v))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("d", [64, 128])
def test_a_rope_table_may_start_anywhere(d, fp8):
    torch.manual_seed(d)
    k, v = _small_cache(d, fp8, 4, LMAX)
    qkv = torch.randn(1, 24 * d, device="cuda").half()
    ang = torch.rand(LMAX, d // 2, device="cuda")
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    moved = torch.empty(table.numel() + 2, device="cuda")[2:].view_as(table).copy_(table)
    assert moved.data_ptr() % 16 == 8
    assert torch.equal(_plain(d, fp8, qkv, k.clone(), v.clone(), 300, table, 16, 4), _plain(d, fp8, qkv, k.clone(), v.clone(), 300, moved, 16, 4))


@pytest.mark.parametrize("d,fp8", [(64, False), (64, True), (128, False), (128, True)])
def test_heads_of_two_gib(d, fp8):
    """past what a 32-bit offset reaches: the register form, and the result of a small cache with the same keys"""
    torch.manual_seed(d)
    lmax = (1 << 31) // (d * (1 if fp8 else 2))
    ks, vs = _small_cache(d, fp8, 1, LMAX)
    kd = torch.zeros(1, 1, lmax, d, dtype=ks.dtype, device="cuda")
    vd = torch.zeros(1, 1, d, lmax, dtype=vs.dtype, device="cuda")
    kd[:, :, :LMAX], vd[..., :LMAX] = ks, vs
    qkv = torch.randn(1, 10 * d, device="cuda").half()
    ang = torch.rand(LMAX, d // 2, device="cuda")
    table = torch.stack([ang.cos(), ang.sin()], -1).contiguous()
    a, b = _plain(d, fp8, qkv, kd, vd, 1000, table, 8, 1), _plain(d, fp8, qkv, ks, vs, 1000, table, 8, 1)
    assert torch.equal(kd[:, :, :LMAX], ks) and torch.equal(vd[..., :LMAX], vs)
    # (each within the bound of _case of the exact result)
    assert ((a.double() - b.double()).norm() / b.double().norm()).item() < 2 * (1.2e-2 if fp8 and d == 128 else 5e-3)
