"""The long-prompt attention (csrc/hip/attn_prefill.hip: 256 queries a workgroup, or 128 in split groups) against float64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# the form that the estimates choose, and each of the three
@pytest.fixture(scope="module", params=[-1, 0, 1, 2])
def hip(request):
    from bigdl_amd.ops import hip as h
    h.lib().bigdl_attn_prefill_force(request.param)
    yield h
    h.lib().bigdl_attn_prefill_force(-1)


def _inputs(b, hq, hkv, sq, lk, d, spread=1.0):
    """q, k as views of a fused row, v transposed in a cache with NaN behind the last key"""
    g = torch.Generator().manual_seed(sq + 3 * lk + d)
    rows = (torch.randn(b, lk, (hq + hkv) * d, generator=g) * spread).half().cuda()
    q = rows[:, lk - sq:, :hq * d].unflatten(-1, (hq, d)).transpose(1, 2)
    k = rows[..., hq * d:].unflatten(-1, (hkv, d)).transpose(1, 2)
    cache = torch.full((b, hkv, d, (lk + 31) // 8 * 8), float("nan"), dtype=torch.float16)
    cache[..., :lk] = torch.randn(b, hkv, d, lk, generator=g).half()
    return q, k, cache.cuda()[..., :lk]


def _reference(q, k, vt, scale, causal, window):
    q, k, v = q.double().cpu(), k.double().cpu(), vt.double().cpu().transpose(2, 3)
    n = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(n, 1), v.repeat_interleave(n, 1)
    pos = torch.arange(q.shape[2])[:, None] + k.shape[2] - q.shape[2]
    keys = torch.arange(k.shape[2])[None]
    hide = torch.zeros(q.shape[2], k.shape[2], dtype=torch.bool)
    if causal:
        hide |= keys > pos
    if window:
        hide |= keys <= pos - window
    w = torch.softmax((q @ k.transpose(2, 3) * scale).masked_fill(hide, -math.inf), -1)
    return (w @ v).transpose(1, 2).flatten(2), (w @ v.abs()).transpose(1, 2).flatten(2)


def _check(out, ref, size):
    # weights round to fp16 (2^-11 each, up to 2^-11 in all of them), fp32 exponents and sums, fp16 result
    assert ((out.double().cpu() - ref).abs() <= 2.0 ** -10 * size + 2.0 ** -11 * ref.abs() + 1e-6).all()


# (batch, heads, kv heads, queries, keys): either form by the number of workgroups; last query block of one query, whole, of one less;
# last key tile of 1, 63 and 64 keys; keys ahead of the queries; heads that divide by 8 and that do not
SHAPES = [(1, 48, 8, 321, 321), (1, 64, 64, 512, 512), (3, 32, 8, 383, 383), (1, 40, 8, 385, 449), (9, 5, 5, 513, 576), (1, 33, 3, 511, 512),
          (2, 64, 8, 640, 703)]


@pytest.mark.parametrize("b,hq,hkv,sq,lk", SHAPES)
@pytest.mark.parametrize("causal", [True, False])
def test_long_prompts(hip, b, hq, hkv, sq, lk, causal):
    q, k, vt = _inputs(b, hq, hkv, sq, lk, 128)
    out = hip.attn_prefill(q, k, vt, scale=128 ** -0.5, causal=causal, v_transposed=True)
    _check(out, *_reference(q, k, vt, 128 ** -0.5, causal, 0))


@pytest.mark.parametrize("sq,lk,window", [(1025, 1025, 0), (1088, 1151, 0), (1100, 1300, 100), (1279, 1280, 1000)])
def test_heads_of_64(hip, sq, lk, window):
    q, k, vt = _inputs(1, 32, 4, sq, lk, 64)
    out = hip.attn_prefill(q, k, vt, scale=0.125, v_transposed=True, window=window)
    _check(out, *_reference(q, k, vt, 0.125, True, window))


@pytest.mark.parametrize("window", [1, 64, 65, 300])
@pytest.mark.parametrize("hq", [16, 64])
def test_windows(hip, hq, window):
    q, k, vt = _inputs(1, hq, 8, 1030 if hq == 16 else 400, 1030, 128)
    out = hip.attn_prefill(q, k, vt, scale=0.09, v_transposed=True, window=window)
    _check(out, *_reference(q, k, vt, 0.09, True, window))


def test_running_maximum_that_jumps(hip):
    # scores that grow along the keys by far more than the lazily followed maximum may lag
    q, k, vt = _inputs(1, 64, 8, 400, 400, 128, spread=4.0)
    out = hip.attn_prefill(q, k, vt, scale=1.0, v_transposed=True)
    ref, size = _reference(q, k, vt, 1.0, True, 0)
    # (exponents of a few hundred: 2^-23 of them in fp32 on top)
    assert ((out.double().cpu() - ref).abs() <= 2.0 ** -9 * size + 2.0 ** -11 * ref.abs() + 1e-6).all()


def test_fragment_order_and_rows_apart(hip):
    q, k, vt = _inputs(2, 32, 8, 400, 400, 128)
    rows = hip.attn_prefill(q, k, vt, scale=0.09, v_transposed=True)
    wide = torch.full((2, 400, 32 * 128 + 64), 7.0, dtype=torch.float16, device="cuda")
    hip.attn_prefill(q, k, vt, scale=0.09, v_transposed=True, out=wide[..., :32 * 128])
    assert torch.equal(wide[..., :32 * 128], rows) and (wide[..., 32 * 128:] == 7).all()
    frags = hip.attn_prefill(q, k, vt, scale=0.09, v_transposed=True, frags=True)
    m, n = 800, 32 * 128
    order = frags.data[:n * ((m + 15) // 16) * 16].view(n // 32, (m + 15) // 16, 4, 16, 8)
    assert torch.equal(order.permute(1, 3, 0, 2, 4).reshape(-1, n)[:m], rows.view(m, n))
