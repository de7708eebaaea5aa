"""The few-row product of a q6_k weight: rows that start between two dwords, ragged last quads and items, one and many rows a wavefront."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu


def _exact(raw, n, k):
    """the weights in 64 bits: 32 codes of 32 j .. of a half from low dwords j & 1, nibble j >> 1, and high bits 2 j"""
    b = raw.view(-1, 210)
    ql, qh, sc = b[:, :128].int(), b[:, 128:192].int(), b[:, 192:208].contiguous().view(torch.int8).double()
    d = b[:, 208:].contiguous().view(torch.float16).double()
    out = []
    for half in range(2):
        low, high = ql[:, 64 * half:64 * half + 64], qh[:, 32 * half:32 * half + 32]
        for j in range(4):
            c = (low[:, 32 * (j & 1):32 * (j & 1) + 32] >> (4 * (j >> 1)) & 15 | (high >> (2 * j) & 3) << 4) - 32
            out.append(c * sc[:, 8 * half + 2 * j:8 * half + 2 * j + 2].repeat_interleave(16, 1) * d)
    return torch.cat(out, 1).view(n, k)


@pytest.mark.parametrize("n,k", [(1, 256), (333, 256), (40, 768), (96, 2048), (17, 2304), (40, 9984), (33, 16640), (2064, 8192), (8500, 512)])
def test_rows_between_dwords(n, k):
    from bigdl_amd.ops import hip
    g = torch.Generator().manual_seed(n + k)
    raw = host.quantize(torch.randn(n, k, generator=g) * 0.05, Q.Q6_K).view(-1)
    w = _exact(raw, n, k)
    buf = torch.full((raw.numel() + 256,), 0xFF, dtype=torch.uint8)        # the bytes around are NaN scales
    buf[16:16 + raw.numel()] = raw
    dev = buf.cuda()[16:16 + raw.numel()]
    for m in (1, 2, 3, 4):
        x = torch.randn(m, k, generator=g)
        x[0] *= 2e-6                                                         # a row of fp16's subnormal numbers alone
        x = x.half()
        y = hip.gemm_q6k(x.cuda(), dev, n, k, out_dtype=torch.float32).cpu().double()
        # fp32 sums: dot 4, scale 4, one a quad of blocks, six across lanes (2^-24 each); the tile kernel takes what is wider than
        # 40960 elements in all and rounds the weights to fp16
        wide = m * ((k // 256 + 3) // 4) * 1024 > 40960
        bound = 2.0 ** -11 if wide else (14 + (k + 1023) // 1024) * 2.0 ** -24
        err, mag = (y - x.double() @ w.t()).abs(), x.double().abs() @ w.abs().t()
        assert bool((err <= bound * mag + 1e-30).all()), (m, (err / mag.clamp_min(1e-30)).max().item())
