"""RMSNorm at the edges of a thread's pieces (256 threads of eight elements, fewer wavefronts for narrow rows): against 64 bits, sums in place,
with and without a residual."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,h", [(1, 8), (5, 512), (3, 520), (700, 1024), (3, 1032), (2, 1536), (3, 1544), (5, 2040), (5, 2048), (3, 2056), (2, 4096),
                                    (3, 8184), (2, 16384)])
def test_widths(rows, h, dtype):
    from bigdl_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(h)
    x, r, w = (torch.randn(*s, device="cuda", generator=g).to(dtype) for s in ((rows, h), (rows, h), (h,)))
    ulp = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -23}[dtype]

    def ref(t):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-5) * (w.double() + 1.0)

    # one rounding of the result; fp32 sums of squares (2^-24 times the depth of the sum) and a handful of fp32 operations: 2^-20
    plain = ref(x.double())
    assert ((hip.rms_norm(x, w, 1e-5, offset=1.0).double() - plain).abs() <= plain.abs() * (ulp + 2.0 ** -20) + 1e-7).all()
    total = x.double() + r.double()
    want = ref(total)
    added = r.clone()
    got = hip.rms_norm(x, w, 1e-5, offset=1.0, residual=added, res_out=added)          # the residual stream is summed in place
    assert ((got.double() - want).abs() <= want.abs() * (ulp + 2.0 ** -20) + 1e-7).all()
    assert ((added.double() - total).abs() <= total.abs() * ulp + 1e-7).all()


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("rows,h", [(1, 8), (5, 2056), (3, 4096), (2, 8200)])
def test_parts(rows, h, parts):
    from bigdl_amd.ops import hip
    g = torch.Generator(device="cuda").manual_seed(h + parts)
    slabs = torch.randn(parts, rows, h, device="cuda", generator=g)
    r, w, bias = (torch.randn(*s, device="cuda", generator=g).half() for s in ((rows, h), (h,), (h,)))
    for b in (None, bias):
        for res in (None, r):
            total = slabs.double().sum(0) + (0 if b is None else b.double()) + (0 if res is None else res.double())
            want = total * torch.rsqrt(total.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
            added = torch.empty_like(r)
            got = hip.rms_norm(hip.Parts(slabs, b), w, 1e-5, residual=res, res_out=added)
            # as above; a sum that cancels keeps the error of its terms: 2^-23 of their magnitudes, scaled like the result
            mag = slabs.double().abs().sum(0) + 8
            scale = (want / total).abs().nan_to_num(0, 0, 0)
            assert ((got.double() - want).abs() <= want.abs() * (2.0 ** -11 + 2.0 ** -20) + mag * scale * 2.0 ** -22 + 1e-7).all()
            assert ((added.double() - total).abs() <= total.abs() * 2.0 ** -11 + mag * 2.0 ** -22).all()


def _sum_of_squares(v):
    """v fp32 [rows, h], h up to 2048, as the kernel adds it up: eight elements a thread, each square rounded with the sum and not before
    (80 bits hold the square and the sum), 64 threads by halves, four wavefronts one after the other"""
    t = np.zeros((v.shape[0], 256, 8), np.float32)
    t.reshape(v.shape[0], -1)[:, :v.shape[1]] = v
    s = np.zeros(t.shape[:2], np.float32)
    for j in range(8):
        wide = t[:, :, j].astype(np.longdouble)
        s = (wide * wide + s).astype(np.float32)
    s = s.reshape(-1, 4, 64)
    while s.shape[2] > 1:
        s = s[:, :, :s.shape[2] // 2] + s[:, :, s.shape[2] // 2:]
    s = s[:, :, 0]
    return ((s[:, 0] + s[:, 1]) + s[:, 2]) + s[:, 3]


@pytest.mark.parametrize("kind", ["plain", "add", "parts"])
@pytest.mark.parametrize("h", [8, 512, 2048])
def test_squares_are_added_unrounded(h, kind):
    """eps takes all but 2^-17 of the mean away, so that the last bit of the sum of squares is 2^-8 of the result"""
    from bigdl_amd.ops import hip
    rows = 64
    g = torch.Generator().manual_seed(h)
    x, y = torch.randn(rows, h, generator=g), torch.randn(rows, h, generator=g)
    r, w = torch.randn(rows, h, generator=g).half(), torch.ones(h)
    if kind == "plain":
        args, v = (x.cuda(), w.cuda()), x
    elif kind == "add":
        # (small residuals: sums of more than 12 bits, whose squares fp32 does not hold)
        r = (r.float() * 2.0 ** -9).half()
        args, v = (x.half().cuda(), w.half().cuda()), x.half().float() + r.float()
    else:
        args, v = (hip.Parts(torch.stack([x, y]).cuda(), None), w.half().cuda()), r.float() + (x + y)
    mean = _sum_of_squares(v.numpy()) / np.float32(h)
    for i in range(rows):
        eps = float(-mean[i] * np.float32(1 - 2.0 ** -17))
        res = None if kind == "plain" else r.cuda()
        got = hip.rms_norm(*args, eps, residual=res)[i].double().cpu()
        want = v[i].double() / np.sqrt(float(mean[i] + np.float32(eps)))
        # one rounding to fp16, the root's few units and one product in fp32
        assert ((got - want).abs() <= want.abs() * (2.0 ** -11 + 2.0 ** -20) + 1e-6).all(), i
