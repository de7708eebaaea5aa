"""Products of a q6_k weight that the block kernels do not take: what PyTorch has to see goes through its own operations."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import host

pytestmark = pytest.mark.gpu
N, K = 96, 512


@pytest.fixture(scope="module")
def weight():
    from bigdl_amd.transformers.low_bit_linear import FP4Params
    w = torch.randn(N, K, generator=torch.Generator().manual_seed(1)) * 0.05
    p = FP4Params(host.quantize(w, Q.Q6_K), quantized=True, _shape=(N, K), qtype=Q.Q6_K).to("cuda")
    return p, host.dequantize(p.data.cpu(), Q.Q6_K, (N, K)).double()


def _x(m, dtype=torch.float16, seed=2):
    return torch.randn(m, K, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _close(got, ref):
    # fp16 weights and results: 2^-11 each, on rows of 512 products
    torch.testing.assert_close(got.detach().cpu().double(), ref, rtol=2e-3, atol=8e-3)


@pytest.mark.parametrize("m", [1, 20, 128])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_gradient_in_eval_mode(weight, m, dtype):
    """gradients pass through a frozen layer that is not in training mode"""
    from bigdl_amd.transformers.low_bit_linear import LowBitLinear
    p, w = weight
    lin = LowBitLinear(K, N, qtype=Q.Q6_K, bias=False)
    lin.weight = p
    lin.eval()
    x = _x(m, dtype).requires_grad_()
    y = lin(x)
    _close(y, x.detach().cpu().double() @ w.t())
    dy = torch.randn(m, N, generator=torch.Generator().manual_seed(3)).to(dtype)
    y.backward(dy.cuda())
    _close(x.grad, dy.double() @ w)
    with torch.no_grad():
        assert not lin(x).requires_grad


def test_transforms_and_traces(weight):
    from bigdl_amd.transformers.low_bit_linear import lowbit_matmul
    p, w = weight
    f = lambda t: lowbit_matmul(t, p, N)
    x, v = _x(5), _x(5, seed=4)
    xd, vd = x.cpu().double(), v.cpu().double()
    jac = torch.autograd.functional.jacobian(f, x[:1])
    _close(jac[0, :, 0], w)
    with torch.autograd.forward_ad.dual_level():
        out = torch.autograd.forward_ad.unpack_dual(f(torch.autograd.forward_ad.make_dual(x, v)))
        _close(out.tangent, vd @ w.t())
    _close(torch.vmap(lambda r: f(r[None])[0])(x), xd @ w.t())
    traced = torch.jit.trace(f, (x,), check_trace=False)
    _close(traced(v), vd @ w.t())
    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False) as count:
        y = f(x)
    _close(y, xd @ w.t())
    assert count.get_total_flops() == 2 * 5 * N * K


def test_types_and_shapes_outside_the_kernels(weight):
    from bigdl_amd.transformers.low_bit_linear import lowbit_matmul
    p, w = weight
    x = _x(3, torch.float64)
    y = lowbit_matmul(x, p, N)
    assert y.dtype == torch.float64
    _close(y, x.cpu() @ w.t())
    assert lowbit_matmul(x[:0].half(), p, N).shape == (0, N)
    with pytest.raises((ValueError, RuntimeError)):
        lowbit_matmul(x.half()[:, :256].contiguous(), p, N)
