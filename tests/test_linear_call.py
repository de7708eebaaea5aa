"""The native call of a few-row product (csrc/torch_ext/linear_call.cpp) against the Python way it shortens: what it declines, and
the same bits where it does not."""
import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import hip, host
from bigdl_amd.transformers import low_bit_linear as lbl

CALL = (64, 256, Q.SYM_INT4, 64 * 256 // 2 + 64 * 8 * 2, 16, 256)


def _module():
    if not hip.linear_call_path().exists():
        pytest.skip("not built")


@pytest.fixture()
def fresh():
    hip.linear_call.cache_clear()
    yield
    hip.linear_call.cache_clear()


@pytest.mark.parametrize("content", [None, b"", b"not a library"], ids=["missing", "empty", "text"])
def test_a_module_that_does_not_load_leaves_the_calls_to_python(monkeypatch, tmp_path, fresh, content, recwarn):
    path = tmp_path / "bigdl_linear_call.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(hip, "linear_call_path", lambda: path)
    assert hip.linear_call()(torch.zeros(1, 256).half(), torch.zeros(CALL[3], dtype=torch.uint8), *CALL) is None
    assert hip.linear_call() is hip.linear_call()
    assert len([w for w in recwarn if "linear_call" in str(w.message)]) == (content is not None)


def test_a_module_for_another_pytorch_is_not_looked_at(monkeypatch):
    path = hip.linear_call_path()
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    assert hip.linear_call_path() != path and hip.linear_call_path().parent == path.parent


def test_the_other_libraries_are_built_where_this_one_cannot_be(monkeypatch, capsys):
    from bigdl_amd.csrc import build
    done = []
    for name in ("ragged", "host", "hip"):
        monkeypatch.setattr(build, f"build_{name}", lambda *args, name=name, **kw: done.append(name) or name)

    def fails(cmd):
        raise RuntimeError("no such header")

    monkeypatch.setattr(build, "_run", fails)
    assert build.build_all(force=True) == ("host", "hip") and done == ["ragged", "host", "hip"]
    assert "no such header" in capsys.readouterr().err


def test_declines_what_is_not_on_the_gpu():
    _module()
    product = hip.linear_call()
    w = torch.zeros(CALL[3], dtype=torch.uint8)
    for x in (torch.zeros(1, 256).half(), torch.zeros(1, 256), torch.nn.Parameter(torch.zeros(1, 256).half()), None, 3):
        assert product(x, w, *CALL) is None
    assert product(torch.zeros(1, 256).half(), w) is None
    with pytest.raises(TypeError):
        product(torch.zeros(1, 256).half(), w, "64", *CALL[1:])


def _linear(qname, n, k, seed=0):
    lin = lbl.LowBitLinear(k, n, Q.ggml_tensor_qtype[qname], bias=False)
    w = torch.randn(n, k, generator=torch.Generator().manual_seed(seed)) * k ** -0.5
    lin.weight = lbl.FP4Params(host.quantize(w, lin.qtype), quantized=True, _shape=(n, k), qtype=lin.qtype)
    return lin.to("cuda").eval()


@pytest.fixture()
def both(monkeypatch):
    """the module's result, its result without the native call, and whether that took the call"""
    _module()
    native = hip.linear_call()

    def run(lin, x):
        took = []

        def counted(*args):
            y = native(*args)
            took.append(y is not None)
            return y

        monkeypatch.setattr(hip, "linear_call", lambda: counted)
        a = lin(x)
        monkeypatch.setattr(hip, "linear_call", lambda: lambda *args: None)
        b = lin(x)
        monkeypatch.setattr(hip, "linear_call", lambda: native)
        return a, b, any(took)
    return run


def _same(a, b):
    return a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 2, 16, 17, 32, 33, 100, 256, 257])
@pytest.mark.parametrize("qname,n,k", [("sym_int4", 72, 256), ("asym_int5", 1040, 288), ("fp8_e4m3", 256, 1024), ("q6_k", 40, 512)])
def test_same_bits(both, qname, n, k, rows):
    lin = _linear(qname, n, k)
    x = torch.randn(rows, k, device="cuda", dtype=torch.float16)
    with torch.no_grad():
        a, b, took = both(lin, x)
        assert _same(a, b) and took == (rows <= (128 if qname == "q6_k" else 256))
        a, b, took = both(lin, x.view(1, rows, k))
        assert _same(a, b) and a.shape == (1, rows, n) and took == (rows <= (128 if qname == "q6_k" else 256))


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [torch.enable_grad, torch.no_grad, torch.inference_mode])
@pytest.mark.parametrize("rows", [1, 18, 100])
def test_views_take_the_native_call(both, mode, rows):
    """What a model passes: hidden states of three dimensions, which are flattened by a view, and pieces of larger tensors"""
    lin = _linear("sym_int4", 128, 512)
    with mode():
        wide = torch.randn(2, rows, 1024, device="cuda", dtype=torch.float16)
        for x in (wide[:1, :, :512].contiguous(), wide[:, :, 512:].contiguous(), wide[0, :, :512], wide.view(-1, 512)[rows:2 * rows],
                  (wide[:1] * 2).view(1, 2 * rows, 512)):
            a, b, took = both(lin, x)
            assert took and _same(a, b) and a.shape == (*x.shape[:-1], 128)
    with torch.autograd.forward_ad.dual_level():
        x = torch.randn(1, rows, 512, device="cuda", dtype=torch.float16)
        a, b, took = both(lin, torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
        assert not took and _same(a, b)
    x = torch.randn(1, rows, 512, device="cuda", dtype=torch.float16, requires_grad=True)
    a, b, took = both(lin, x * 1)
    assert not took and _same(a, b) and a.requires_grad == b.requires_grad


@pytest.mark.gpu
def test_other_inputs_go_the_python_way_or_agree(both):
    lin = _linear("sym_int4", 128, 256)
    wide = torch.randn(8, 512 + 3, device="cuda", dtype=torch.float16)
    flat = torch.randn(4 * 256 + 8, device="cuda", dtype=torch.float16)
    for x in (wide[:, :256], wide[:, 3:259], wide[::2, :256], flat[8:1032].view(4, 256),
              torch.randn(256, 8, device="cuda", dtype=torch.float16).t(), flat[:256].expand(5, 256)):
        a, b, _ = both(lin, x)
        assert _same(a, b)
    for dtype, rows, native in ((torch.bfloat16, 3, True), (torch.bfloat16, 17, True), (torch.bfloat16, 32, True),
                                (torch.bfloat16, 33, False), (torch.float32, 3, False)):
        a, b, took = both(lin, torch.randn(rows, 256, device="cuda").to(dtype))
        assert _same(a, b) and took == native
    a, b, took = both(_linear("sym_int4", 128, 4096), torch.randn(16, 4096, device="cuda").bfloat16())
    assert _same(a, b) and not took                        # 64 Ki values: converted by a kernel of the package
    a, b, took = both(_linear("q6_k", 40, 512), torch.randn(3, 512, device="cuda").bfloat16())
    assert _same(a, b) and not took
    a, b, took = both(lin, torch.empty(0, 256, device="cuda", dtype=torch.float16))
    assert _same(a, b) and not took
    with torch.inference_mode():
        a, b, took = both(lin, torch.randn(3, 256, device="cuda", dtype=torch.float16))
        assert _same(a, b) and took and a.is_inference() and b.is_inference()
    x = torch.randn(3, 256, device="cuda", dtype=torch.float16, requires_grad=True)
    a, b, took = both(lin, x)
    assert _same(a, b) and not took and a.requires_grad == b.requires_grad
    with pytest.raises(RuntimeError):                      # rows off 16 bytes: refused as before
        lin(flat[1:1025].view(4, 256))
    with pytest.raises(ValueError):
        lin(torch.randn(3, 128, device="cuda", dtype=torch.float16))


@pytest.mark.gpu
def test_observed_q6k_inputs_keep_their_operations(both):
    from torch.utils._python_dispatch import TorchDispatchMode
    lin = _linear("q6_k", 40, 512)
    x = torch.randn(3, 512, device="cuda", dtype=torch.float16)

    class Seen(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Seen.ops += 1
            return func(*args, **(kwargs or {}))

    with Seen():
        a, b, took = both(lin, x)
    assert not took and Seen.ops > 2 and _same(a, b)
    a, b, took = both(lin, torch.vmap(lambda r: r * 1)(x))
    assert took and _same(a, b)
    out = torch.vmap(lambda r: lin(r[None])[0])(x)
    assert torch.allclose(out, lin(x), atol=2e-3, rtol=2e-2)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        a, b, took = both(lin, dual)
        tangents = [torch.autograd.forward_ad.unpack_dual(t).tangent for t in (a, b)]
        assert not took and tangents[0] is not None and torch.equal(*tangents)


@pytest.mark.gpu
def test_streams_and_graphs():
    _module()
    lin = _linear("sym_int4", 512, 1024)
    x = torch.randn(40, 1024, device="cuda", dtype=torch.float16)
    with torch.no_grad():
        want = lin(x)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = lin(x)
        torch.cuda.current_stream().wait_stream(side)
        assert torch.equal(y, want)
        graph, static = torch.cuda.CUDAGraph(), x.clone()
        with torch.cuda.graph(graph):
            y = lin(static)
        for i in range(3):
            new = torch.randn_like(x)
            static.copy_(new)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, lin(new))
