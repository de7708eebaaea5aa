"""Entry points that take tensors in place of their addresses: the native callables and ctypes' agree on what they pass and refuse."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

from bigdl_amd.ops import hip


def _both(name):
    L = hip.lib()
    fn = L.__getitem__(name)
    fn.argtypes = dict(bigdl_rms_norm=[ctypes.c_void_p] * 5 + [ctypes.c_int64, ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_float,
                                                              ctypes.c_int, ctypes.c_int, ctypes.c_void_p])[name]
    return getattr(L, name), hip._by_address(fn)


def test_every_launcher_is_bound():
    L = hip.lib()
    if not hip.linear_call_path().exists():
        pytest.skip("not built")
    for name in hip._LAUNCHERS:
        assert type(getattr(L, name)).__name__ == "builtin_function_or_method", name


def _sources():
    """the signatures of the entry points in csrc/hip, as hip._signature writes them"""
    kinds = {"int": "i", "int64_t": "l", "float": "f"}
    out = {}
    for path in (Path(hip.__file__).parent.parent / "csrc" / "hip").glob("*.hip"):
        for result, name, args in re.findall(r'extern "C" (\w+) (bigdl_\w+)\(([^)]*)\)', path.read_text()):
            types = [re.sub(r"\s*\w+$", "", re.sub(r"\bconst\b", "", a).strip()) for a in args.split(",")]
            out[name] = "".join("p" if "*" in t or t == "hipStream_t" else kinds.get(t, "?") for t in (result, *types))
    return out


def test_signatures_are_those_of_the_sources():
    declared, sources = hip.lib().signatures, _sources()
    assert set(declared) == {*hip._LAUNCHERS, *hip._LINEAR_CALLS}
    assert declared == {name: sources[name] for name in declared}
    if hip.linear_call_path().exists():
        assert hip._load_calls(hip.linear_call_path()).signatures() == declared


def _library(changed=None):
    """the library again, with the types of one entry point changed"""
    types = {"p": ctypes.c_void_p, "i": ctypes.c_int, "l": ctypes.c_int64, "f": ctypes.c_float}
    L = ctypes.CDLL(str(hip._LIB_PATH))
    for name, text in hip.lib().signatures.items():
        fn = getattr(L, name)
        fn.restype, *fn.argtypes = (types[c] for c in text)
        if name == changed:
            fn.argtypes = [*fn.argtypes[:-1], ctypes.c_int, fn.argtypes[-1]]
    return L


def test_other_signatures_are_not_bound(monkeypatch):
    if not hip.linear_call_path().exists():
        pytest.skip("not built")
    native = "builtin_function_or_method"
    L = _library()
    hip._bind_launchers(L)
    assert all(type(getattr(L, name)).__name__ == native for name in hip._LAUNCHERS)
    L = _library("bigdl_gemm_prompt")
    with pytest.warns(UserWarning, match="bigdl_gemm_prompt$"):
        hip._bind_launchers(L)
    assert [name for name in hip._LAUNCHERS if type(getattr(L, name)).__name__ != native] == ["bigdl_gemm_prompt"]
    for changed, declines in (("bigdl_gemm_rows", True), ("bigdl_rms_norm", False)):
        L = _library(changed)
        L.signatures = {name: hip._signature(getattr(L, name)) for name in hip.lib().signatures}
        monkeypatch.setattr(hip, "lib", lambda: L)
        hip.linear_call.cache_clear()
        if declines:
            with pytest.warns(UserWarning, match="bigdl_gemm_rows"):
                assert hip.linear_call() is hip._declined
        else:
            assert hip.linear_call() is not hip._declined
        monkeypatch.undo()
    hip.linear_call.cache_clear()
    hip.linear_call()


def test_arguments_are_checked():
    native, by_ctypes = _both("bigdl_rms_norm")
    t = torch.zeros(8).half()
    for fn in (native, by_ctypes):
        # (a width that no kernel takes: refused by the entry point itself, no launch)
        assert fn(t, None, t, t, None, 1, 0, 8, 1e-5, 0.0, 0, 0, 0) != 0
        for bad in ((t,), (t, None, t, t, None, "1", 8, 8, 1e-5, 0.0, 0, 0, 0), (t, None, t, 1.5, None, 1, 8, 8, 1e-5, 0.0, 0, 0, 0)):
            with pytest.raises((TypeError, AttributeError, ctypes.ArgumentError)):
                fn(*bad)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width", [(1, 128), (77, 4096), (3, 4104)])
def test_same_results_either_way(monkeypatch, rows, width):
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, r, w = (torch.randn(*s, device="cuda", generator=g).half() for s in ((rows, width), (rows, width), (width,)))
    native, by_ctypes = _both("bigdl_rms_norm")
    outs = []
    for fn in (native, by_ctypes):
        monkeypatch.setattr(hip.lib(), "bigdl_rms_norm", fn)
        added = torch.empty_like(x)
        outs.append((hip.rms_norm(x, w, 1e-5, residual=r, res_out=added), added))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
