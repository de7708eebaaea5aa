"""Entry points that take tensors in place of their addresses: the native callables and ctypes' agree on what they pass and refuse."""
import ctypes

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
