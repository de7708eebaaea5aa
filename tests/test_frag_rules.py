"""Which products take x in fragment order, and who takes such x: decisions that need no GPU."""
from types import SimpleNamespace

import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.models import decoder as D
from bigdl_amd.ops import hip

QT = Q.ggml_tensor_qtype["sym_int4"]


def test_x_in_fragment_order_is_not_rows():
    """only the entry points that ask for the type take it: to all others it would be rows of permuted values"""
    x = hip.Frags(torch.zeros(hip.frag_halves(48, 256), dtype=torch.float16), 48, 256)
    with pytest.raises(ValueError, match="rows"):
        hip._need_cuda(x)


@pytest.mark.parametrize("gemv_max,taken", [(16, True), (63, True), (64, False)])
def test_engine_gives_gemv_rows(monkeypatch, gemv_max, taken):
    """the products that ``gemv_lowbit`` runs (BIGDL_GEMV_MAX_ROWS) take rows"""
    monkeypatch.setattr(D, "GEMV_MAX_ROWS", gemv_max)
    lin = SimpleNamespace(fused=True, n=4096, k=4096, qtype=QT)
    eng = SimpleNamespace(prefill_fused=True, prefill_fp8=False)
    for prompt in (False, True):
        assert D.NativeDecoder._takes_frags(eng, 64, lin, prompt=prompt) == taken
