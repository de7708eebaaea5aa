"""Which products take x in fragment order, and who takes such x: decisions that need no GPU."""
from types import SimpleNamespace

import pytest
import torch

from bigdl_amd import qtypes as Q
from bigdl_amd.models import decoder as D
from bigdl_amd.ops import hip
from bigdl_amd.transformers.low_bit_linear import lowbit_matmul, lowbit_rows

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


@pytest.mark.parametrize("kind", [0, 1])
def test_rows_far_apart_stay_with_the_other_kernels(kind):
    """a call that the rule takes is one that the launcher accepts: rows 16 bytes aligned, the last one within 2^31 elements.  300 last
    positions of sequences of 2048 tokens are 600 K row widths."""
    m, k = 300, 4544
    assert hip.gemm_lowbit_frag(m, 4544, k, QT, k, False, kind)
    assert hip.gemm_lowbit_frag(m, 4544, k, QT, 1 << 22, False, kind)
    assert not hip.gemm_lowbit_frag(m, 4544, k, QT, 2048 * k, False, kind)
    assert not hip.gemm_lowbit_frag(m, 4544, k, QT, k + 4, False, kind)


@pytest.mark.parametrize("name,n,k", [("asym_int4", 14336, 4128), ("sym_int8", 14336, 4128), ("sym_int4", 4672, 4544)])
def test_many_rows_go_in_pieces(monkeypatch, name, n, k):
    """no multiple of 128 columns: calls of up to FRAG_MAX_ROWS rows, as measured; of 4096 rows the first two were slower than before"""
    qt = Q.ggml_tensor_qtype[name]
    assert hip.gemm_lowbit_frag(hip.FRAG_MAX_ROWS, n, k, qt) and not hip.gemm_lowbit_frag(hip.FRAG_MAX_ROWS + 1, n, k, qt)
    got = []
    monkeypatch.setattr(hip, "gemm_lowbit", lambda x, *a, out, **kw: got.append((x[0, 0].item(), x.shape[0], out[0, 0].item(), out.shape[0])))
    rows = torch.arange(4196).half()[:, None].repeat(1, 8)[:, :1]
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: rows.expand(4196, n))
    lowbit_rows(rows.expand(4196, k), None, qt, n, k)
    assert got == [(0, 2048, 0, 2048), (2048, 2048, 2048, 2048), (4096, 100, 4096, 100)]


@pytest.mark.parametrize("rows,asked", [(17, 0), (32, 0), (33, 1)])
def test_few_bf16_rows_ask_nothing(monkeypatch, rows, asked):
    """a call of 17 to 32 bf16 rows is bound by the host and the rule never takes it"""
    w = SimpleNamespace(is_cuda=True, _shape=(256, 256), qlayout="t16", qtype=QT)
    calls = []
    monkeypatch.setattr(hip, "gemm_lowbit_frag", lambda *a: calls.append(a) or False)
    monkeypatch.setattr(hip, "gemm_lowbit", lambda x, *a, **kw: x)
    y = lowbit_matmul(torch.ones(rows, 256, dtype=torch.bfloat16), w, 256)
    assert y.dtype == torch.float16 and len(calls) == asked


def test_scratch_sizes_are_the_librarys():
    """remembered per library: what one answers is not taken for another's"""
    lib = hip.lib()
    args = (64, 4096, 11008, 11008, QT, 0, 0, 0)
    assert hip._gemm_floats(lib, *args) == lib.bigdl_gemm_lowbit_workspace(*args) > 0

    class Other:
        def bigdl_gemm_lowbit_workspace(self, *a):
            return 7

    assert hip._gemm_floats(Other(), *args) == 7


@pytest.mark.parametrize("name,m,n,k,split", [("nf4", 34, 2048, 5632, False), ("fp4", 98, 1792, 14336, False),
                                              ("nf4", 70, 1280, 11776, True), ("sym_int4", 36, 1856, 11136, True)])
def test_a_split_is_worth_its_launch(name, m, n, k, split):
    """split K: a second launch, so only where the estimate is ahead by more than it may be off"""
    qt = Q.ggml_tensor_qtype[name]
    floats = hip.lib().bigdl_gemm_frag_workspace(m, n, k, qt, 0, 2)
    assert (floats > 0) == split and floats % (m * n) == 0


def test_out_and_fragment_order_exclude_each_other(monkeypatch):
    monkeypatch.setattr(hip, "_need_cuda", lambda *t: None)
    monkeypatch.setattr(hip, "_stream", lambda: 0)
    monkeypatch.setattr(hip, "lib", lambda: SimpleNamespace(bigdl_rms_norm=lambda *a: 0, bigdl_attn_prefill=lambda *a: 0))
    monkeypatch.setattr(hip, "_gemm_frag_dense", lambda *a, out, **kw: out)
    monkeypatch.setattr(hip, "gemm_lowbit_frag", lambda *a: True)
    x, w = torch.zeros(48, 128, dtype=torch.float16), torch.zeros(hip._t16_nbytes(QT, 128, 128), dtype=torch.uint8)
    q = x.view(1, 48, 1, 128).transpose(1, 2)
    for call in (lambda **kw: hip.rms_norm(x, x[0], 1e-5, frags=True, **kw),
                 lambda **kw: hip.gemm_lowbit_ex(x, w, QT, 128, 128, w2=w, out_frags=True, **kw),
                 lambda **kw: hip.attn_prefill(q, q, q, scale=1.0, frags=True, **kw)):
        assert type(call()) is hip.Frags
        with pytest.raises(ValueError, match="no out"):
            call(out=torch.empty_like(x))


def test_a_forced_prompt_plan_does_not_choose_the_kernel():
    """the choice is remembered by the product's sizes, so it may not depend on what a sweep forces for its own calls"""
    lib = hip.lib()
    for m, n, k in ((400, 4096, 11008), (512, 4096, 11008), (512, 12288, 4096), (512, 14336, 4096)):
        free = lib.bigdl_gemm_lowbit_frag(m, n, k, k, QT, 0, 0, 0)
        try:
            for cfg, splitk in ((0, 1), (2, 1), (2, 8)):
                hip.gemm_prompt_force(cfg, splitk)
                assert lib.bigdl_gemm_lowbit_frag(m, n, k, k, QT, 0, 0, 0) == free
        finally:
            hip.gemm_prompt_force()


@pytest.mark.parametrize("name,m,n,k,pair,kind,taken", [
    # rows, with the pass that orders them: measured ahead by a tenth and more
    ("sym_int8", 203, 4672, 4544, 0, 0, True), ("sym_int4", 256, 4096, 4096, 0, 0, True), ("sym_int4", 160, 4096, 4096, 0, 0, True),
    ("asym_int4", 300, 4096, 14336, 0, 0, True),
    # behind: a short K, which does not hide the exchange of the sums (nf4 18 -> 37 us), grids of several turns, a single row block
    ("nf4", 437, 11616, 640, 0, 0, False), ("fp8_e5m2", 341, 11504, 1536, 0, 0, False), ("sym_int4", 256, 14336, 4096, 0, 0, False),
    ("sym_int4", 64, 12288, 4096, 0, 0, False), ("fp8_e5m2", 35, 4160, 10880, 0, 0, False), ("sym_int4", 59, 2368, 9152, 1, 0, False),
    # alike on the GPU, a launch more for the host
    ("sym_int8", 90, 4096, 4544, 0, 0, False),
    # bf16 rows need a pass in any case
    ("sym_int4", 77, 4096, 4096, 0, 1, True), ("sym_int4", 32, 4096, 4096, 0, 1, False),
    # x that its producer writes in that order: a decode batch of 33 and 64, a prompt of 300 tokens; of 512 the pair is the prompt kernel's
    ("nf4", 33, 4096, 14336, 0, 3, True), ("sym_int4", 64, 4096, 11008, 0, 3, True), ("sym_int4", 64, 11008, 4096, 1, 3, True),
    ("sym_int4", 300, 12288, 4096, 0, 3, True), ("sym_int4", 512, 11008, 4096, 1, 3, False), ("nf4", 512, 14336, 4096, 1, 3, False),
    ("nf4", 513, 4096, 4096, 0, 3, False)])
def test_kernel_of_a_product(name, m, n, k, pair, kind, taken):
    assert hip.lib().bigdl_gemm_lowbit_frag(m, n, k, k, Q.ggml_tensor_qtype[name], pair, kind, 0) == taken


def test_a_pair_in_front_of_such_a_product():
    """the next product's pass, 4 us, is saved where the pair's result goes out in that order"""
    qt = Q.ggml_tensor_qtype["nf4"]
    taken = [[hip.gemm_lowbit_frag(m, 5632, 2048, qt, None, True, 3, out) for m in range(257, 513)] for out in (False, True)]
    assert sum(taken[0]) < sum(taken[1]) and all(b or not a for a, b in zip(*taken))
