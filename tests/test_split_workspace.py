"""The scratch memory of products whose partial sums pass through memory."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from bigdl_amd import qtypes as Q
from bigdl_amd.ops import hip, host

QT = Q.ggml_tensor_qtype["sym_int4"]


class _Allocations(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ptrs = set()

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        if "empty" in str(func):
            self.ptrs.add(out.data_ptr())
        return out


class _Library:
    """stands for the kernels' library: two K splits, one slab, and the workspace address that each launch is given"""
    at = {"bigdl_gemm_lowbit": 5, "bigdl_gemm_prompt": 5, "bigdl_gemm_lowbit_ex": 12, "bigdl_gemm_frag_dense": 7}

    def __init__(self):
        self.got, self.names = [], []

    def __getattr__(self, name):
        if name in self.at:
            return lambda *a: self.names.append(name) or self.got.append(a[self.at[name]]) or 0
        return lambda *a: 4096 if name.endswith("workspace") else 2


@pytest.fixture(autouse=True)
def _choices_of_the_real_library():
    """what the stand-in below answers is not remembered"""
    yield
    hip.gemm_lowbit_frag.cache_clear()


@pytest.mark.parametrize("call,frag", [("gemm_lowbit", False), ("gemm_lowbit_ex", False), ("gemm_prompt", False), ("gemm_lowbit", True),
                                       ("gemm_lowbit_ex", True)])
def test_every_call_allocates_its_own_scratch(monkeypatch, call, frag):
    """A buffer kept between calls is freed when a larger one takes its place, while captured graphs go on writing to it:
    what a launch gets must have been allocated by that call (under capture: from the graph's pool)."""
    lib = _Library()
    lib.bigdl_gemm_lowbit_frag = lambda *a: int(frag)          # (asked for more than 32 rows)
    hip.gemm_lowbit_frag.cache_clear()
    monkeypatch.setattr(hip, "lib", lambda: lib)
    monkeypatch.setattr(hip, "_need_cuda", lambda *t: None)
    monkeypatch.setattr(hip, "_stream", lambda: 0)
    n, k = 32, 256
    w = torch.zeros(host.device_nbytes(QT, n, k), dtype=torch.uint8)
    keep = []
    for m in (20, 20, 40, 20):
        x = torch.zeros(m, k, dtype=torch.float16)
        with _Allocations() as made:
            keep.append(getattr(hip, call)(x, w, QT, n, k))
        assert lib.got[-1] in made.ptrs
    assert len(lib.got) == 4 and lib.names.count("bigdl_gemm_frag_dense") == int(frag)


@pytest.mark.parametrize("m,n,k,pair,norms,floats", [
    (64, 11008, 4096, 1, 0, 0), (17, 14336, 4096, 1, 0, 0),      # a pair on the few-row kernel is combined in registers
    (64, 4096, 4096, 0, 0, 0),
    (64, 4096, 11008, 0, 0, 2 * 64 * 4096),            # the few-row kernel's two K splits
    (64, 11008, 4096, 1, 1, 2 * 2 * 64 * 11008),       # a folded norm: tile kernel, both products of two K splits through scratch
    (64, 12288, 4096, 0, 1, 3 * 64 * 12288),
    (300, 14336, 4096, 0, 0, 0)])
def test_scratch_is_that_of_the_kernel_that_runs(m, n, k, pair, norms, floats):
    assert hip.lib().bigdl_gemm_lowbit_workspace(m, n, k, k, QT, pair, norms, 0) == floats


@pytest.mark.parametrize("name,m,n,k,tile", [
    # slower on the few-row kernel by a tenth and more: narrow outputs of a long K, grids of several turns
    ("sym_int4", 65, 1024, 14336, True), ("asym_int4", 128, 2048, 14336, True), ("sym_int8", 128, 1024, 8192, True),
    ("sym_int4", 192, 4096, 11008, True),
    # faster there by a tenth and more; unsplit, so without scratch, which the tile kernel would need at these sizes
    ("sym_int4", 64, 4096, 4096, False), ("asym_int4", 128, 4096, 4096, False), ("sym_int8", 128, 2048, 2048, False),
    ("sym_int4", 128, 1024, 4096, False), ("nf4", 192, 2048, 5632, False), ("fp6", 65, 6144, 4096, False),
    # up to 64 rows and three turns, whatever the estimates say
    ("sym_int4", 33, 14336, 4096, False), ("sym_int4", 64, 14336, 4096, False), ("sym_int8", 64, 12288, 4096, False)])
def test_kernel_of_a_product(name, m, n, k, tile):
    floats = hip.lib().bigdl_gemm_lowbit_workspace(m, n, k, k, Q.ggml_tensor_qtype[name], 0, 0, 0)
    assert (floats > 0) == tile


@pytest.mark.parametrize("name,m,n,k,pair,norm,few", [
    # two turns of the few-row kernel for three to seven rows (28672 x 8192, 3 rows: 50.8 -> 75.4 us), small x, narrow outputs
    ("sym_int4", 3, 28672, 8192, 1, 0, 0), ("sym_int8", 4, 28672, 8192, 0, 0, 0), ("sym_int4", 3, 32000, 4096, 0, 0, 0),
    ("sym_int4", 4, 11008, 4096, 0, 0, 0), ("sym_int4", 8, 5632, 2048, 0, 0, 0), ("sym_int4", 7, 8192, 4096, 0, 0, 0),
    ("sym_int4", 12, 32000, 4096, 0, 0, 0), ("fp6", 16, 4096, 4096, 0, 0, 0), ("sym_int8", 4, 14336, 4096, 1, 0, 0),
    # and where it is ahead by a tenth and more
    ("asym_int4", 12, 6144, 4096, 0, 0, 1), ("asym_int4", 12, 14336, 4096, 1, 0, 1), ("asym_int4", 12, 4096, 14336, 0, 0, 1),
    ("sym_int4", 16, 32000, 4096, 0, 0, 1), ("sym_int4", 8, 11008, 4096, 1, 0, 1), ("fp6", 16, 11008, 4096, 0, 0, 1),
    ("sym_int4", 7, 4096, 11008, 0, 0, 1), ("sym_int8", 6, 8192, 8192, 0, 0, 1), ("sym_int4", 2, 32000, 4096, 1, 0, 0),
    # with a folded norm
    ("asym_int4", 12, 32000, 4096, 0, 1, 1), ("asym_int4", 8, 128256, 4096, 0, 1, 0), ("sym_int4", 8, 5632, 2048, 0, 1, 1),
    ("sym_int4", 5, 8192, 4096, 0, 1, 0), ("sym_int4", 5, 14336, 4096, 1, 1, 1), ("fp4", 3, 28672, 8192, 1, 1, 0)])
def test_kernel_of_a_few_rows(name, m, n, k, pair, norm, few):
    assert hip.lib().bigdl_gemv_lowbit_few_rows(m, n, k, Q.ggml_tensor_qtype[name], pair, norm) == few


@pytest.mark.gpu
def test_a_captured_split_product_outlives_larger_calls():
    """capture, a call that needs more scratch, new allocations, replay: the replays write to none of them"""
    g = torch.Generator().manual_seed(1)
    n, k, m = 4096, 11008, 64                                     # K split over workgroups
    w = (torch.randint(0, 256, (host.device_nbytes(QT, n, k),), dtype=torch.uint8, generator=g) & 0xBF).cuda()
    wide = (torch.randint(0, 256, (host.device_nbytes(QT, 8192, 256),), dtype=torch.uint8, generator=g) & 0xBF).cuda()
    x = torch.randn(m, k, generator=g).half().cuda()
    want = hip.gemm_lowbit(x, w, QT, n, k)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = hip.gemm_lowbit(x, w, QT, n, k)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    for rows in (600, 1500):
        hip.gemm_prompt(torch.ones(rows, 256, dtype=torch.float16, device="cuda"), wide, QT, 8192, 256, out_dtype=torch.float32)
        fresh = [torch.full((1 << 20,), float(i), device="cuda") for i in range(48)]
        x.copy_(torch.randn(m, k, generator=g).half())
        graph.replay()
        want = hip.gemm_lowbit(x, w, QT, n, k)
        assert torch.equal(out, want)
        assert all(bool((t == i).all()) for i, t in enumerate(fresh))
        del fresh
