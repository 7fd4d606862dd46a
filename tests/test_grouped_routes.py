"""Which kernel a grouped GEMM call goes to: the dispatch alone, on CPU tensors and a recorder in the kernels' place."""
import pytest
import torch

from llm_weighted_consensus_amd import ops


class Recorder:
    """Stands for the extension: notes each call's name and the core it asks for."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            core = args[-1] if name in ("gemm8g_bf16", "gemm8g_fp8") else None
            self.calls.append((name, core))
        return call


@pytest.fixture
def taken(monkeypatch):
    r = Recorder()
    monkeypatch.setattr(ops, "kernels", lambda: r)
    return r.calls


def _call(rows, G=4, N=128, K=128, fp8=False, **kw):
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16
    A, W = torch.zeros(rows, K, dtype=dt), torch.zeros(G, N, K, dtype=dt)
    scales = dict(a_scale=torch.ones(rows), w_scale=torch.ones(G, N)) if fp8 else {}
    ops.grouped_gemm(A, W, torch.zeros(G + 1, dtype=torch.int32), **scales, **kw)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("rows", [1, 2000])
def test_forced_expert_kernels(taken, monkeypatch, fp8, swiglu, rows):
    """LWC_MOE_GEMM names the kernel of fp8 and bf16 experts alike, at any row count."""
    own = "gemm8g_fp8" if fp8 else "gemm8g_bf16"
    for mode, want in (("classic", ("grouped_gemm", None)), ("g2", (own, 2)), ("g8", (own, 8))):
        taken.clear()
        monkeypatch.setattr(ops, "MOE_GEMM", mode)
        _call(rows, fp8=fp8, swiglu=swiglu)
        assert taken[0] == want and [n for n, _ in taken[1:]] == (["silu_mul"] if swiglu and mode == "classic" else [])


def _bf16(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("form", ["expanded rows", "overlapping rows", "output beyond A", "fewer rows than A", "longer output", "no K"])
def test_bf16_forms_that_stay_with_the_128_row_kernel(taken, form):
    """Calls that the small-tile and 256-row kernels answer differently from the 128-row kernel: A's rows at one address or
    overlapping (their buffers would end early: zeros), and what they would refuse, or take though it was refused."""
    G, N, K, rows, out, kw = 4, 128, 128, 512, None, {}
    A = _bf16(rows, K)
    if form == "expanded rows":
        A = _bf16(1, K).expand(rows, K)
    elif form == "overlapping rows":
        A = _bf16(rows * 64 + K).as_strided((rows, K), (64, 1))
    elif form == "output beyond A":
        kw["rows"] = rows + 16
    elif form == "fewer rows than A":
        kw["rows"] = rows - 16
    elif form == "longer output":
        kw.update(out=_bf16(rows + 16, N), a_rows=torch.zeros(rows + 16, dtype=torch.int32), rows=rows)
    else:
        K, A = 0, _bf16(rows, 0)
    ops.grouped_gemm(A, _bf16(G, N, K), torch.zeros(G + 1, dtype=torch.int32), **kw)
    assert [n for n, _ in taken] == ["grouped_gemm"]


@pytest.mark.parametrize("swiglu", [False, True])
def test_bf16_rows_of_a_wider_matrix_and_gathered_rows(taken, swiglu):
    G, N, K, rows = 4, 1024, 128, 512
    for A, kw in ((_bf16(rows, K + 8)[:, :K], {}), (_bf16(9, K), dict(a_rows=torch.zeros(rows, dtype=torch.int32)))):
        taken.clear()
        ops.grouped_gemm(A, _bf16(G, N, K), torch.zeros(G + 1, dtype=torch.int32), swiglu=swiglu, **kw)
        assert [n for n, _ in taken] == ["gemm8g_bf16"]


@pytest.mark.parametrize("N,K,G,rows,core", [
    # (what measured fastest, ``ops._grouped_bf16``)
    (4096, 14336, 8, 400, 8), (14336, 4096, 2, 192, 8), (2048, 7168, 8, 192, 2), (4096, 14336, 2, 256, 0), (2048, 7168, 8, 16, 2),
    (14336, 4096, 2, 16, 2), (4096, 14336, 4, 16, 0), (4096, 14336, 2, 16, 0), (2048, 7168, 4, 16, 0), (512, 1024, 8, 16, 2),
    (1536, 2048, 128, 8, 2), (1536, 2048, 128, 44, 0), (1536, 2048, 128, 160, 2), (2048, 768, 128, 44, 0), (2048, 768, 128, 160, 2),
    (2048, 512, 256, 16, 0), (2048, 512, 256, 160, 0), (2816, 2048, 64, 44, 2), (4096, 3072, 64, 44, 2), (28672, 4096, 8, 16, 2), (6144, 16384, 8, 4, 0), (6144, 16384, 8, 16, 2),
    # fewer than four rows a group; N off 16, which the 128-row kernel does not take
    (14336, 4096, 8, 3, 0), (328, 4096, 2, 16, 2), (328, 4096, 2, 200, 8)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_bf16_kernel_by_sizes(taken, monkeypatch, N, K, G, rows, core, swiglu):
    if swiglu and N % 64:
        pytest.skip("SwiGLU pairs blocks of 32")
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: None)   # (no result is needed)
    monkeypatch.setattr(ops, "silu_mul", lambda *a, **kw: None)
    ops.grouped_gemm(_Shape(G * rows, K), _Shape(G, N, K), None, swiglu=swiglu)
    assert taken[0] == (("gemm8g_bf16", core) if core else ("grouped_gemm", None))


@pytest.mark.parametrize("N,K,G,rows,core", [
    # (less than three rows a group, ``ops._few_bf16``: rows of all groups)
    (14336, 4096, 8, 2, 2), (14336, 4096, 8, 3, 0), (14336, 4096, 8, 5, 0), (14336, 4096, 8, 24, 0), (14336, 4096, 8, 31, 0), (4096, 14336, 8, 4, 0),
    (4096, 14336, 8, 8, 2), (4096, 14336, 8, 23, 2), (4096, 14336, 8, 24, 0), (4096, 7168, 8, 2, 0), (4096, 7168, 8, 4, 2), (4096, 8192, 8, 4, 0), (1536, 2048, 128, 64, 2), (2048, 768, 128, 128, 0),
    (4096, 4096, 2, 4, 0), (6144, 16384, 8, 8, 0), (328, 4096, 64, 128, 0)])
def test_bf16_kernel_of_few_rows(taken, monkeypatch, N, K, G, rows, core):
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: None)   # (no result is needed)
    ops.grouped_gemm(_Shape(rows, K), _Shape(G, N, K), None)
    assert taken[0] == (("gemm8g_bf16", core) if core else ("grouped_gemm", None))


@pytest.mark.parametrize("N,K,G,rows,few", [
    # (what measured fastest, ``ops._few_fp8``: rows of all groups)
    (28672, 4096, 8, 2, True), (4096, 14336, 8, 2, False), (4096, 14336, 8, 4, True), (4096, 16384, 8, 4, True), (2816, 2048, 32, 8, True),
    (4096, 4096, 2, 1, True), (2048, 768, 128, 400, False), (2048, 512, 256, 64, False), (2048, 7168, 8, 255, True), (2048, 7168, 8, 8, False), (2048, 7168, 8, 16, True), (4096, 8192, 8, 2, False)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_fp8_kernel_of_few_rows(taken, monkeypatch, N, K, G, rows, few, swiglu):
    """Row scales either way: the middle of an expert stays out of MX form below 32 rows a group."""
    monkeypatch.setattr(ops, "silu_mul", lambda *a, **kw: None)
    scales = dict(a_scale=torch.ones(rows), w_scale=torch.ones(G, N))
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: None)   # (no result is needed)
    ops.grouped_gemm(_Shape(rows, K, dtype=torch.float8_e4m3fn), _Shape(G, N, K, dtype=torch.float8_e4m3fn), None, swiglu=swiglu, **scales)
    assert ops._few_fp8(rows, G, N, K) == few
    assert taken[0] == (("gemm8g_fp8", 2) if few else ("grouped_gemm", None))
    assert not ops.moe_mx_ok(torch.zeros(rows, 128, dtype=torch.float8_e4m3fn), torch.zeros(G, 256, 128, dtype=torch.float8_e4m3fn),
                             torch.zeros(G, 128, 128, dtype=torch.float8_e4m3fn), rows)


@pytest.mark.parametrize("form", ["expanded rows", "overlapping rows", "output beyond A", "fewer rows than A", "slots", "strided scales", "N off 16"])
def test_fp8_forms_of_few_rows_that_stay_with_the_128_row_kernel(taken, form):
    G, N, K, rows = 4, 256, 1024, 16
    f8 = lambda *s: torch.zeros(*s, dtype=torch.float8_e4m3fn)  # noqa: E731
    A, sc, kw = f8(rows, K), torch.ones(rows), {}
    if form == "expanded rows":
        A = f8(1, K).expand(rows, K)
    elif form == "overlapping rows":
        A = f8(rows * 64 + K).as_strided((rows, K), (64, 1))
    elif form == "output beyond A":
        kw["rows"] = rows + 16
    elif form == "fewer rows than A":
        kw["rows"] = rows - 2
    elif form == "slots":
        kw["max_slots"] = 9
    elif form == "strided scales":
        sc = torch.ones(2 * rows)[::2]
    else:
        N = 264
    ops.grouped_gemm(A, f8(G, N, K), torch.zeros(G + 1, dtype=torch.int32), a_scale=sc, w_scale=torch.ones(G, N), **kw)
    assert [n for n, _ in taken] == ["grouped_gemm"]


class _Shape:
    """A contiguous operand of which only the layout is looked at."""
    device = "cpu"

    def __init__(self, *shape, dtype=torch.bfloat16):
        self.shape, self.dtype = shape, dtype

    def stride(self, i):
        n = 1
        for d in self.shape[i + 1:]:
            n *= d
        return n

    def data_ptr(self):
        return 0

    def is_contiguous(self):
        return True

    def element_size(self):
        return self.dtype.itemsize
