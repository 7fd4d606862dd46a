"""When a projection that no one tuned may run on a kernel of its own in the library call's place."""
import pytest
import torch
from torch.autograd import forward_ad

from llm_weighted_consensus_amd.ops import gemm_plan


def test_plain_tensors():
    x, w = torch.randn(2, 3), torch.nn.Parameter(torch.randn(4, 3), requires_grad=False)
    assert gemm_plan._plain(x, w)
    w.requires_grad_()
    with torch.no_grad():
        assert gemm_plan._plain(x, w)
    assert not gemm_plan._plain(x, w)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_duals_keep_the_library(which):
    with forward_ad.dual_level():
        ts = [torch.randn(2, 3) for _ in range(3)]
        assert gemm_plan._plain(*ts)
        ts[which] = forward_ad.make_dual(ts[which], torch.randn(2, 3))
        assert not gemm_plan._plain(*ts)
    assert gemm_plan._plain(*[torch.randn(2, 3)])


def test_transforms_modes_and_traces_keep_the_library():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    seen = []

    def f(x):
        seen.append(gemm_plan._plain(x))
        return x * 2

    x = torch.randn(3, 4)
    torch.vmap(f)(x)
    torch.func.jvp(f, (x,), (x,))
    torch.func.grad(lambda x: f(x).sum())(x)
    with FlopCounterMode(display=False):
        f(x)
    with FakeTensorMode():
        f(torch.randn(2))
    make_fx(f)(x)
    torch.jit.trace(f, (x,), check_trace=False)
    assert seen and not any(seen)
    f(x)
    assert seen[-1]


@pytest.mark.parametrize("M,N,K,epi,core", [
    # (what measured faster than the library, ``gemm_plan._untuned``, and beside it what did not)
    (5614, 28672, 4096, "swiglu", "g8"), (4700, 14336, 2048, "swiglu", "g8"), (9000, 8192, 1024, "swiglu", "g8"),
    (7500, 4096, 2048, "swiglu", "blas"), (5121, 8192, 4096, "swiglu", "blas"), (4608, 28672, 4096, "swiglu", "blas"),
    (10000, 32768, 8192, "swiglu", "blas"), (5, 28672, 4096, "swiglu", "g2"), (64, 16384, 2048, "swiglu", "g2"),
    (5, 4096, 8192, "swiglu", "blas"), (24, 16384, 8192, "swiglu", "blas"),
    (65, 28672, 4096, "swiglu", "blas"), (5, 4096, 4096, "plain", "gv"), (16, 8192, 1024, "residual", "gv"),
    (16, 16384, 1024, "plain", "blas"), (5, 6144, 4096, "plain", "blas"), (17, 4096, 4096, "plain", "blas"),
    (32, 4096, 14336, "residual", "blas"), (33, 4096, 14336, "residual", "g2"), (64, 16384, 1024, "plain", "g2"),
    (48, 8192, 4096, "plain", "blas"), (64, 14336, 4096, "plain", "blas"), (65, 4096, 14336, "plain", "blas"),
    (654, 22016, 4096, "swiglu", "g8"), (1900, 27648, 5120, "swiglu", "g8"), (913, 25600, 5120, "swiglu", "blas"), (1283, 25600, 5120, "swiglu", "g8"), (544, 28672, 4096, "swiglu", "blas"),
    (1901, 28672, 4096, "swiglu", "blas"), (2401, 28672, 4096, "swiglu", "g8"), (3601, 28672, 4096, "swiglu", "blas"),
    (1095, 14336, 4096, "swiglu", "blas"), (1095, 32768, 4096, "swiglu", "blas"), (777, 4096, 14336, "residual", "g8"),
    (777, 4096, 14336, "plain", "blas"), (896, 4096, 11008, "residual", "g8"), (897, 4096, 11008, "residual", "blas"), (960, 4096, 12800, "residual", "blas"),
    (961, 4096, 12800, "residual", "g8"), (913, 4096, 14336, "residual", "g8"), (1901, 4096, 14336, "residual", "blas"), (777, 5120, 13824, "residual", "blas")])
def test_untuned_rule(M, N, K, epi, core):
    assert gemm_plan._untuned(M, N, K, epi) == core


@pytest.mark.parametrize("N,K,epi,rows", [
    (128256, 4096, "plain", {1: "g2", 32: "g2", 33: "blas"}), (32000, 4096, "plain", {5: "g2"}), (31992, 4096, "plain", {5: "blas"}),
    (50304, 2048, "plain", {1: "g2"}), (49144, 2048, "plain", {1: "blas"}), (151936, 1984, "plain", {1: "blas"}), (65536, 8256, "plain", {1: "blas"}),
    (131072, 8192, "plain", {1: "blas"}), (128256, 4096, "residual", {5: "blas"}),
    (4096, 14336, "residual", {1: "g2", 24: "g2", 25: "blas"}), (4096, 14336, "plain", {5: "blas"}), (4088, 14336, "residual", {5: "blas"}),
    (4096, 11008, "residual", {24: "g2"}), (4096, 10944, "residual", {24: "blas"}), (5120, 14336, "residual", {1: "g2"}), (5128, 14336, "residual", {1: "blas"}),
    (4096, 14400, "residual", {1: "blas"})])
def test_untuned_rule_of_few_rows(N, K, epi, rows):
    assert {M: gemm_plan._untuned(M, N, K, epi) for M in rows} == rows


@pytest.mark.parametrize("M,N,K,own", [(4096, 4096, 512, False), (4097, 4096, 512, True), (4096, 4096, 896, False), (4096, 4096, 1024, True),
                                       (2048, 4096, 1024, False), (2049, 4096, 1024, True), (5000, 2048, 768, False), (8682, 2048, 512, True),
                                       (8682, 2048, 384, False), (1024, 4096, 12288, True), (1024, 4096, 8192, False)])
def test_dense_fp8_core_rule(M, N, K, own):
    """Which of the dense fp8 cores measured faster: gemm8p's from 1024 deep on where its tiles are at most the CUs, from 512 beyond."""
    from llm_weighted_consensus_amd import ops

    x, w = (torch.empty(r, K, dtype=torch.float8_e4m3fn) for r in (M, N))
    assert ops._fp8_gemm8p(M, N, K, object(), x, w) == own


@pytest.mark.parametrize("M,N,K,tile,past", [
    (1, 8192, 2040, (64, 64), False), (1, 8192, 2048, (64, 64), True), (48, 256000, 3584, (64, 64), True), (49, 128256, 4096, (64, 64), False),
    (64, 65536, 8192, (64, 64), True), (64, 128256, 2048, (64, 64), True), (64, 81920, 4096, (64, 64), False), (65, 65536, 8192, (64, 64), False),
    (128, 65536, 8192, (128, 128), True), (128, 128256, 4096, (128, 128), False), (128, 128256, 4096, (128, 192), True), (129, 65536, 8192, (128, 192), False),
    (160, 28672, 4096, (192, 128), False), (160, 128256, 4096, (192, 128), False)])
def test_weights_past_the_caches_rule(M, N, K, tile, past):
    """Weights pass the caches by where that measured faster: read by one tile of rows, and few rows or not too wide."""
    from llm_weighted_consensus_amd import ops

    assert ops.kernels().gemm2w_past_caches(M, N, K, *tile) == past


@pytest.mark.parametrize("N,K,rows", [
    (4608, 12288, {1: "blas", 7: "blas", 8: "g2", 24: "g2"}), (4736, 11008, {1: "g2", 24: "g2"}), (4160, 13952, {1: "g2"}), (4744, 11264, {1: "g2", 24: "g2"}),
    (4096, 12288, {1: "blas", 16: "blas", 17: "g2"}), (4096, 13824, {16: "blas", 24: "g2"}), (4096, 13952, {1: "g2", 16: "g2"}), (4096, 11072, {1: "g2"}),
    (5120, 13824, {1: "blas", 7: "blas", 8: "g2", 24: "g2"}), (5120, 13312, {1: "g2"}), (4672, 13312, {1: "blas", 8: "g2"}), (4992, 14080, {5: "g2"})])
def test_untuned_down_of_few_rows(N, K, rows):
    """Inside the range of down projections that gemm2w takes: rows, widths and depths at which the library measured faster keep it."""
    assert {M: gemm_plan._untuned(M, N, K, "residual") for M in rows} == rows


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,epi", [(32008, 4096, "plain"), (50304, 2048, "plain"), (4104, 11072, "residual"), (5120, 13824, "residual"), (4096, 11072, "residual"), (4744, 11072, "residual")])
def test_untuned_few_rows_of_wide_and_deep_weights(gpu, N, K, epi):
    """The results of both against fp64 of the same operands (bound: one bf16 rounding, doubled; fp32 sums), rows of another stride and
    a residual off 16 bytes, which the library keeps, among them."""
    g = torch.Generator().manual_seed(K)
    W = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(gpu)
    for M in (1, 5, 16, 17, 24):
        A = torch.randn(M, K + 8, generator=g).to(torch.bfloat16).to(gpu)[:, :K]
        if epi == "plain":
            got, ref = gemm_plan.linear(A, W), A.double() @ W.double().t()
            torch.testing.assert_close(got.double(), ref, rtol=2 ** -8, atol=2e-4)
            continue
        for off in (0, 1):
            C = torch.randn(M * N + off, generator=g).to(torch.bfloat16).to(gpu)[off:].view(M, N)
            ref = A.double() @ W.double().t() + C.double()
            torch.testing.assert_close(gemm_plan.linear_add_(A, W, C).double(), ref, rtol=2 ** -8, atol=2e-4)


@pytest.mark.parametrize("times,core", [
    ({"blas": 100, "g8": 89}, "g8"), ({"blas": 100, "g8": 91}, "blas"), ({"blas": 100, "g8": 101}, "blas"), ({"blas": 100, "g2": 102}, "g2"),
    ({"blas": 100, "g2": 104}, "blas"), ({"blas": 100, "g8": 95, "g2": 102}, "g2"), ({"blas": 100, "g8": 95, "g2": 104}, "blas"),
    ({"blas": 100, "g8": 85, "g2": 95}, "g8"), ({"blas": 100}, "blas")])
def test_encoder_core_of_timings(monkeypatch, times, core):
    """gemm8p needs its lead over every other core, in front of the library as behind it; a tie goes to the other own cores."""
    monkeypatch.setattr(gemm_plan, "TIMINGS", {})
    monkeypatch.setattr(gemm_plan, "_time_between", lambda fn, x: fn())
    assert gemm_plan._pick("key", {n: (lambda v=v: v) for n, v in times.items()}, None) == core
    assert gemm_plan.TIMINGS == {"key": times}


@pytest.mark.parametrize("times,core", [
    ({"blas": 100, "g8": 99}, "g8"), ({"blas": 100, "g8": 92, "g2": 94}, "g8"), ({"blas": 100, "g8": 94, "g2": 92}, "g2"), ({"blas": 100, "g8": 101}, "blas")])
def test_exact_gelu_where_it_is_as_fast(monkeypatch, times, core):
    """The library's GELU is the tanh form: a core with the exact one need not lead to be taken for FFN1, as it must elsewhere."""
    monkeypatch.setattr(gemm_plan, "TIMINGS", {})
    monkeypatch.setattr(gemm_plan, "_time_between", lambda fn, x: fn())
    runs = {n: (lambda v=v: v) for n, v in times.items()}
    assert gemm_plan._pick((8192, 4096, 1024, "bias_gelu"), runs, None) == core
    if times["g8"] > 90 and "g2" not in times:
        assert gemm_plan._pick((8192, 4096, 1024, "bias"), runs, None) == "blas"


@pytest.mark.gpu
@pytest.mark.parametrize("n,most", [(256, 16), (16384, 8)])
def test_encoder_cores_are_timed_in_few_calls(gpu, monkeypatch, n, most):
    """A request waits while the cores of a new size are timed: sixteen calls of each, eight of those that take a millisecond."""
    monkeypatch.setattr(gemm_plan, "TIMINGS", {})
    x, w = torch.ones(n, n, device=gpu, dtype=torch.bfloat16), torch.ones(n, n, device=gpu, dtype=torch.bfloat16)
    made = {"blas": 0, "g2": 0, "g8": 0}

    def call(core):
        made[core] += 1
        x @ w
    assert gemm_plan._pick("key", {c: (lambda c=c: call(c)) for c in made}, x) in made
    assert all(0 < v <= most for v in made.values()) and all(v > 0 for v in gemm_plan.TIMINGS["key"].values())


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rows", [
    (4096, 11008, {384: "blas", 385: "g8", 4096: "blas", 4097: "g8", 4608: "g8", 4609: "blas", 6145: "g8", 7425: "blas"}),
    (3848, 14336, {544: "g8", 7424: "g8", 8193: "g8", 12033: "blas", 13824: "g8", 13825: "blas"}), (3840, 14336, {385: "blas", 4097: "blas"}),
    (2048, 8192, {65: "g2", 128: "g2", 129: "blas"}), (3840, 17472, {100: "g2"}), (3848, 17472, {100: "blas"}), (4104, 8192, {65: "blas"}),
    (2040, 8192, {65: "blas"}), (2048, 8128, {65: "blas"})])
def test_untuned_down_projections(gpu, N, K, rows):
    """Both sides of the rule's lines, and its results against fp64 of the same operands (bound: one bf16 rounding, doubled; fp32 sums)."""
    g = torch.Generator().manual_seed(K)
    W = (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).to(gpu)
    for M, core in rows.items():
        A, C = (torch.randn(M, n, generator=g).to(torch.bfloat16).to(gpu) for n in (K, N))
        if (M, N, K, "residual") not in gemm_plan._CHOICE and (N, K, "residual") not in gemm_plan._BUCKETS and gemm_plan.MODE == "auto":
            assert gemm_plan._backend(A, W, "residual", None, C)[0] == core
        if core == "blas":
            continue
        ref = A.double() @ W.double().t() + C.double()
        torch.testing.assert_close(gemm_plan.linear_add_(A, W, C).double(), ref, rtol=2 ** -8, atol=2e-4)


@pytest.mark.parametrize("room", [True, False])
def test_timings_without_room_say_so(monkeypatch, caplog, room):
    """A shape timed on cached weights, because the buffer that passes them through found no room, is named in the log and table."""
    key = (4, 64, 64, "plain")
    for d in ("_CHOICE", "TIMINGS"):
        monkeypatch.setattr(gemm_plan, d, {})
    monkeypatch.setattr(gemm_plan, "WARM", set())
    monkeypatch.setattr(gemm_plan, "_evict_buffer", lambda device: torch.ones(1) if room else None)
    monkeypatch.setattr(gemm_plan, "_own_ok", lambda *a: False)
    timed = []
    monkeypatch.setattr(gemm_plan, "_time", lambda *a, **kw: timed.append("cached") or 1.0)
    monkeypatch.setattr(gemm_plan, "_time_step", lambda *a, **kw: timed.append("memory") or 1.0)
    with caplog.at_level("WARNING"):
        assert gemm_plan._tune(torch.zeros(4, 64), torch.zeros(64, 64), "plain", 0, None, *key[:3], key) == "blas"
    assert set(timed) == {"memory" if room else "cached"} and bool(caplog.records) == (not room)
    assert (gemm_plan.table()["4x64x64:plain"].get("weights") == "cached") == (not room)


@pytest.mark.gpu
def test_forward_mode_and_vmap_through_untuned_projections(gpu):
    """The tangent of an untuned call (it was lost in silence), and a batch of them under vmap (it raised).  Bound: bf16 results
    of sums of K terms in another order."""
    M, N, K = 8, 4096, 4096
    x, t = (torch.randn(M, K, device=gpu).to(torch.bfloat16) for _ in range(2))
    w = (torch.randn(N, K, device=gpu) * K ** -0.5).to(torch.bfloat16)
    assert gemm_plan._untuned(M, N, K, "plain") != "blas"
    with forward_ad.dual_level():
        y = forward_ad.unpack_dual(gemm_plan.linear(forward_ad.make_dual(x, t), w))
        torch.testing.assert_close(y.tangent, torch.nn.functional.linear(t, w), rtol=2 ** -7, atol=2 ** -7)
    both = torch.vmap(lambda z: gemm_plan.linear(z, w))(torch.stack([x, t]))
    torch.testing.assert_close(both, torch.nn.functional.linear(torch.stack([x, t]), w), rtol=2 ** -7, atol=2 ** -6)
