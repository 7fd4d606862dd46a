"""The fused projections and attention of small decode steps (csrc/kernels/step_fuse.h) against float64.

Bounds: a bf16 output is within 2^-8 of its value (half a unit in the last place is 2^-9, the row scale and SwiGLU's own fp32
arithmetic stay below the other half) plus what fp32 sums in another order leave of the terms' magnitudes (2^-18 of their sum)."""
import pytest
import torch

from llm_weighted_consensus_amd import ops

pytestmark = pytest.mark.gpu
DEV, EPS = "cuda", 1e-5


def _rand(*shape, seed=0, s=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * s).to(torch.bfloat16)


def _partials(x, P):
    return x.float().pow(2).view(x.shape[0], P, -1).sum(-1).contiguous()


def _close(got, ref, mag):
    err = (got.double() - ref).abs()
    assert (err <= ref.abs() * 2.0 ** -8 + mag * 2.0 ** -18 + 1e-30).all(), float((err - ref.abs() * 2.0 ** -8).max())


def _scaled(x, w):
    xd, wd = x.double(), w.double()
    rs = torch.rsqrt(xd.pow(2).mean(1, keepdim=True) + EPS)
    return rs * (xd @ wd.t()), rs * (xd.abs() @ wd.abs().t())


def _ws():
    return ops.new_gemm8p_workspace(torch.device(DEV))


@pytest.mark.parametrize("core", [1, 2])
@pytest.mark.parametrize("M,K,N,P", [(1, 4096, 192, 4), (5, 384, 64, 12), (16, 2048, 128, 128), (17, 256, 6400, 8), (33, 4096, 64, 256),
                                     (63, 1024, 128, 32), (64, 14336, 64, 4)])
def test_row_scaled(core, M, K, N, P):
    x, w = _rand(M, K, seed=1, s=3.0), _rand(N, K, seed=2, s=0.05)
    x[0] *= 2.0 ** -20   # eps counts
    ss = _partials(x, P)
    ref, mag = _scaled(x, w)
    _close(ops.step_project(x, w, core, ss, EPS, ws=_ws()), ref, mag)
    wi = ops.swiglu_interleave(w) if N % 64 == 0 else None
    h = N // 2
    gate, up = ref[:, :h], ref[:, h:]
    act = gate * torch.sigmoid(gate)
    # the gate's own error reaches the product through silu (slope at most 1.1) times up
    _close(ops.step_project(x, wi, core, ss, EPS, swiglu=True, ws=_ws()), act * up,
           1.1 * mag[:, :h] * up.abs() + act.abs() * mag[:, h:] + (act * up).abs())


@pytest.mark.parametrize("core", [1, 2])
@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (7, 512, 128), (17, 14336, 1024), (31, 128, 8192), (64, 1024, 4096)])
def test_residual_leaves_sums_of_squares(core, M, K, N):
    P = ops.step_partials(core, N)
    if not P:
        with pytest.raises(RuntimeError):   # (N / 16 partials of 8192 columns: more than the next projection takes)
            ops.step_project(_rand(M, K), _rand(N, K), core, torch.empty(M, N // 16, device=DEV), EPS, residual=_rand(M, N))
        return
    x, w, r = _rand(M, K, seed=3), _rand(N, K, seed=4, s=0.02), _rand(M, N, seed=5)
    ss = torch.full((M, P), float("nan"), device=DEV)
    ref = r.double() + x.double() @ w.double().t()
    out = ops.step_project(x, w, core, ss, EPS, residual=r, ws=_ws())
    assert out.data_ptr() == r.data_ptr()
    _close(r, ref, r.double().abs() + x.double().abs() @ w.double().abs().t())
    torch.testing.assert_close(ss.double(), _partials(r, P).double(), rtol=1e-5, atol=0)  # (32 fp32 terms)


def test_many_columns_on_weight_streams():
    """Core 2 with more than four units of 16 columns a CU and with two tiles a CU (csrc/kernels/gemm1s.hip): rows scaled in both, and
    sums of squares of pairs of units."""
    test_row_scaled(2, 61, 256, 35328, 8)
    test_row_scaled(2, 64, 512, 22016, 16)
    test_residual_leaves_sums_of_squares(2, 37, 5120, 6144)
    test_qkv_into_the_cache(2, 33, 152, 10, 128, 256)


@pytest.mark.parametrize("core", [1, 2])
@pytest.mark.parametrize("M,Hq,Hkv,D,K", [(1, 32, 8, 128, 4096), (3, 4, 1, 64, 256), (17, 6, 2, 192, 512), (64, 8, 8, 128, 1024)])
def test_qkv_into_the_cache(core, M, Hq, Hkv, D, K):
    NB, BS = 2 * M + 2, 16
    x, w = _rand(M, K, seed=6, s=2.0), _rand((Hq + 2 * Hkv) * D, K, seed=7, s=0.05)
    g = torch.Generator().manual_seed(8)
    slots = torch.randperm(NB * BS, generator=g)[:M].int()
    if M > 1:
        slots[1] = -1   # a padded row
    pos = torch.randint(0, 500, (M,), generator=g).int().to(DEV)
    ang = torch.outer(torch.arange(500.0), 0.01 ** (torch.arange(D // 2) / (D // 2)))
    cos, sin = ang.cos().to(DEV).contiguous(), ang.sin().to(DEV).contiguous()
    kc, vc = _rand(NB, Hkv, BS, D, seed=9), _rand(NB, Hkv, BS // 4, D, 4, seed=10)
    k0, v0 = kc.clone(), vc.clone()
    q = ops.step_qkv(x, w, core, _partials(x, 4), EPS, pos, slots.to(DEV), cos, sin, kc, vc, Hq, ws=_ws())
    ref, mag = _scaled(x, w)
    _close(q, ref[:, :Hq * D], mag[:, :Hq * D])
    k, km = (t[:, Hq * D:(Hq + Hkv) * D].view(M, Hkv, 2, D // 2) for t in (ref, mag))
    v, vm = (t[:, (Hq + Hkv) * D:].view(M, Hkv, D) for t in (ref, mag))
    c, s = cos[pos.long()].double()[:, None], sin[pos.long()].double()[:, None]
    k1 = torch.stack([k[:, :, 0] * c - k[:, :, 1] * s, k[:, :, 1] * c + k[:, :, 0] * s], 2).flatten(2)
    # k is rounded before it is rotated: half a unit of either half besides the sum's own
    km = (km.sum(2, keepdim=True) + k.abs().sum(2, keepdim=True) * 2.0 ** 10).expand(-1, -1, 2, -1).flatten(2)
    for i, sl in enumerate(slots.tolist()):
        if sl < 0:
            continue
        b, o = divmod(sl, BS)
        _close(kc[b, :, o], k1[i], km[i])
        _close(vc[b, :, o // 4, :, o % 4], v[i], vm[i])
        k0[b, :, o], v0[b, :, o // 4, :, o % 4] = kc[b, :, o], vc[b, :, o // 4, :, o % 4]
    assert torch.equal(kc, k0) and torch.equal(vc, v0)   # and nothing else changed


@pytest.mark.parametrize("Hq,Hkv,splits", [(32, 8, 16), (8, 8, 2), (16, 1, 5), (16, 1, 40), (24, 8, 4)])
def test_splits_added_up_in_the_attention(Hq, Hkv, splits):
    ctx = [1, 16, 17, 127, 128, 129, 256, 257, 1000, 2048, 0]
    B, D, BS = len(ctx), 128, 16
    W = max(ctx) // BS + 1
    bt = torch.randperm(B * W, generator=torch.Generator().manual_seed(1)).view(B, W).int().to(DEV)
    kc, vc = _rand(B * W, Hkv, BS, D, seed=2), _rand(B * W, Hkv, BS // 4, D, 4, seed=3)
    q = _rand(B, Hq * D, seed=4)
    cl = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    counts = torch.zeros(B, Hkv, dtype=torch.int32, device=DEV)
    ref = ops.paged_decode(q, kc, vc, bt, cl, Hq, D ** -0.5)
    for _ in range(3):
        out = ops.paged_decode(q, kc, vc, bt, cl, Hq, D ** -0.5, num_splits=splits, counts=counts)
        assert int(counts.abs().sum()) == 0
        # both round softmax weights to bf16 (2^-9 of terms of magnitude 1 whose weighted mean this is) and the result
        assert (out.float() - ref.float()).abs().max() < 2.0 ** -6
    assert torch.equal(out[-1], torch.zeros_like(out[-1]))
    assert torch.equal(out, ops.paged_decode(q, kc, vc, bt, cl, Hq, D ** -0.5, num_splits=splits))  # added up by a second kernel


@pytest.mark.parametrize("T,d,per", [(1, 128, 1), (5, 4096, 8), (64, 768, 0), (3, 8200, 300)])
def test_embedding_step(T, d, per):
    table = _rand(50, d, seed=11)
    ids = torch.tensor([i * 7 % 60 - 2 for i in range(T)], dtype=torch.int32, device=DEV)
    x, ss, counts = ops.embedding_step(table, ids, per)
    assert torch.equal(x, ops.embedding(table, ids)) and counts.shape == (T, per) and int(counts.abs().sum()) == 0
    torch.testing.assert_close(ss.double().sum(1), x.double().pow(2).sum(1), rtol=1e-5, atol=0)
