"""Llama decoder + engine on the GPU: kernel-path forward vs an fp32 PyTorch forward, paged decode
consistency with prefill, prefix-sharing fork/COW, hipGraph replay equivalence."""
import pytest
import torch

from tests import torch_ref as ref

pytestmark = pytest.mark.gpu


def _cos(a, b):
    a, b = a.float().flatten(), b.float().flatten()
    return (a @ b / (a.norm() * b.norm())).item()


@pytest.fixture(scope="module")
def tiny(gpu):
    from llm_weighted_consensus_amd.models.config import decoder_config
    from llm_weighted_consensus_amd.models.llama import LlamaModel

    return LlamaModel(decoder_config("llama-tiny"), device=gpu, seed=0, max_position=1024)


def test_prefill_and_decode_match_reference(tiny, gpu):
    from llm_weighted_consensus_amd.models.llama import KVCache

    m = tiny
    cache = KVCache(m.cfg, 64, 16, gpu)
    g = torch.Generator(device="cpu").manual_seed(0)
    toks = torch.randint(0, m.cfg.vocab_size, (40,), generator=g).to(gpu)
    ref_logits = ref.llama_forward(m, toks)  # [40, V]
    # prefill the first 33 tokens into blocks 0..2, then decode 7 tokens one by one
    P = 33
    slots = torch.arange(P, dtype=torch.int32, device=gpu)
    cu = torch.tensor([0, P], dtype=torch.int32, device=gpu)
    lg = m.prefill(toks[:P].int(), torch.arange(P, dtype=torch.int32, device=gpu), slots, cu, P,
                   torch.tensor([P - 1], device=gpu), cache)
    assert _cos(lg[0], ref_logits[P - 1]) > 0.995
    bt = torch.arange(4, dtype=torch.int32, device=gpu).view(1, 4)
    for t in range(P, 40):
        dl = m.decode(toks[t:t + 1].int(), torch.tensor([t], dtype=torch.int32, device=gpu),
                      torch.tensor([t], dtype=torch.int32, device=gpu), bt,
                      torch.tensor([t + 1], dtype=torch.int32, device=gpu), cache, num_splits=2)
        assert _cos(dl[0], ref_logits[t]) > 0.995, t


@pytest.mark.parametrize("step_ab", ["0", "1"])
def test_engine_greedy_graph_equivalence_and_fork(tiny, gpu, step_ab, monkeypatch):
    """Graph replay == eager decode, greedy.  With the in-step A/B on (engine._step_ab), the graph engine runs
    first: its A/B installs the winning plan in the model, which the eager engine then runs too."""
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer

    monkeypatch.setenv("LWC_STEP_AB", step_ab)
    monkeypatch.setenv("LWC_STEP_AB_MIN", "1")  # the tiny model's buckets are small
    tok = ByteTokenizer(tiny.cfg.vocab_size)
    prompts = [tok.encode("hello world, this is a prompt of some length " * 2), tok.encode("short")]
    sp = SamplingParams(temperature=0.0, max_tokens=24, ignore_eos=True)
    outs = []
    for graphs in ((True, False) if step_ab == "1" else (False, True)):
        eng = LLMEngine(tiny, tok, num_blocks=256, max_batch=16, max_model_len=512, use_graphs=graphs)
        outs.append(eng.generate(prompts, sp, n=3))
        assert eng.bm.num_free == 256  # everything released
    assert outs[0] == outs[1]
    for group in outs[0]:
        assert all(c == group[0] for c in group)  # greedy children of one prompt agree
        assert all(len(c) == 24 for c in group)
    # greedy engine output == greedy over the fp32 reference forward (first tokens; bf16 drift later)
    p = torch.tensor(prompts[0], device=gpu)
    first = int(ref.llama_forward(tiny, p)[-1].argmax())
    assert outs[0][0][0][0] == first


def test_engine_prefix_sharing_equivalence(tiny, gpu):
    """The cascade (prefix-shared) attention path gives the same greedy continuations."""
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer

    tok = ByteTokenizer(tiny.cfg.vocab_size)
    prompts = [tok.encode("x" * 70 + " a shared prompt longer than a few KV blocks"), tok.encode("y" * 33)]
    sp = SamplingParams(temperature=0.0, max_tokens=12, ignore_eos=True)
    outs = []
    for share in (False, True):
        eng = LLMEngine(tiny, tok, num_blocks=256, max_batch=16, max_model_len=512, prefix_sharing=share)
        outs.append(eng.generate(prompts, sp, n=5))
    same = sum(a == b for ga, gb in zip(*outs) for ca, cb in zip(ga, gb) for a, b in zip(ca, cb))
    total = sum(len(c) for g in outs[0] for c in g)
    assert same >= 0.95 * total, (same, total)


def test_engine_sampling_seeded(tiny, gpu):
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer

    tok = ByteTokenizer(tiny.cfg.vocab_size)
    eng = LLMEngine(tiny, tok, num_blocks=256, max_batch=32, max_model_len=512)
    sp = SamplingParams(temperature=1.0, top_p=0.9, max_tokens=16, ignore_eos=True, seed=1234, top_logprobs=5,
                        logprobs=True)
    a = eng.generate([tok.encode("abc")], sp, n=4)
    b = eng.generate([tok.encode("abc")], sp, n=4)
    assert a == b
    assert len({tuple(x) for x in a[0]}) > 1  # different children sample differently


def test_engine_export_import_prefill_equivalence(tiny, gpu):
    """Candidate-parallel path: a prompt prefilled by export_prefill and started via add_request(prefilled=)
    samples exactly what the engine's own prefill path samples (same seeds)."""
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer
    from llm_weighted_consensus_amd.parallel.prefill_share import all_gather_prefills

    tok = ByteTokenizer(tiny.cfg.vocab_size)
    prompts = [tok.encode("z" * 40 + " exported prompt"), tok.encode("q" * 16)]  # partial + exact block
    sp = SamplingParams(temperature=0.9, top_p=0.9, max_tokens=10, ignore_eos=True, seed=77)
    a = LLMEngine(tiny, tok, num_blocks=256, max_batch=16, max_model_len=512)
    want = a.generate(prompts, sp, n=3)
    b = LLMEngine(tiny, tok, num_blocks=256, max_batch=16, max_model_len=512)
    kv, lg, nbl = b.export_prefill(prompts)
    assert b.bm.num_free == 256 and kv.shape[2] == sum(nbl) and len(nbl) == 2
    shared = all_gather_prefills(kv, lg, nbl)  # single process: plain split
    groups = [b.add_request(p, sp, n=3, prefilled=shared[i]) for i, p in enumerate(prompts)]
    while b.has_work():
        b.step()
    got = [[list(s.tokens) for s in g.seqs] for g in groups]
    assert got == want
    assert b.bm.num_free == 256


@pytest.mark.parametrize("fused", ["0", "ffn2", "all"])
def test_encoder_layers_on_gemm8p_launched_natively(gpu, monkeypatch, fused):
    """Projections on gemm8p are launched from native code too, over the stream's workspace: the loop's bits."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.bert import BertEncoder
    from llm_weighted_consensus_amd.models.config import encoder_config
    from llm_weighted_consensus_amd.ops import gemm_plan

    m = BertEncoder(encoder_config("bge-small-en-v1.5"), device=gpu, seed=5)
    m.fused_residual = fused
    args = m.pack([[(7 * i + j) % 900 + 1 for j in range(n)] for i, n in enumerate([300, 2, 64, 129])])
    monkeypatch.setattr(gemm_plan, "MODE", "g8")
    taken, native = [], ops.encoder_layers
    monkeypatch.setattr(ops, "encoder_layers", lambda *a: taken.append(native(*a)) or taken[-1])
    y = m.forward_packed(*args)
    assert len(taken) == 1 and taken[0] is not None
    monkeypatch.setattr(ops, "encoder_layers", lambda *a: None)
    assert torch.equal(y, m.forward_packed(*args))


@pytest.mark.parametrize("fused", ["0", "ffn2", "all"])
@pytest.mark.parametrize("cores", [["blas"] * 4, ["blas", "g2", "g8", "blas"], ["g2", "blas", "blas", "g8"]])
def test_encoder_layers_with_the_library_launched_natively(gpu, monkeypatch, cores, fused):
    """Layers with projections on the library are launched from native code as well: the loop's bits, eagerly and as a graph; a
    weight that asks for a gradient leaves them to the loop."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.bert import BertEncoder
    from llm_weighted_consensus_amd.models.config import encoder_config
    from llm_weighted_consensus_amd.ops import gemm_plan

    m = BertEncoder(encoder_config("bge-small-en-v1.5"), device=gpu, seed=5)
    for L in m.layers:
        for n in ("bqkv", "bo", "b1", "b2"):
            getattr(L, n).normal_(0.0, 0.1)
    m.fused_residual = fused
    args = m.pack([[(7 * i + j) % 900 + 1 for j in range(n)] for i, n in enumerate([300, 2, 64, 129])])
    L, T = m.layers[0], args[0].shape[0]
    epis = ("bias", "enc_residual" if fused == "all" else "bias", "bias_gelu", "bias" if fused == "0" else "enc_residual")
    monkeypatch.setattr(gemm_plan, "_CHOICE", {(gemm_plan._m_bucket(T), *w.shape, e): c
                                               for w, e, c in zip((L.wqkv, L.wo, L.w1, L.w2), epis, cores)})
    taken, native = [], ops.encoder_layers_mixed
    monkeypatch.setattr(ops, "encoder_layers_mixed", lambda *a: taken.append(native(*a)) or taken[-1])
    y = m.forward_packed(*args)
    assert len(taken) == 1 and taken[0] is y
    if "g8" not in cores:   # (the capture's stream has no workspace)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            z = m.forward_packed(*args)
        for _ in range(3):
            graph.replay()
            assert torch.equal(y, z)
            m.forward_packed(*args)
    monkeypatch.setattr(ops, "encoder_layers_mixed", lambda *a: None)
    assert torch.equal(y, m.forward_packed(*args))
    monkeypatch.setattr(ops, "encoder_layers_mixed", native)
    m.layers[2].wo.requires_grad_(True)
    assert native(torch.zeros_like(y), [t for L in m.layers for t in (L.wqkv, L.bqkv, L.wo, L.bo, L.ln1_g, L.ln1_b, L.w1, L.b1, L.w2, L.b2,
                                                                     L.ln2_g, L.ln2_b)], args[2], 300, 12, 32, m.scale, 1e-12, [0] * 4,
                  False, False) is None


@pytest.mark.parametrize("how", ["dual weight", "dual bias", "mode", "subclass"])
def test_encoder_layers_with_the_library_stay_visible(gpu, monkeypatch, how):
    """Layers with projections on the library run call by call where forward-mode duals, a dispatch mode or a subclass
    would see those calls (out= forms refuse duals), and give the same bits."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode

    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.bert import BertEncoder
    from llm_weighted_consensus_amd.models.config import encoder_config
    from llm_weighted_consensus_amd.ops import gemm_plan

    m = BertEncoder(encoder_config("bge-small-en-v1.5"), device=gpu, seed=5)
    args = m.pack([[(7 * i + j) % 900 + 1 for j in range(n)] for i, n in enumerate([64, 29])])
    monkeypatch.setattr(gemm_plan, "MODE", "blas")
    taken, native = [], ops.encoder_layers_mixed
    monkeypatch.setattr(ops, "encoder_layers_mixed", lambda *a: taken.append(native(*a)) or taken[-1])
    want = m.forward_packed(*args)
    assert taken.pop() is want
    L, calls = m.layers[3], []

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), kw=None):
            calls.append(func.name())
            return func(*a, **(kw or {}))

    class Other(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, a=(), kw=None):
            calls.append(func.__name__)
            with torch._C.DisableTorchFunctionSubclass():
                return func(*a, **(kw or {}))

    if how == "mode":
        with Seen():
            got = m.forward_packed(*args)
        assert calls.count("aten::addmm") >= 24
    elif how == "subclass":
        L.wo = L.wo.as_subclass(Other)
        got = m.forward_packed(*args)
        assert "linear" in calls
    else:
        with forward_ad.dual_level():
            n = "wo" if how == "dual weight" else "bo"
            monkeypatch.setattr(L, n, forward_ad.make_dual(getattr(L, n), torch.ones_like(getattr(L, n))))
            got = forward_ad.unpack_dual(m.forward_packed(*args)).primal
    assert taken == [None] and torch.equal(got, want)


@pytest.mark.parametrize("core", [0, 4, -1])
def test_encoder_layers_refuse_other_cores(gpu, core):
    """A core that no kernel stands for is an error, not gemm2w."""
    from llm_weighted_consensus_amd import ops

    d, f = 64, 256
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=gpu)  # noqa: E731
    weights = [z(3 * d, d), z(3 * d), z(d, d), z(d), z(d), z(d), z(f, d), z(f), z(d, f), z(d), z(d), z(d)]
    cu = torch.tensor([0, 5], dtype=torch.int32, device=gpu)
    assert ops.encoder_layers(z(5, d), weights, cu, 5, 2, 32, 0.2, 1e-6, [2, 2, 2, 3], False, False).shape == (5, d)
    with pytest.raises(RuntimeError, match="cores are 1 to 3"):
        ops.encoder_layers(z(5, d), weights, cu, 5, 2, 32, 0.2, 1e-6, [2, core, 2, 2], False, False)


@pytest.mark.parametrize("down,choices", [(150, ["g2", "g2", "g2", "g2"]),       # all native: the ties keep their cores
                                          (90, ["blas", "g2", "g2", "blas"])])    # the library for one: what is faster than it, and the exact GELU
def test_encoder_ties_go_to_native_layers_alone(gpu, monkeypatch, down, choices):
    """A core that is no faster than the library is taken where the whole layer is launched from native code, and nowhere else; all are
    chosen before the first projection runs, so that the first pass gives the later ones' bits."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.bert import BertEncoder
    from llm_weighted_consensus_amd.models.config import encoder_config
    from llm_weighted_consensus_amd.ops import gemm_plan

    m = BertEncoder(encoder_config("bge-small-en-v1.5"), device=gpu, seed=5)
    m.fused_residual = "ffn2"
    args = m.pack([[(7 * i + j) % 900 + 1 for j in range(n)] for i, n in enumerate([300, 2, 64, 129])])
    for d in ("_CHOICE", "TIMINGS"):
        monkeypatch.setattr(gemm_plan, d, {})
    blas = {1152: 100, 384: 120, 1536: 100}
    picked = gemm_plan._pick

    def pick(key, runs, x):
        lib = down if key[3] == "enc_residual" else blas[key[1]]
        for f in runs.values():
            f()
        times = {n: lambda: 102 for n in runs} | {"blas": lambda: lib}
        return picked(key, times, x)
    monkeypatch.setattr(gemm_plan, "_pick", pick)
    monkeypatch.setattr(gemm_plan, "_time_between", lambda fn, x: fn())
    monkeypatch.setattr(gemm_plan, "EXCLUDE", gemm_plan.EXCLUDE | {"g8", "gv"})
    native, run = [], ops.encoder_layers
    monkeypatch.setattr(ops, "encoder_layers", lambda *a: native.append(1) or run(*a))
    first = m.forward_packed(*args)
    L = m.layers[0]
    got = [gemm_plan._CHOICE[(gemm_plan._m_bucket(args[0].shape[0]), *w.shape, e)]
           for w, e in ((L.wqkv, "bias"), (L.wo, "bias"), (L.w1, "bias_gelu"), (L.w2, "enc_residual"))]
    assert got == choices and len(native) == (down == 150)
    assert torch.equal(first, m.forward_packed(*args))


@pytest.mark.parametrize("core,lens", [("gv", [5, 1, 40]), ("g2", [5, 1, 40]), ("g2", [300, 2, 64, 129])])
@pytest.mark.parametrize("fused", ["0", "ffn2", "all"])
def test_encoder_layers_launched_natively(gpu, monkeypatch, core, lens, fused):
    """The natively launched layers run the loop's kernels: the same bits, and the loop itself where a weight lies at an odd
    address or a projection has another core."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.bert import BertEncoder
    from llm_weighted_consensus_amd.models.config import encoder_config
    from llm_weighted_consensus_amd.ops import gemm_plan

    m = BertEncoder(encoder_config("bge-small-en-v1.5"), device=gpu, seed=5)
    m.fused_residual = fused
    args = m.pack([[(7 * i + j) % 900 + 1 for j in range(n)] for i, n in enumerate(lens)])
    monkeypatch.setattr(gemm_plan, "MODE", core)
    taken, native = [], ops.encoder_layers
    monkeypatch.setattr(ops, "encoder_layers", lambda *a: taken.append(native(*a)) or taken[-1])
    y = m.forward_packed(*args)
    assert len(taken) == 1 and taken[0] is not None
    monkeypatch.setattr(ops, "encoder_layers", lambda *a: None)
    assert torch.equal(y, m.forward_packed(*args))
    monkeypatch.setattr(ops, "encoder_layers", lambda *a: taken.append(native(*a)) or taken[-1])
    w = m.layers[1].w2
    m.layers[1].w2 = torch.cat([w.flatten()[:1], w.flatten()])[1:].view(w.shape)   # two bytes off
    if core == "gv":
        torch.testing.assert_close(y, m.forward_packed(*args))
    else:
        assert torch.isfinite(m.forward_packed(*args).float()).all()
    assert len(taken) == 2 and taken[1] is None
    m.layers[1].w2 = w
    monkeypatch.setattr(gemm_plan, "MODE", "blas")
    m.forward_packed(*args)
    assert len(taken) == 2


@pytest.mark.parametrize("fused", ["ffn2", "all", "0"])
@pytest.mark.parametrize("arch", ["bge-small-en-v1.5", "bert-tiny"])
def test_bert_encoder_matches_reference(gpu, arch, fused):
    """HIP encoder (LN, varlen bidirectional attention incl. head_dim 32, bias+GELU, pooling) vs the
    fp32 PyTorch reference forward of the same weights; ``fused``: which of o / FFN2 add into the residual stream
    in their GEMM epilogue, the LayerNorm then taking their bias (default "ffn2"), else projection + LN(x + r)."""
    from llm_weighted_consensus_amd.models.bert import BertEncoder
    from llm_weighted_consensus_amd.models.config import encoder_config

    m = BertEncoder(encoder_config(arch), device=gpu, seed=5)
    m.fused_residual = fused
    lists = [[101] + list(range(1000, 1000 + n)) + [102] for n in (3, 40, 77, 130)]
    ids, pos, cu, max_len = m.pack(lists)
    h = m.forward_packed(ids, pos, cu, max_len)
    ref = m.forward_reference(ids, pos, cu)
    for i in range(len(lists)):
        s0, s1 = int(cu[i]), int(cu[i + 1])
        assert _cos(h[s0:s1], ref[s0:s1]) > 0.995, (arch, i)
    e, _ = m.embed_packed(ids, pos, cu, max_len)
    er = BertEncoder.pool_reference(ref, cu, m.cfg.pooling)
    assert (e - er).abs().max().item() < 2e-2


@pytest.mark.parametrize("fp8", [False, True])
def test_mixtral_moe_matches_reference_and_engine(gpu, fp8):
    """Mixtral MoE decoder (router top-2, grouped MFMA expert GEMMs, combine; fp8 experts) vs the fp32
    reference, then greedy generation through the engine (cascade + graphs) with prefill/decode agreeing."""
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer
    from llm_weighted_consensus_amd.models.config import decoder_config
    from llm_weighted_consensus_amd.models.llama import KVCache
    from llm_weighted_consensus_amd.models.mixtral import MixtralModel

    m = MixtralModel(decoder_config("mixtral-tiny"), device=gpu, seed=2, max_position=1024, fp8=fp8)
    g = torch.Generator(device="cpu").manual_seed(1)
    toks = torch.randint(0, m.cfg.vocab_size, (37,), generator=g).to(gpu)
    ref_logits = ref.llama_forward(m, toks)
    cache = KVCache(m.cfg, 16, 16, gpu)
    P = 37
    lg = m.prefill(toks.int(), torch.arange(P, dtype=torch.int32, device=gpu), torch.arange(P, dtype=torch.int32,
                   device=gpu), torch.tensor([0, P], dtype=torch.int32, device=gpu), P,
                   torch.tensor([P - 1], device=gpu), cache)
    # measured 0.99999 (bf16) / 0.9990 (fp8) over seeds 2-4 (scripts/mixtral_cos_probe.py); the bounds leave room
    # for a near-tie router flip.  (They were 0.99 / 0.985 while the router's softmax was wrong — README.)
    assert _cos(lg[0], ref_logits[P - 1]) > (0.998 if fp8 else 0.999)
    tok = ByteTokenizer(m.cfg.vocab_size)
    eng = LLMEngine(m, tok, num_blocks=1024, max_batch=160, max_model_len=512, cascade_min_batch=1)
    sp = SamplingParams(temperature=0.0, max_tokens=8, ignore_eos=True)
    outs = eng.generate([tok.encode("mixture of experts " * 3)], sp, n=130)
    assert all(o == outs[0][0] for o in outs[0])  # greedy children agree (cascade tiles > 1 per group)
    assert eng.bm.num_free == 1024


def test_decoder_embedder_last_token(tiny, gpu):
    """e5-mistral-style embedder: cache-less encode == the fp32 reference forward's final normed state of the
    last token (pooled, unit norm), independent of batch packing."""
    from llm_weighted_consensus_amd.models.embedder import DecoderEmbedder

    emb = DecoderEmbedder(tiny)
    lists = [[5, 6, 7, 8, 9] * 7, [11, 12, 13], list(range(100, 190))]
    e, _ = emb.embed(lists)
    assert torch.allclose(e.norm(dim=-1), torch.ones(3, device=gpu), atol=1e-3)
    for i, tl in enumerate(lists):
        t = torch.tensor(tl, device=gpu)
        cfg = tiny.cfg
        # reference: hidden state before lm_head = rmsnorm(x) at the last position
        x = ref.llama_hidden(tiny, t)[-1]
        r = torch.nn.functional.normalize(x, dim=0)
        assert _cos(e[i], r) > 0.995
        solo, _ = emb.embed([tl])
        assert _cos(solo[0], e[i]) > 0.999


def test_prefill_with_cached_prefix_matches_full_prefill(tiny, gpu):
    """Cross-request prefix cache at the model level: prefilling only a prompt's tail on top of its cached
    head blocks (key ranges gathered from the paged cache) gives the full prefill's last-token logits."""
    import numpy as np

    from llm_weighted_consensus_amd.models.llama import KVCache

    m = tiny
    cache = KVCache(m.cfg, 64, 16, gpu)
    g = torch.Generator(device="cpu").manual_seed(3)
    P, C = 53, 32  # 2 cached blocks, 21 new tokens
    toks = torch.randint(0, m.cfg.vocab_size, (P,), generator=g).to(gpu).int()
    ar = torch.arange(P, dtype=torch.int32, device=gpu)
    full = m.prefill(toks, ar, ar, torch.tensor([0, P], dtype=torch.int32, device=gpu), P,
                     torch.tensor([P - 1], device=gpu), cache)
    # second sequence: blocks 0,1 shared with the first, tail in blocks 8.. (slots 128..)
    slots_tail = torch.arange(128, 128 + P - C, dtype=torch.int32, device=gpu)
    k_slots = torch.cat([torch.arange(C, device=gpu), slots_tail.long()])
    ctx = {"k_slots": k_slots, "cu_k": torch.tensor([0, P], dtype=torch.int32, device=gpu),
           "q_lens": [P - C], "k_lens": [P]}
    part = m.prefill(toks[C:], ar[C:], slots_tail, torch.tensor([0, P - C], dtype=torch.int32, device=gpu), P - C,
                     torch.tensor([P - C - 1], device=gpu), cache, ctx=ctx)
    assert _cos(part[0], full[0]) > 0.999


def test_engine_prefix_cache_reuses_blocks_across_requests(tiny, gpu):
    """Two requests sharing a long prompt head: with the prefix cache the second prefills only its tail,
    yet greedy continuations equal the uncached engine's."""
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer

    tok = ByteTokenizer(tiny.cfg.vocab_size)
    head = "system: select the response among the choices below. " * 3
    p1, p2 = tok.encode(head + "voter one keys A B"), tok.encode(head + "voter two keys Q R T")
    sp = SamplingParams(temperature=0.0, max_tokens=10, ignore_eos=True)
    outs = []
    for cache_on in (False, True):
        eng = LLMEngine(tiny, tok, num_blocks=256, max_batch=16, max_model_len=512, prefix_caching=cache_on)
        a = eng.generate([p1], sp, n=2)
        b = eng.generate([p2], sp, n=2)
        outs.append((a, b))
        if cache_on:
            assert eng.stats["prefix_cache_tokens"] >= (len(tok.encode(head)) // 16 - 1) * 16
            assert eng.bm.num_free == 256  # cached blocks are evictable capacity
            assert eng.bm.num_cached_blocks > 0
        else:
            assert eng.stats["prefix_cache_tokens"] == 0
    assert outs[0] == outs[1]


def test_engine_prefix_cache_shares_heads_within_one_batch(tiny, gpu):
    """Voters of one score request arrive together: the shared head is computed once (wave 1) and the
    other prompts take it from the cache (wave 2), with unchanged greedy output."""
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer

    tok = ByteTokenizer(tiny.cfg.vocab_size)
    head = "user: which answer is right? " * 4
    prompts = [tok.encode(head + f"system: keys {k}") for k in ("A B", "C D E", "F G", "H")]
    sp = SamplingParams(temperature=0.0, max_tokens=8, ignore_eos=True)
    outs, stats = [], []
    for cache_on in (False, True):
        eng = LLMEngine(tiny, tok, num_blocks=256, max_batch=16, max_model_len=512, prefix_caching=cache_on)
        outs.append(eng.generate(prompts, sp, n=1))
        stats.append(dict(eng.stats))
    assert outs[0] == outs[1]
    saved = stats[0]["prefill_tokens"] - stats[1]["prefill_tokens"]
    assert saved == stats[1]["prefix_cache_tokens"] >= 3 * 96


def test_fp8_dense_decoder_embedder_and_prefill(gpu):
    """fp8 dense projections (config 5's e5-mistral embedder; e4m3 weights with per-channel scales, row-
    quantised activations into the fp8 library GEMM): embeddings and prefill logits track the fp32
    reference of the dequantised weights; the engine decodes with them (graphs on)."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.engine.engine import LLMEngine
    from llm_weighted_consensus_amd.engine.sampling import SamplingParams
    from llm_weighted_consensus_amd.engine.tokenizer import ByteTokenizer
    from llm_weighted_consensus_amd.models.config import decoder_config
    from llm_weighted_consensus_amd.models.embedder import DecoderEmbedder
    from llm_weighted_consensus_amd.models.llama import LlamaModel

    m = LlamaModel(decoder_config("llama-tiny"), device=gpu, seed=3, max_position=1024, fp8_dense=True)
    assert isinstance(m.layers[0].wqkv, ops.Fp8Weight) and not m._dense_residual
    lists = [list(range(40, 100)), [7, 8, 9, 10]]
    e, _ = DecoderEmbedder(m).embed(lists)
    for i, tl in enumerate(lists):
        r = torch.nn.functional.normalize(ref.llama_hidden(m, torch.tensor(tl, device=gpu))[-1], dim=0)
        assert _cos(e[i], r) > 0.99
    tok = ByteTokenizer(m.cfg.vocab_size)
    eng = LLMEngine(m, tok, num_blocks=256, max_batch=16, max_model_len=512)
    out = eng.generate([tok.encode("fp8 projections " * 4)], SamplingParams(temperature=0.0, max_tokens=6,
                                                                          ignore_eos=True), n=2)
    assert len(out[0]) == 2 and out[0][0] == out[0][1] and len(out[0][0]) == 6


@pytest.mark.parametrize("qkv_bn", [192, 256])
def test_folded_norm_chain_matches_unfolded(tiny, gpu, qkv_bn):
    """Folded RMSNorm decode chain (models/llama.py, gemm4w RS modes): the norm weights live in the projection
    weights (the model's norms are ones), the o / down residual epilogues emit the row scales the next
    projection applies — the decode logits equal the unfolded path's (norm kernels + projections) and the fp32
    reference forward.  qkv_bn 192: both producers gemm4w RS 2 (schedules 32 / 64); 256: the down
    producer by rms_rowsumsq after the planner's residual GEMM."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.llama import KVCache

    if not ops.GEMM4W:
        pytest.skip("gemm4w is switched off: a GPU fault of unknown cause in the first headline run with its rewritten main loop")
    m = tiny
    assert m.norm_folded and bool((m.layers[0].attn_norm == 1).all())
    cache = KVCache(m.cfg, 64, 16, gpu)
    g = torch.Generator(device="cpu").manual_seed(3)
    toks = torch.randint(0, m.cfg.vocab_size, (36,), generator=g).to(gpu)
    ref_logits = ref.llama_forward(m, toks)
    P = 35
    slots = torch.arange(P, dtype=torch.int32, device=gpu)
    cu = torch.tensor([0, P], dtype=torch.int32, device=gpu)
    m.prefill(toks[:P].int(), torch.arange(P, dtype=torch.int32, device=gpu), slots, cu, P,
              torch.tensor([P - 1], device=gpu), cache)
    B = 300  # rows: one sequence repeated (ragged last m-tile of the chain's 256-row tiles)
    bt = torch.arange(4, dtype=torch.int32, device=gpu).view(1, 4).expand(B, 4).contiguous()
    args = (toks[P:P + 1].int().expand(B).contiguous(), torch.full((B,), P, dtype=torch.int32, device=gpu),
            torch.full((B,), P, dtype=torch.int32, device=gpu), bt, torch.full((B,), P + 1, dtype=torch.int32,
                                                                                 device=gpu), cache)
    if m.chain is None:
        m.chain = ops.NormChain(8192, m.cfg.hidden, m.cfg.rms_eps, gpu)
    saved = dict(m.chain_m)
    try:
        m.chain_m[B] = {"attn": False, "mlp": False, "final": False, "qkv_bn": qkv_bn, "o": "plain", "down": "plain"}
        assert not m.chain_ok(B)
        base = m.decode(*args, num_splits=1).float()
        m.chain_m[B] = {"attn": True, "mlp": True, "final": True, "qkv_bn": qkv_bn,
                        "o": "own64" if qkv_bn == 256 else "own32", "down": "sumsq" if qkv_bn == 256 else "own64"}
        assert m.chain_ok(B)
        got = m.decode(*args, num_splits=1).float()
    finally:
        m.chain_m.clear()
        m.chain_m.update(saved)
    assert _cos(got, base) > 0.9995
    assert (got - base).abs().max() < 0.05 * base.abs().max()
    assert _cos(got[B - 1], ref_logits[P]) > 0.995 and _cos(got[0], ref_logits[P]) > 0.995


def test_folded_norms_keep_encode_and_logits_with_real_norm_weights(gpu):
    """Norm folding with NON-unit norm weights (random init has unit ones, which hide a dropped weight): the
    folded model's prefill logits and its encode() hidden states (the decoder-as-embedder output, which has
    no lm_head to carry the final norm weight) equal the unfolded model's."""
    from llm_weighted_consensus_amd.models.config import decoder_config
    from llm_weighted_consensus_amd.models.llama import KVCache, LlamaModel

    cfg = decoder_config("llama-tiny")
    gen = torch.Generator(device="cpu").manual_seed(11)

    def norm():
        return (0.5 + torch.rand(cfg.hidden, generator=gen)).to(gpu, torch.bfloat16)

    norms = [(norm(), norm()) for _ in range(cfg.layers)]
    final = norm()
    models = []
    for fold in (False, True):
        m = LlamaModel(cfg, device=gpu, seed=5, max_position=512, fold_norms=False)
        for L, (na, nm) in zip(m.layers, norms):
            L.attn_norm, L.mlp_norm = na.clone(), nm.clone()
        m.final_norm = final.clone()
        if fold:
            m._fold_norms()
            assert m.norm_folded and bool((m.final_norm == 1).all())
        models.append(m)
    a, b = models
    P = 29
    toks = torch.randint(0, cfg.vocab_size, (P,), generator=gen).to(gpu).int()
    pos = torch.arange(P, dtype=torch.int32, device=gpu)
    cu = torch.tensor([0, P], dtype=torch.int32, device=gpu)
    ea = a.encode(toks, pos, cu, P).float()
    eb = b.encode(toks, pos, cu, P).float()
    assert _cos(ea, eb) > 0.9995 and (ea - eb).abs().max() < 0.05 * ea.abs().max()
    last = torch.tensor([P - 1], device=gpu)
    la = a.prefill(toks, pos, pos, cu, P, last, KVCache(cfg, 16, 16, gpu)).float()
    lb = b.prefill(toks, pos, pos, cu, P, last, KVCache(cfg, 16, 16, gpu)).float()
    assert _cos(la, lb) > 0.9995


@pytest.mark.parametrize("arch", ["bge-small-en-v1.5", "bge-base-en-v1.5", "bge-large-en-v1.5"])
@pytest.mark.parametrize("lens", [[1], [12], [16], [17], [32], [5, 1, 9], [3, 13, 1, 15], [1] * 32])
def test_few_row_encoder_matches_reference(gpu, monkeypatch, arch, lens):
    """The encoder's kernels for few rows at the edges of their row tiles and of texts within them, against the fp32 layers:
    no further off than the general kernels are, but for the spread of two roundings (2 x).  A weight at an odd address is
    left to the general ones."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models import bert
    from llm_weighted_consensus_amd.models.config import encoder_config

    m = bert.BertEncoder(encoder_config(arch), device=gpu, seed=5)
    for L in m.layers:   # biases and gains that matter
        for n in ("bqkv", "bo", "b1", "b2", "ln1_b", "ln2_b"):
            getattr(L, n).normal_(0.0, 0.1)
        L.ln1_g.normal_(1.0, 0.1)
        L.ln2_g.normal_(1.0, 0.1)
    args = m.pack([[(37 * i + 11 * j) % 900 + 1 for j in range(n)] for i, n in enumerate(lens)])
    taken, few = [], ops.encoder_few
    monkeypatch.setattr(ops, "encoder_few", lambda *a: taken.append(few(*a)) or taken[-1])
    y = m.forward_packed(*args)
    assert len(taken) == 1 and taken[0] is y
    monkeypatch.undo()
    ref = m.forward_reference(*args[:3])
    monkeypatch.setattr(bert, "FEW_ROWS", 0)
    plain = m.forward_packed(*args)
    err = lambda t: ((t.float() - ref).norm() / ref.norm()).item()  # noqa: E731
    assert err(y) < 2 * err(plain) and err(y) < 0.03, (err(y), err(plain))
    monkeypatch.setattr(bert, "FEW_ROWS", 32)
    w = m.layers[-1].w2
    m.layers[-1].w2 = torch.cat([w.flatten()[:1], w.flatten()])[1:].view(w.shape)   # two bytes off
    assert ops.encoder_few(m.word, m.pos_type, args[0], args[1], m.emb_ln_g, m.emb_ln_b,
                           [t for L in m.layers for t in bert._layer_tensors(L)], args[2], m.cfg.heads, m.scale, 1e-12) is None


@pytest.mark.parametrize("arch", ["bge-small-en-v1.5", "bge-base-en-v1.5"])
@pytest.mark.parametrize("lens", [[5, 4, 6], [12, 17, 3]])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_few_row_encoder_keeps_infinities_to_their_text(gpu, monkeypatch, arch, lens, value):
    """A text with a token whose embedding is not finite changes no other text of its batch, as with the general kernels: the
    others' rows are what they are beside an ordinary token, but for the order of the attention's sums (bf16 layers: 0.01)."""
    from llm_weighted_consensus_amd.models import bert
    from llm_weighted_consensus_amd.models.config import encoder_config

    m = bert.BertEncoder(encoder_config(arch), device=gpu, seed=5)
    texts = [[(37 * i + 11 * j) % 900 + 1 for j in range(n)] for i, n in enumerate(lens)]
    args = m.pack(texts)
    want = m.forward_packed(*args).float()
    texts[1][1] = 29999
    m.word[29999] = value
    bad = slice(lens[0], lens[0] + lens[1])
    for few in (32, 0):
        monkeypatch.setattr(bert, "FEW_ROWS", few)
        got = m.forward_packed(*m.pack(texts)).float()
        assert not torch.isfinite(got[bad]).any()
        for rows in (slice(0, lens[0]), slice(lens[0] + lens[1], None)):
            assert torch.isfinite(got[rows]).all() and (got[rows] - want[rows]).norm() < 0.02 * want[rows].norm(), few


@pytest.mark.parametrize("arch,n", [("bge-small-en-v1.5", 14), ("bge-small-en-v1.5", 32), ("bge-base-en-v1.5", 9), ("bge-large-en-v1.5", 20)])
def test_few_row_encoder_hands_on_what_this_call_made(gpu, arch, n):
    """One launch holds the whole stack and its stages hand rows to each other through scratch memory that the next call gets
    again: calls on other inputs, one after the other, on two streams at once and as a graph that is replayed on them, all
    give the bits of a call by itself."""
    from llm_weighted_consensus_amd.models import bert
    from llm_weighted_consensus_amd.models.config import encoder_config

    m = bert.BertEncoder(encoder_config(arch), device=gpu, seed=5)
    inputs = [m.pack([[(37 * i + 11 * j + 50 * k) % 900 + 1 for j in range(n // 2)] for i in range(2)])[:3] for k in range(3)]
    want = []
    for a in inputs:
        want.append(m.forward_packed(*a, n))
        torch.cuda.synchronize()
    assert not torch.equal(want[0], want[1])
    got = [(k % 3, m.forward_packed(*inputs[k % 3], n)) for k in range(12)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    for k in range(40):
        with torch.cuda.stream(streams[k % 2]):
            got.append((k % 3, m.forward_packed(*inputs[k % 3], n)))
    torch.cuda.synchronize()
    assert all(torch.equal(y, want[k]) for k, y in got)
    ids = inputs[0][0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = m.forward_packed(ids, *inputs[0][1:], n)
    for k in (0, 1, 2, 1, 0):
        ids.copy_(inputs[k][0])
        graph.replay()
        assert torch.equal(y, want[k])
        m.forward_packed(*inputs[2], n)


def test_few_row_encoder_of_more_layers_than_a_launch(gpu, monkeypatch):
    """A stack of 26 layers is two launches: the second goes on from what the first left.  The bound as above."""
    from dataclasses import replace

    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models import bert
    from llm_weighted_consensus_amd.models.config import encoder_config

    m = bert.BertEncoder(replace(encoder_config("bge-small-en-v1.5"), layers=26), device=gpu, seed=5)
    args = m.pack([[7, 9, 11, 13, 500], [3] * 6])
    taken, few = [], ops.encoder_few
    monkeypatch.setattr(ops, "encoder_few", lambda *a: taken.append(few(*a)) or taken[-1])
    y = m.forward_packed(*args)
    assert len(taken) == 1 and taken[0] is y
    ref = m.forward_reference(*args[:3])
    monkeypatch.setattr(bert, "FEW_ROWS", 0)
    plain = m.forward_packed(*args)
    err = lambda t: ((t.float() - ref).norm() / ref.norm()).item()  # noqa: E731
    assert err(y) < 2 * err(plain) and err(y) < 0.03, (err(y), err(plain))


# the core of each projection of a decode step (None: the library, with the norm and RoPE kernels in front of it)
_STEP_CORES = {"gv": ["gv"] * 5, "g2": ["g2"] * 5, "library o and head": ["gv", None, "g2", "g2", None], "library qkv and down": [None, "gv", "g2", None, "gv"],
               "library gate|up": ["g2", "g2", None, "gv", "g2"]}


@pytest.mark.parametrize("cores", list(_STEP_CORES))
@pytest.mark.parametrize("B,longest,splits", [(1, 600, 1), (1, 600, 4), (17, 400, 3), (64, 60, 1)])
def test_decode_step_without_kernels_between_its_gemms(gpu, monkeypatch, cores, B, longest, splits):
    """The decode step of few rows (norms, RoPE and cache writes in the projections, splits added up in the attention) over
    three layers with norm weights other than one, every projection on a core of its own and some on the library: logits
    and cached rows against the fp32 forward, no further off than the step of separate kernels but for the spread of two
    roundings (2 x); nothing else in the cache changes, a row without a slot writes nothing; a captured step gives the same bits."""
    from llm_weighted_consensus_amd import ops
    from llm_weighted_consensus_amd.models.config import decoder_config
    from llm_weighted_consensus_amd.models.llama import KVCache, LlamaModel
    from llm_weighted_consensus_amd.ops import gemm_plan

    cfg = decoder_config("llama-tiny", layers=3, ffn=1536)   # (every projection of a shape of its own)
    gen = torch.Generator(device="cpu").manual_seed(B + splits)
    m = LlamaModel(cfg, device=gpu, seed=7, max_position=1024, fold_norms=False)
    norm = lambda: (0.5 + torch.rand(cfg.hidden, generator=gen)).to(gpu, torch.bfloat16)  # noqa: E731
    for L in m.layers:
        L.attn_norm, L.mlp_norm = norm(), norm()
    m.final_norm = norm()
    m._fold_norms()
    lens = [int(n) for n in torch.randint(3, longest, (B,), generator=gen)]
    lens[0] = longest                                     # the last position is what the step decodes
    texts = [torch.randint(0, cfg.vocab_size, (n,), generator=gen).to(gpu) for n in lens]
    nb = [-(-n // 16) for n in lens]
    width, first = max(nb), [1 + sum(nb[:b]) for b in range(B)]
    cache = KVCache(cfg, sum(nb) + 1, 16, gpu)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)  # noqa: E731
    tables = torch.zeros(B, width, dtype=torch.int32, device=gpu)
    for b in range(B):
        tables[b, :nb[b]] = torch.arange(first[b], first[b] + nb[b])
    past = [n - 1 for n in lens]
    cu = i32([0] + torch.tensor(past).cumsum(0).tolist())
    m.prefill(torch.cat([t[:-1] for t in texts]).int(), i32([p for n in past for p in range(n)]),
              i32([first[b] * 16 + p for b in range(B) for p in range(past[b])]), cu, max(past), (cu[1:] - 1).long(), cache)
    slots = [first[b] * 16 + past[b] for b in range(B)]
    live = list(range(B))
    if B == 17:                                           # a padded row, as the engine has them
        slots[5], lens[5], past[5] = -1, 1, 0
        tables[5] = 0
        live.remove(5)
    args = (torch.stack([t[-1] for t in texts]).int(), i32(past), i32(slots), tables, i32(lens), cache)
    before = cache.pool.clone()
    taken = []
    for name in ("step_qkv", "step_project"):
        f = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda x, w, core, *a, _f=f, _n=name, **kw: taken.append((_n, tuple(w.shape), core)) or _f(x, w, core, *a, **kw))
    monkeypatch.setattr(gemm_plan, "MODE", "auto")
    L, want, ss = m.layers[0], [], True
    shapes = [(L.wqkv, "plain"), (L.wo, "residual"), (L.w_gate_up, "swiglu"), (L.w_down, "residual"), (m.lm_head, "plain")]
    for (w, epi), c in zip(shapes, _STEP_CORES[cores]):
        monkeypatch.setitem(gemm_plan._CHOICE, (B, w.shape[0], w.shape[1], epi), c or "blas")
    for li in range(cfg.layers):                          # who takes part: a projection behind one that left no sums does not
        for (w, epi), c in list(zip(shapes, _STEP_CORES[cores]))[:4] + ([(shapes[4], _STEP_CORES[cores][4])] if li + 1 == cfg.layers else []):
            if c and (ss or epi == "residual"):
                want.append(("step_qkv" if w is L.wqkv else "step_project", tuple(w.shape), {"gv": 1, "g2": 2}[c]))
            ss = bool(c) if epi == "residual" else ss
    got = m.decode(*args, num_splits=splits)
    assert taken == want
    after = cache.pool.clone()
    cache.pool.copy_(before)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m.decode(*args, num_splits=splits)
    for _ in range(3):
        cache.pool.copy_(before)
        out.fill_(float("nan"))
        graph.replay()
        assert torch.equal(out[live], got[live]) and torch.equal(cache.pool, after)
        assert torch.equal(m.decode(*args, num_splits=splits)[live], got[live])
    cache.pool.copy_(before)
    monkeypatch.setenv("LWC_DECODE_QROPE", "0")           # the step of separate kernels
    n = len(taken)
    plain = m.decode(*args, num_splits=splits)
    assert len(taken) == n
    refs = torch.stack([ref.llama_forward(m, texts[b])[-1] for b in live])
    err = lambda t: ((t[live].float() - refs).norm() / refs.norm()).item()  # noqa: E731
    assert err(got) < 2 * err(plain) and err(got) < 0.03, (err(got), err(plain))
    ours, theirs, was = (t.view(cfg.layers, 2, -1, cfg.kv_heads, 16 * cfg.head_dim) for t in (after, cache.pool, before))
    blocks = torch.zeros(ours.shape[2], dtype=torch.bool, device=gpu)
    blocks[[slots[b] // 16 for b in live]] = True
    assert torch.equal(ours[:, :, ~blocks], was[:, :, ~blocks])
    wrote, expect = (after != before), (cache.pool != before)
    assert (wrote.sum() - expect.sum()).abs() <= 0.01 * expect.sum()      # (a value may round to what was there)
    assert ((ours.float() - theirs.float()).norm() <= 0.02 * (theirs.float() - was.float()).norm())
