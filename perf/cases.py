"""Work that users of this framework have it do, as cases that can be timed and compared.

A case is one pass through the public entry points: a decode step of a batch of sequences (captured into a graph
once, as the engine keeps one per batch bucket), the prefill of a batch of prompts, the fused sampler over a step's
logits, the embedding of texts, the embedding consensus over sampled candidates.  Decoders run with a few layers of
their real width (every layer of a stack costs the same) and their whole vocabulary; encoders run whole.

  llama    Llama-3-8B layers, bf16: the sampler of the consensus server
  mixtral  Mixtral-8x7B layers in bf16; mixtral-fp8: the same with fp8 experts and projections
  limatar  low-rank attention and retention layers, routed experts with a shared one, a dense clamped unit
  merudra  grouped attention and gated delta rule layers, routed and identity experts, input convolutions
  bge-*    the BERT encoders behind /embeddings and the consensus score
  e5       e5-mistral-7b layers as a last-token embedder, fp8 projections

Weights are random and the same in every case of a model (a server loads them once); prompts, contexts, cached keys
and values and candidates come from the seed.  Cached rows hold what the projections of normalised rows give (normal,
standard deviation 1.28); routers are as decisive as trained ones (logits a few units apart); the embeddings of the fp8
and routed models are scaled so that a layer changes the residual stream by a fraction, as in trained ones (else the
rounding of e4m3 activations compounds from layer to layer until two correct runs have little in common).
"""
import gc
import json
import math
import os
import random
import shutil
import tempfile
from array import array

import numpy as np
import torch

from llm_weighted_consensus_amd import ops
from llm_weighted_consensus_amd.embeddings.consensus import EmbeddingConsensus
from llm_weighted_consensus_amd.engine.engine import BUCKETS, cascade_table_size, cascade_tiles
from llm_weighted_consensus_amd.models.bert import BertEncoder
from llm_weighted_consensus_amd.models.config import LimatarConfig, MerudraConfig, decoder_config, encoder_config
from llm_weighted_consensus_amd.models.embedder import DecoderEmbedder
from llm_weighted_consensus_amd.models.limatar import LimatarModel
from llm_weighted_consensus_amd.models.llama import KVCache, LlamaModel
from llm_weighted_consensus_amd.models.merudra import MerudraModel
from llm_weighted_consensus_amd.models.mixtral import MixtralModel

DEV = "cuda"
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
BLOCK = 16                     # tokens per cache block, the engine's default
WEIGHT_SEED = 1234
KV_STD = 1.28                  # 0.02 * sqrt(4096): keys and values of unit-RMS rows
LAYERS = {"llama": 4, "mixtral": 2, "mixtral-fp8": 2, "e5": 3}
STREAM = {"mixtral": 256.0, "mixtral-fp8": 256.0, "e5": 256.0}   # embedding scale (a power of two: exact in bf16)
MAX_POS = 8192
MODEL_LEN = 4096               # the engine's default limit: how wide its block tables are
ENCODERS = {"bge-small": "bge-small-en-v1.5", "bge-base": "bge-base-en-v1.5", "bge-large": "bge-large-en-v1.5"}


def listed():
    return [
        # one chat user: the latency of a single sequence's next token
        {"name": "decode llama 1", "path": "decode", "model": "llama", "requests": 1, "n": 1, "prompt": 210, "spread": 0.0, "own": 37},
        # the voters of concurrent score requests: unrelated sequences of very different lengths in one step
        {"name": "decode llama 61 ragged", "path": "decode", "model": "llama", "requests": 61, "n": 1, "prompt": 900, "spread": 0.8, "own": 21},
        # the consensus workload: 64 requests x 64 candidates that share their prompt, half way through 128 tokens
        {"name": "decode llama 64x64", "path": "decode", "model": "llama", "requests": 64, "n": 64, "prompt": 256, "spread": 0.0, "own": 64},
        # the same step's sampling: temperature 0.8, top-p 0.95 over the whole vocabulary
        {"name": "sample 4096", "path": "sample", "rows": 4096, "vocab": 128256, "temperature": 0.8, "top_p": 0.95, "top_k": 0, "logprobs": 0},
        # an admission wave of a quiet server: a few prompts of odd lengths
        {"name": "prefill llama 5 ragged", "path": "prefill", "model": "llama", "prompts": 5, "tokens": 260, "spread": 0.7},
        # candidates of the mixture-of-experts sampler, 8 requests x 64
        {"name": "decode mixtral-fp8 8x64", "path": "decode", "model": "mixtral-fp8", "requests": 8, "n": 64, "prompt": 256, "spread": 0.0, "own": 64},
        # a batch of prompts of the low-rank attention / retention design, the engine's whole prefill budget
        {"name": "prefill limatar 8x2048", "path": "prefill", "model": "limatar", "prompts": 8, "tokens": 2048, "spread": 0.0},
        # a serving batch of the delta rule / routed experts design at mixed contexts
        {"name": "decode merudra 64", "path": "decode", "model": "merudra", "requests": 64, "n": 1, "prompt": 1000, "spread": 0.5, "own": 16},
        # one search query to be embedded: the smallest call of the embeddings endpoint
        {"name": "embed bge-small 1", "path": "embed", "model": "bge-small", "texts": 1, "tokens": 12, "spread": 0.0},
        # one request's 64 candidates scored against each other, answers of different lengths
        {"name": "consensus bge-large 1x64", "path": "consensus", "model": "bge-large", "requests": 1, "n": 64, "tokens": 120, "spread": 0.6},
        # the encoder's batch workload: 64 requests x 64 candidates of 128 tokens
        {"name": "consensus bge-base 64x64", "path": "consensus", "model": "bge-base", "requests": 64, "n": 64, "tokens": 128, "spread": 0.0},
        # documents through the fp8 decoder-embedder
        {"name": "embed e5 64", "path": "embed", "model": "e5", "texts": 64, "tokens": 129, "spread": 0.4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode", "decode", "prefill", "prefill", "sample", "embed", "consensus"])
    spread = rng.choice([0.0, 0.3, 0.8])
    if path == "decode":
        model = rng.choice(["llama", "llama", "mixtral", "mixtral-fp8", "limatar", "limatar", "merudra", "merudra"])
        n = rng.choice([1, 1, 8, 32, 64]) if model not in ("limatar", "merudra") else 1
        rows = _log_int(rng, 1, 4096 if model == "llama" and n > 1 else 1024 if n > 1 else 128)
        return {"path": path, "model": model, "requests": max(1, rows // n), "n": n, "prompt": _log_int(rng, 40, 2000 if n == 1 else 600),
                "spread": spread, "own": _log_int(rng, 1, 128)}
    if path == "prefill":
        model = rng.choice(["llama", "llama", "mixtral", "mixtral-fp8", "limatar", "limatar", "merudra", "merudra"])
        total, prompts = _log_int(rng, 16, 16384), _log_int(rng, 1, 24)
        return {"path": path, "model": model, "prompts": prompts, "tokens": max(4, min(2048, total // prompts)), "spread": spread}
    if path == "sample":
        return {"path": path, "rows": _log_int(rng, 1, 4096), "vocab": rng.choice([128256, 32000]), "temperature": rng.choice([0.0, 0.7, 1.0]),
                "top_p": rng.choice([1.0, 0.9, 0.95]), "top_k": rng.choice([0, 0, 40]), "logprobs": rng.choice([0, 5, 20])}
    if path == "embed":
        model = rng.choice(["bge-small", "bge-base", "bge-large", "e5"])
        return {"path": path, "model": model, "texts": _log_int(rng, 1, 512 if model != "e5" else 128), "tokens": _log_int(rng, 8, 300), "spread": spread}
    return {"path": path, "model": rng.choice(["bge-small", "bge-base", "bge-large"]), "requests": _log_int(rng, 1, 24),
            "n": rng.choice([3, 16, 32, 64]), "tokens": _log_int(rng, 16, 200), "spread": spread}


# ---------------------------------------------------------------------------------------------- models
_HELD = {}     # model name -> its weights on the GPU; one model at a time, as a server would hold it


def _held(name, make):
    if name not in _HELD:
        _HELD.clear()
        gc.collect()
        torch.cuda.empty_cache()
        _HELD[name] = make()
    return _HELD[name]


def _layer_list_config(name):
    """config.json of the layer-list designs at the width of an 8B model, two layers: one of each mixer."""
    d, H, G, D, ff, V = 4096, 32, 8, 128, 14336, 32000
    if name == "limatar":
        moe = {"kind": "moe", "expert": {"ff": ff // 2}, "router": {"experts": 8, "top": 2}, "shared": {"ff": ff // 8}}
        dense = {"kind": "dense", "ff": ff, "limit": 7.0}
        lat = {"heads": H, "dim": D, "rot_dim": D // 2, "vdim": D, "q_rank": 3 * d // 8, "kv_rank": 4 * D, "scale": (D + D // 2) ** -0.5,
               "rot": {"base": 10000.0, "dims": D // 2, "scaling": {"factor": 4.0, "original": 1024, "fast": 32.0, "slow": 1.0}}}
        ret = {"heads": H, "dim": D, "vdim": D, "decay": [1.0 - 2.0 ** (-4 - 4 * h / (H - 1)) for h in range(H)],
               "rot": {"base": 10000.0, "dims": D}}
        return {"architecture": "Limatar", "layers": [{"type": "latent_attention", "mixer": lat, "mlp": moe},
                                                      {"type": "retention", "mixer": ret, "mlp": dense}],
                "norm": {"eps": 1e-6}, "vocab": V, "width": d}
    mlp = {"kind": "moe", "expert": {"ff": ff // 2}, "router": {"experts": 8, "identity": 2, "top": 2}}
    att = {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "q_temp": {"coef": 0.1, "every": 512}}
    return {"architecture": "Merudra", "canon": {"taps": 4},
            "layers": [{"type": "attention", "mixer": att, "mlp": mlp},
                       {"type": "delta", "mixer": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "conv": 4}, "mlp": mlp}],
            "norm": {"eps": 1e-5}, "token_side": {"dim": 64}, "vocab": V, "width": d}


def _layer_list_shapes(name):
    """name -> shape of the checkpoint's tensors."""
    c = _layer_list_config(name)
    d, V = c["width"], c["vocab"]
    out = {"embed": (V, d), "final.norm": (d,)}
    if name == "merudra":
        out.update({"side.embed": (V, c["token_side"]["dim"] * len(c["layers"])), "head": (V, d)})
    else:
        out["embed.norm"] = (d,)
    for i, L in enumerate(c["layers"]):
        m, p, e = L["mixer"], f"l{i}.", L["mlp"]
        H, D, Dv = m["heads"], m["dim"], m["vdim"]
        if name == "limatar":
            out.update({p + n: (d,) for n in ("norm1", "norm1b", "norm2", "norm2b")})
            if L["type"] == "latent_attention":
                R, C, Q = m["rot_dim"], m["kv_rank"], m["q_rank"]
                out.update({p + "mix.dq": (Q, d), p + "mix.dq.norm": (Q,), p + "mix.uq": (H * (D + R), Q), p + "mix.dkv": (C + R, d),
                            p + "mix.dkv.norm": (C,), p + "mix.uk": (H * D, C), p + "mix.uv": (H * Dv, C), p + "mix.sink": (H,)})
            else:
                out.update({p + "mix.q": (H * D, d), p + "mix.k": (H * D, d), p + "mix.v": (H * Dv, d)})
            out.update({p + "mix.g": (H * Dv, d), p + "mix.o": (d, H * Dv)})
        else:
            taps, sd, G = c["canon"]["taps"], c["token_side"]["dim"], m["kv_heads"]
            for s, n in (("1", "mixer"), ("2", "experts")):
                out.update({p + "norm" + s: (d,), p + "canon" + s: (d, taps), p + "rg" + s: (d, d), p + "rg" + s + ".b": (d,)})
            out.update({p + "dwa": (i + 2,), p + "side.gate": (sd, d), p + "side.proj": (d, sd), p + "side.norm": (d,)})
            if L["type"] == "attention":
                out.update({p + "mix.q": (H * D, d), p + "mix.q.b": (H * D,), p + "mix.k": (G * D, d), p + "mix.k.b": (G * D,)})
            else:
                out.update({p + "mix.q": (G * D, d), p + "mix.q.conv": (G * D, m["conv"]), p + "mix.k": (G * D, d),
                            p + "mix.k.conv": (G * D, m["conv"]), p + "mix.v": (H * Dv, d), p + "mix.v.conv": (H * Dv, m["conv"]),
                            p + "mix.b": (H, d), p + "mix.a": (H, d), p + "mix.A_log": (H,), p + "mix.dt_bias": (H,), p + "mix.norm": (Dv,)})
            out.update({p + "mix.g": (H * Dv, d), p + "mix.o": (d, H * Dv)})
        if e["kind"] == "dense":
            out.update({p + "mlp.gate": (e["ff"], d), p + "mlp.up": (e["ff"], d), p + "mlp.down": (d, e["ff"])})
            continue
        r, ff = e["router"], e["expert"]["ff"]
        outs = r["experts"] + r.get("identity", 0)
        out.update({p + "mlp.router": (outs, d), p + ("mlp.router.b" if name == "limatar" else "mlp.correction"): (outs,)})
        for x in range(r["experts"]):
            out.update({f"{p}mlp.e{x}.gate": (ff, d), f"{p}mlp.e{x}.up": (ff, d), f"{p}mlp.e{x}.down": (d, ff)})
        if "shared" in e:
            sf = e["shared"]["ff"]
            out.update({p + "mlp.shared.gate": (sf, d), p + "mlp.shared.up": (sf, d), p + "mlp.shared.down": (d, sf)})
    return out


def _layer_list_weights(name):
    """The checkpoint's tensors on the GPU (bf16)."""
    g = torch.Generator(device=DEV).manual_seed(WEIGHT_SEED)
    out = {}
    for key, shape in _layer_list_shapes(name).items():
        leaf = key.split(".")[-1]
        t = torch.randn(shape, generator=g, device=DEV)
        if leaf in ("norm1", "norm2", "norm1b", "norm2b", "norm"):
            about = 0.0 if name == "limatar" and not key.endswith((".dq.norm", ".dkv.norm")) else 1.0
            t = about + 0.1 * t
        elif leaf.startswith("canon"):
            t = 0.2 * t
        elif leaf == "conv":
            t = 0.5 * t
        elif leaf == "b" and len(shape) == 1:
            t = 0.1 * t
        elif leaf == "dwa":
            t = 0.15 * t
            t[-1] += 1.0
        elif leaf == "correction":
            t = 0.05 * t
        elif leaf == "router":
            t = t * (6.0 / math.sqrt(shape[-1]))
        elif leaf in ("embed", "sink", "A_log", "dt_bias"):
            t = t * (0.5 if leaf == "A_log" else 1.0)
        else:
            t = t / math.sqrt(shape[-1])
        out[key] = t.to(BF16)
    return out


def _save(tensors, path):
    """A .safetensors file: header length, header, the tensors' bytes one after the other."""
    head, at = {}, 0
    for k, t in tensors.items():
        n = t.numel() * t.element_size()
        head[k] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + n]}
        at += n
    raw = json.dumps(head).encode()
    raw += b" " * (-len(raw) % 8)
    with open(path, "wb") as f:
        f.write(len(raw).to_bytes(8, "little") + raw)
        for t in tensors.values():
            t.contiguous().view(torch.uint8).cpu().numpy().tofile(f)


def _make_layer_list(name):
    folder = tempfile.mkdtemp(prefix="lwc_model_")
    try:
        _save(_layer_list_weights(name), os.path.join(folder, "model.safetensors"))
        cls, cfg = (LimatarModel, LimatarConfig) if name == "limatar" else (MerudraModel, MerudraConfig)
        return cls(cfg.from_dict(_layer_list_config(name), name=name), device=DEV, weights_path=folder)
    finally:
        shutil.rmtree(folder, ignore_errors=True)


def _decoder_cfg(name):
    return decoder_config({"llama": "llama-3-8b", "e5": "e5-mistral-7b"}.get(name, "mixtral-8x7b"), layers=LAYERS[name])


def _make(name):
    if name in ENCODERS:
        return BertEncoder(encoder_config(ENCODERS[name]), device=DEV, seed=WEIGHT_SEED)
    if name == "llama":
        return LlamaModel(_decoder_cfg(name), device=DEV, seed=WEIGHT_SEED, max_position=MAX_POS)
    if name.startswith("mixtral"):
        m = MixtralModel(_decoder_cfg(name), device=DEV, seed=WEIGHT_SEED, max_position=MAX_POS, fp8=name == "mixtral-fp8")
        m.embed.mul_(STREAM[name])
        return m
    if name == "e5":
        m = LlamaModel(_decoder_cfg(name), device=DEV, seed=WEIGHT_SEED, max_position=MAX_POS, fp8_dense=True, fold_norms=False)
        m.embed.mul_(STREAM[name])
        return DecoderEmbedder(m, max_tokens=512)
    return _make_layer_list(name)


def _model(name):
    return _held(name, lambda: _make(name))


# ---------------------------------------------------------------------------------------------- inputs
def _lengths(case, count, mean, least=2):
    """Lengths of a case's sequences: the same for every seed, as the sizes of its outputs follow from them."""
    rng = random.Random(json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True))
    return [max(least, int(round(mean * (1.0 + case["spread"] * rng.uniform(-1.0, 1.0))))) for _ in range(count)]


def _vocab(name):
    return 32000 if name in ("limatar", "merudra") else _decoder_cfg(name).vocab_size


class _Batch:
    """A decode batch: every request's sequences share the whole blocks of its prompt; each has its own rows after
    them.  Rows of the cache are numbered request by request, shared rows first."""

    def __init__(self, case, seed):
        rng = random.Random(seed * 7919 + 1)
        R, n = case["requests"], case["n"]
        prompt = _lengths(case, R, case["prompt"])
        self.R, self.n, self.B = R, n, R * n
        self.past = [p + case["own"] - 1 for p in prompt]                       # rows already cached per sequence
        self.shared = [p // BLOCK * BLOCK if n > 1 else 0 for p in prompt]
        self.own = [a - s for a, s in zip(self.past, self.shared)]
        self.rows = sum(s + n * o for s, o in zip(self.shared, self.own))
        self.prompt = prompt
        self.tokens = [rng.randrange(1 << 30) % _vocab(case["model"]) for _ in range(self.B)]
        need = sum(s // BLOCK + n * (o // BLOCK + 1) for s, o in zip(self.shared, self.own))
        self.blocks = need + 1                                                  # block 0 stands under padded rows
        free = (np.random.RandomState(seed & 0x7FFFFFFF).permutation(need) + 1).astype(np.int64)
        width = max(MODEL_LEN // BLOCK, max(p // BLOCK + 1 for p in self.past))
        self.bucket = next(b for b in BUCKETS if b >= self.B)
        bt = np.zeros((self.bucket, width), np.int32)
        slot_rows, at = [], 0
        self.slots = np.full(self.bucket, -1, np.int32)
        self.positions = np.zeros(self.bucket, np.int32)
        self.ctx = np.ones(self.bucket, np.int32)
        for r in range(R):
            ns, no = self.shared[r] // BLOCK, self.own[r] // BLOCK + 1
            sh = free[at:at + ns]
            ow = free[at + ns:at + ns + n * no].reshape(n, no)
            at += ns + n * no
            b0 = r * n
            bt[b0:b0 + n, :ns] = sh
            bt[b0:b0 + n, ns:ns + no] = ow
            slot_rows.append((sh[:, None] * BLOCK + np.arange(BLOCK)).reshape(-1))
            own_slots = (ow[:, :, None] * BLOCK + np.arange(BLOCK)).reshape(n, -1)
            slot_rows.append(own_slots[:, :self.own[r]].reshape(-1))
            self.slots[b0:b0 + n] = own_slots[:, self.own[r]]
            self.positions[b0:b0 + n] = self.past[r]
            self.ctx[b0:b0 + n] = self.past[r] + 1
        self.tables = bt
        self.slot_rows = np.concatenate(slot_rows)


def _kv_rows(seed, layer, rows, width):
    """Cached key and value rows of one layer [rows, width] (keys as cached: rotated already)."""
    g = torch.Generator(device=DEV).manual_seed(seed * 131 + layer)
    return (torch.randn(rows, width, generator=g, device=DEV, dtype=F32) * KV_STD).to(BF16)


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(DEV)


def _capture(step):
    """``step`` captured into a graph, as the engine does for a batch bucket; its output tensor is rewritten by every replay."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def _prepare_decode(case, seed):
    model, b = _model(case["model"]), _Batch(case, seed)
    model.tune_gemms(b.bucket)
    cfg, layer_list = model.cfg, case["model"] in ("limatar", "merudra")
    cache = model.new_cache(b.blocks, BLOCK) if layer_list else KVCache(cfg, b.blocks, BLOCK, model.device)
    tok = np.zeros(b.bucket, np.int32)
    tok[:b.B] = b.tokens
    d = {"tokens": _i32(tok), "positions": _i32(b.positions), "slots": _i32(b.slots), "tables": _i32(b.tables), "ctx": _i32(b.ctx)}
    extra, state = {}, None
    if layer_list:
        state = model.new_state(b.B)
        _fill_context(case, seed, model, b, cache, state)
        ss = np.full(b.bucket, state.scratch, np.int32)
        ss[:b.B] = np.arange(b.B)
        extra = {"state": state, "state_slots": _i32(ss)}
    else:
        kvw = 2 * cfg.kv_heads * cfg.head_dim
        slots = _i32(b.slot_rows)
        for li in range(cfg.layers):
            rows = _kv_rows(seed, li, b.rows, kvw)
            for a in range(0, b.rows, 1 << 16):
                part = rows[a:a + (1 << 16)]
                qkv = torch.cat([part.new_zeros(part.shape[0], cfg.heads * cfg.head_dim), part], 1)
                # position 0 turns nothing: the rows enter the cache as they are
                ops.rope_kv_write(qkv, torch.zeros(part.shape[0], dtype=torch.int32, device=DEV), model.cos, model.sin, cache.k[li],
                                  cache.v[li], cfg.heads, cfg.kv_heads, cfg.head_dim, slots=slots[a:a + (1 << 16)], rope_q=False)
        # the engine's choice of attention: shared prompts read once per tile of sequences in large batches, else
        # the reduction over the context split until enough workgroups run
        if case["n"] > 1 and b.bucket >= 128 and max(b.shared):
            per = ops.cascade_rows_per_tile(cfg.heads // cfg.kv_heads)
            tiles = np.zeros((cascade_table_size(b.bucket, per), 3), np.int32)
            cascade_tiles([(r * b.n, b.n, b.shared[r] // BLOCK) for r in range(b.R)], per, tiles)
            extra["cascade_tiles"] = _i32(tiles)
        else:
            extra["num_splits"] = min(max(1, min(16, -(-1024 // (b.bucket * cfg.kv_heads)))), max(1, b.tables.shape[1] // 4))

    def step():
        return model.decode(d["tokens"], d["positions"], d["slots"], d["tables"], d["ctx"], cache, **extra)

    if state is not None:   # the run before the capture advances the scratch slot, not the sequences
        real = extra["state_slots"].clone()
        extra["state_slots"].fill_(state.scratch)
        step()
        extra["state_slots"].copy_(real)
        side = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            logits = step()
    else:
        graph, logits = _capture(step)
    return {"case": case, "graph": graph, "logits": logits, "rows": b.B, "cache": cache, "state": state, "keep": (d, extra)}


def _state_outputs(case, state, n):
    """The recurrent matrices of the first ``n`` slots."""
    return {} if state is None else {"S": state["S.1"][:n]}


def _context_tokens(case, seed, b):
    """What the sequences of a layer-list batch have been fed so far, sequence by sequence."""
    rng = np.random.RandomState((seed * 31 + 5) & 0x7FFFFFFF)
    return [rng.randint(0, _vocab(case["model"]), b.past[r]).astype(np.int64) for r in range(b.R)]


def _portions(model, toks, tables, slots, cache, state, ids):
    """One forward over whole prompts as portions over the paged cache, as the engine prefills these designs."""
    lens = [len(t) for t in toks]
    cu = np.concatenate([[0], np.cumsum(lens)])
    wide = 2 * -(-max(lens) // (2 * BLOCK))
    bt = np.zeros((len(toks), wide), np.int32)
    w = min(wide, tables.shape[1])
    bt[:, :w] = tables[:, :w]
    return {"tokens": _i32(np.concatenate(toks)), "positions": _i32(np.concatenate([np.arange(n) for n in lens])), "slots": _i32(slots),
            "cache": cache, "n_dec": 0, "dec": None,
            "chunk": {"cu_q": _i32(cu), "block_tables": _i32(bt), "k_lens": _i32(lens), "max_q": max(lens), "lens": (lens, lens)},
            "logit_rows": torch.from_numpy(cu[1:] - 1).to(DEV), "state": state, "state_slots": _i32(ids)}


def _fill_context(case, seed, model, b, cache, state):
    toks = _context_tokens(case, seed, b)
    at = np.concatenate([[0], np.cumsum(b.past)])
    a = 0
    while a < b.R:
        e, total = a, 0
        while e < b.R and (e == a or total + b.past[e] <= 16384):
            total += b.past[e]
            e += 1
        model.forward_mixed(**_portions(model, toks[a:e], b.tables[a:e], b.slot_rows[at[a]:at[e]], cache, state, np.arange(a, e)))
        a = e


def _prompts(case, seed):
    lens = _lengths(case, case["prompts"], case["tokens"])
    nr = np.random.RandomState((seed * 31 + 6) & 0x7FFFFFFF)
    return [nr.randint(0, _vocab(case["model"]), n).astype(np.int64) for n in lens]


def _prepare_prefill(case, seed):
    model, toks = _model(case["model"]), _prompts(case, seed)
    lens = [len(t) for t in toks]
    nb = [n // BLOCK + 1 for n in lens]
    free = np.random.RandomState(seed & 0x7FFFFFFF).permutation(sum(nb)).astype(np.int64)
    tables = np.zeros((len(lens), max(nb)), np.int32)
    slots, at = [], 0
    for i, n in enumerate(lens):
        blk = free[at:at + nb[i]]
        at += nb[i]
        tables[i, :nb[i]] = blk
        slots.append((blk[:, None] * BLOCK + np.arange(BLOCK)).reshape(-1)[:n])
    slots = np.concatenate(slots)
    if case["model"] in ("limatar", "merudra"):
        cache, state = model.new_cache(sum(nb), BLOCK), model.new_state(len(lens))
        return {"case": case, "model": model, "args": _portions(model, toks, tables, slots, cache, state, np.arange(len(lens))),
                "cache": cache, "state": state, "rows": len(lens)}
    cache = KVCache(model.cfg, sum(nb), BLOCK, model.device)
    cu = np.concatenate([[0], np.cumsum(lens)])
    args = {"tokens": _i32(np.concatenate(toks)), "positions": _i32(np.concatenate([np.arange(n) for n in lens])), "slots": _i32(slots),
            "cu_seqlens": _i32(cu), "max_seqlen": max(lens), "last_idx": torch.from_numpy(cu[1:] - 1).to(DEV), "cache": cache}
    return {"case": case, "model": model, "args": args, "cache": cache, "state": None, "rows": len(lens)}


def _logits_for(case, seed):
    """A step's logits as language models give them: a broad bulk and a few likely tokens."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    B, V = case["rows"], case["vocab"]
    out = torch.empty(B, V, dtype=BF16, device=DEV)
    for a in range(0, B, 512):
        x = torch.randn(min(512, B - a), V, generator=g, device=DEV) * 2.0
        at = torch.randint(0, V, (x.shape[0], 32), generator=g, device=DEV)
        x.scatter_add_(1, at, 4.0 + 8.0 * torch.rand(at.shape, generator=g, device=DEV))
        out[a:a + 512] = x
    return out


def _prepare_sample(case, seed):
    B = case["rows"]
    full = lambda v, dt: torch.full((B,), v, dtype=dt, device=DEV)  # noqa: E731
    rng = np.random.RandomState(seed & 0x7FFFFFFF)
    args = {"temperature": full(case["temperature"], F32), "top_p": full(case["top_p"], F32), "top_k": full(case["top_k"], torch.int32),
            "min_p": full(0.0, F32), "top_a": full(0.0, F32), "seeds": torch.from_numpy(rng.randint(0, 1 << 62, B, dtype=np.int64)).to(DEV),
            "offsets": torch.from_numpy(rng.randint(0, 2000, B, dtype=np.int64)).to(DEV), "num_logprobs": case["logprobs"],
            "need_logprob": case["logprobs"] > 0}
    return {"case": case, "logits": _logits_for(case, seed), "args": args}


def _texts(case, seed):
    """Token ids of the texts.  Candidates of one request are versions of one answer with some tokens replaced."""
    nr = np.random.RandomState((seed * 31 + 7) & 0x7FFFFFFF)
    V = 32000 if case["model"] == "e5" else 30522
    if case["path"] == "embed":
        return [[nr.randint(1000, 30000, n).tolist() for n in _lengths(case, case["texts"], case["tokens"])]]
    out, n = [], case["n"]
    every = _lengths(case, case["requests"] * n, case["tokens"])
    for r in range(case["requests"]):
        lens = every[r * n:(r + 1) * n]
        base = nr.randint(1000, V, max(lens))
        req = []
        for size in lens:
            t = base[:size].copy()
            swap = nr.rand(size) < 0.9 * nr.rand()
            t[swap] = nr.randint(1000, V, int(swap.sum()))
            req.append(array("i", t.tolist()))
        out.append(req)
    return out


def _prepare_texts(case, seed):
    model, texts = _model(case["model"]), _texts(case, seed)
    if case["path"] == "consensus":
        return {"case": case, "scorer": EmbeddingConsensus(model, tau=0.05, max_tokens=512), "requests": texts}
    return {"case": case, "encoder": model, "texts": texts[0]}


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "sample": _prepare_sample, "embed": _prepare_texts,
            "consensus": _prepare_texts}[case["path"]](case, seed)


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "decode":
        state["graph"].replay()
        return {"logits": state["logits"][:state["rows"]], "cache": state["cache"].pool, **_state_outputs(case, state["state"], state["rows"])}
    if path == "prefill":
        m = state["model"]
        logits = m.prefill(**state["args"]) if state["state"] is None else m.forward_mixed(**state["args"])
        return {"logits": logits, "cache": state["cache"].pool, **_state_outputs(case, state["state"], state["rows"])}
    if path == "sample":
        tok, lp, ids, lps = ops.sample(state["logits"], **state["args"])
        return {"token": tok} if not case["logprobs"] else {"token": tok, "logprob": lp, "top_ids": ids, "top_logprobs": lps}
    if path == "embed":
        return {"embedding": state["encoder"].embed(state["texts"])[0]}
    res = state["scorer"].score(state["requests"])
    # (the winner itself is the largest centrality: versions of one answer come close enough to tie)
    return {"similarity": res.similarity, "centrality": res.centrality, "weights": res.weights}


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _layer_list_sizes(name):
    """Parameters of the layers, those that one row multiplies with, and of these the last layer's behind its mixer."""
    total = active = tail = 0
    for k, shape in _layer_list_shapes(name).items():
        n = math.prod(shape)
        if k in ("embed", "head", "side.embed") or len(shape) == 1:
            continue
        total += n
        used = n / 4 if ".mlp.e" in k else n       # 2 of 8 experts
        active += used
        tail += used if k.startswith("l1.mlp") or k in ("l1.mix.o", "l1.rg2") else 0
    return total, active, tail


def work(case):
    path, name = case["path"], case.get("model")
    if path == "sample":
        return {"bytes": case["rows"] * (2.0 * case["vocab"] + 40), "flops": 4.0 * case["rows"] * case["vocab"]}
    if path in ("embed", "consensus"):
        seqs = case["texts"] if path == "embed" else case["requests"] * case["n"]
        tok = float(seqs * case["tokens"])
        if name == "e5":
            c = _decoder_cfg("e5")
            qkv, rest = c.hidden * c.qkv_dim, c.heads * c.head_dim * c.hidden + 3 * c.hidden * c.ffn
            attn = 2.0 * tok * case["tokens"] * c.heads * c.head_dim
            # (the last layer ends on the texts' last tokens)
            return {"bytes": c.layers * (qkv + rest) + tok * c.hidden * 2,
                    "flops": c.layers * (2.0 * qkv * tok + attn) + 2.0 * rest * (tok * (c.layers - 1) + seqs)}
        c = encoder_config(ENCODERS[name])
        per = 4 * c.hidden ** 2 + 2 * c.hidden * c.ffn
        return {"bytes": 2.0 * c.layers * per + tok * c.hidden * 2 + seqs * c.hidden * 4,
                "flops": c.layers * (2.0 * per * tok + 4.0 * tok * case["tokens"] * c.hidden)}
    V = _vocab(name)
    if path == "decode":
        rows, past = float(case["requests"] * case["n"]), case["prompt"] + case["own"]
        shared = case["prompt"] // BLOCK * BLOCK if case["n"] > 1 else 0
        cached = case["requests"] * shared + rows * (past - shared)
        logits = rows
    else:
        rows, past = float(case["prompts"] * case["tokens"]), case["tokens"] / 2.0
        cached, logits = rows, float(case["prompts"])
    if name in ("limatar", "merudra"):
        total, active, tail = _layer_list_sizes(name)
        hit = 1.0 if rows >= 32 else 0.25
        row_bytes, att, hidden = (2 * 576, 32 * (576 + 512) if path == "decode" else 32 * 320, 4096) if name == "limatar" else (4 * 1024, 32 * 256, 4096)
        seqs = rows if path == "decode" else case["prompts"]
        state = seqs * 32 * 128 * 128 * 4 * (2 if path == "decode" else 1)
        return {"bytes": 2.0 * (total * hit + V * hidden) + cached * row_bytes + state + logits * V * 2,
                "flops": 2.0 * rows * (active - tail) + 2.0 * logits * (tail + V * hidden) + 2.0 * rows * past * att + rows * 32 * 128 * 128 * 6}
    c = _decoder_cfg(name)
    attn = c.hidden * c.qkv_dim + c.heads * c.head_dim * c.hidden
    mlp = 3 * c.hidden * c.ffn
    wb, moe = 1.0 if name == "mixtral-fp8" else 2.0, bool(c.num_experts)
    experts = (8 if rows >= 32 else 2) if moe else 1
    tail = c.heads * c.head_dim * c.hidden + mlp * (2 if moe else 1)     # behind the attention: in the last layer for the wanted rows only
    return {"bytes": wb * c.layers * (attn + experts * mlp) + 2.0 * V * c.hidden + c.layers * cached * 4 * c.kv_heads * c.head_dim + logits * V * 2,
            "flops": 2.0 * rows * (c.layers * c.hidden * c.qkv_dim + (c.layers - 1) * tail) + 2.0 * logits * (tail + V * c.hidden) + 4.0 * c.layers * rows * past * c.heads * c.head_dim}


def tolerance(case):
    if case["path"] == "sample":   # a draw at the edge of a cumulative sum may go either way; ties among equal logits
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.005}
    if case["path"] == "consensus":   # cosines of bf16 encoders: 64 bits are 0.0005 away, the sharper weights 0.003
        return {"rel": 0.01, "max": 0.05}
    return {"rel": 0.03, "max": 0.99}   # bf16 stacks: 64 bits are 0.01 to 0.02 away; single routed rows may change experts


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softmax_rows(s, sink=None):
    if sink is None:
        return torch.softmax(s, -1)
    return torch.softmax(torch.cat([s, sink.view(1, -1, 1, 1).expand(*s.shape[:3], 1)], -1), -1)[..., :-1]


def _attend(q, k, v, lens, scale, causal, sink=None):
    """q [T, H, D], k [T, G, D], v [T, G, Dv] of packed sequences -> [T, H, Dv]."""
    H, G, out, at, i = q.shape[1], k.shape[1], [], 0, 0
    while i < len(lens):
        e, L = i, 0
        while e < len(lens) and (e == i or (e + 1 - i) * H * max(L, lens[e]) ** 2 < 2 ** 28):
            L = max(L, lens[e])
            e += 1
        n = e - i
        idx = torch.full((n, L), -1, dtype=torch.int64)
        for j in range(n):
            idx[j, :lens[i + j]] = at + torch.arange(lens[i + j])
            at += lens[i + j]
        idx = idx.to(DEV)
        ok, src = idx >= 0, idx.clamp(min=0)
        qb, kb, vb = (t[src].transpose(1, 2) for t in (q, k, v))
        if G != H:
            kb, vb = kb.repeat_interleave(H // G, 1), vb.repeat_interleave(H // G, 1)
        s = (qb @ kb.transpose(2, 3)) * scale
        bar = ~ok[:, None, None, :]
        if causal:
            p = torch.arange(L, device=DEV)
            bar = bar | (p[None, :] > p[:, None])
        s = s.masked_fill(bar, -math.inf)
        out.append((_softmax_rows(s, sink) @ vb).transpose(1, 2)[ok])
        i = e
    return torch.cat(out)


def _rope(x, positions, base, dims, scaling=None, pairs="half"):
    """Rotation of the first ``dims`` entries of x [T, ..., D]."""
    i = torch.arange(dims // 2, dtype=F64)
    f, mult = base ** (-2.0 * i / dims), 1.0
    if isinstance(scaling, dict):      # blended frequencies over a ramp of the pair index
        fac, orig = scaling["factor"], scaling["original"]
        at = lambda turns: dims * math.log(orig / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(at(scaling["fast"])), 0), min(math.ceil(at(scaling["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, mult = f / fac * ramp + f * (1.0 - ramp), 0.1 * math.log(fac) + 1.0
    elif scaling:                      # by wavelength, in three bands
        fac, lo, hi, orig = scaling
        wl = 2 * math.pi / f
        s = (orig / wl - lo) / (hi - lo)
        f = torch.where(wl > orig / lo, f / fac, torch.where(wl < orig / hi, f, (1 - s) * f / fac + s * f))
    a = positions.to(F64).view(-1, *[1] * (x.dim() - 1)) * f.to(DEV)
    c, s = torch.cos(a) * mult, torch.sin(a) * mult
    r = x[..., :dims]
    if pairs == "half":
        u, w = r[..., :dims // 2], r[..., dims // 2:]
        r = torch.cat([u * c - w * s, w * c + u * s], -1)
    else:
        u, w = r[..., 0::2], r[..., 1::2]
        r = torch.stack([u * c - w * s, w * c + u * s], -1).flatten(-2)
    return torch.cat([r, x[..., dims:]], -1)


def _fp8(w):
    """What e4m3 weights with one scale per output channel hold."""
    s = w.float().abs().amax(-1).clamp(min=1e-12) / 448.0
    return (w.float() / s.unsqueeze(-1)).to(torch.float8_e4m3fn).to(F64) * s.to(F64).unsqueeze(-1)


def _experts(h, z_ids, z_w, weights):
    out = torch.zeros_like(h)
    for e, (gate, up, down) in enumerate(weights):
        t, j = (z_ids == e).nonzero(as_tuple=True)
        if t.numel():
            x = h[t]
            out.index_add_(0, t, ((_silu(x @ gate().T) * (x @ up().T)) @ down().T) * z_w[t, j][:, None])
    return out


def _exact_llama(name, x_ids, positions, attend, keep, logits=True):
    """Llama-family forward; ``attend(layer, q, k, v)`` runs the attention.  The weights are drawn as the models draw
    theirs from a seed (fp8: the rounded weights; activations stay as they are)."""
    c = _decoder_cfg(name)
    g = torch.Generator(device=DEV).manual_seed(WEIGHT_SEED)
    d, D, H, G, std = c.hidden, c.head_dim, c.heads, c.kv_heads, 0.02

    def rnd(*shape, s=std):
        return (torch.randn(*shape, generator=g, device=DEV, dtype=F32) * s).to(BF16)

    small = std / math.sqrt(2 * c.layers)
    cast = _fp8 if name in ("mixtral-fp8", "e5") else (lambda w: w.to(F64))
    x = rnd(c.vocab_size, d)[x_ids].to(F64) * STREAM.get(name, 1.0)
    for li in range(c.layers):
        if c.num_experts:
            wqkv = torch.cat([rnd(H * D, d), rnd(G * D, d), rnd(G * D, d)])
            wo, router = rnd(d, H * D, s=small), rnd(c.num_experts, d, s=0.1)
            w1, w3, w2 = rnd(c.num_experts, c.ffn, d), rnd(c.num_experts, c.ffn, d), rnd(c.num_experts, d, c.ffn, s=small)
        else:
            wqkv, wo, gu, w2 = rnd(c.qkv_dim, d), rnd(d, H * D, s=small), rnd(2 * c.ffn, d), rnd(d, c.ffn, s=small)
        qkv = _unit(x, c.rms_eps) @ cast(wqkv).T
        q, k, v = (t.reshape(x.shape[0], -1, D) for t in qkv.split([H * D, G * D, G * D], -1))
        q, k = (_rope(t, positions, c.rope_theta, D, c.rope_scaling) for t in (q, k))
        a = attend(li, q, k, v)
        if li + 1 == c.layers and keep is not None:
            a, x = a[keep], x[keep]
        x = x + a.reshape(x.shape[0], -1) @ cast(wo).T
        h = _unit(x, c.rms_eps)
        if c.num_experts:
            top = torch.topk(h @ router.to(F64).T, c.experts_per_token, -1)
            x = x + _experts(h, top.indices, torch.softmax(top.values, -1),
                             [(lambda e=e: cast(w1[e]), lambda e=e: cast(w3[e]), lambda e=e: cast(w2[e])) for e in range(c.num_experts)])
        else:
            w = cast(gu)
            x = x + (_silu(h @ w[:c.ffn].T) * (h @ w[c.ffn:].T)) @ cast(w2).T
    h = _unit(x, c.rms_eps)
    return h @ rnd(c.vocab_size, d).to(F64).T if logits else h


def _exact_decode_llama(case, seed):
    b, c = _Batch(case, seed), _decoder_cfg(case["model"])
    G, D, n = c.kv_heads, c.head_dim, b.n

    def attend(li, q, k, v):
        rows = _kv_rows(seed, li, b.rows, 2 * G * D).view(b.rows, 2, G, D)
        out, at = torch.empty(b.B, c.heads, D, dtype=F64, device=DEV), 0
        for r in range(b.R):
            s, o = b.shared[r], b.own[r]
            sh = rows[at:at + s].to(F64)                                         # [s, 2, G, D]
            ow = rows[at + s:at + s + n * o].view(n, o, 2, G, D).to(F64)
            at += s + n * o
            i = slice(r * n, (r + 1) * n)
            qg = q[i].view(n, G, -1, D)
            ko = torch.cat([ow[:, :, 0], k[i, None]], 1).transpose(1, 2)          # [n, G, o + 1, D]
            vo = torch.cat([ow[:, :, 1], v[i, None]], 1).transpose(1, 2)
            ks, vs = sh[:, 0].transpose(0, 1), sh[:, 1].transpose(0, 1)           # [G, s, D]
            p = torch.softmax(torch.cat([qg @ ks.transpose(1, 2), qg @ ko.transpose(2, 3)], -1) / math.sqrt(D), -1)
            out[i] = (p[..., :s] @ vs + p[..., s:] @ vo).reshape(n, -1, D)
        return out

    pos = torch.from_numpy(b.positions[:b.B].astype(np.int64)).to(DEV)
    return {"logits": _exact_llama(case["model"], torch.tensor(b.tokens, device=DEV), pos, attend, None), "cache": None}


def _packed(toks):
    lens = [len(t) for t in toks]
    return (lens, torch.from_numpy(np.concatenate(toks)).to(DEV), torch.from_numpy(np.concatenate([np.arange(n) for n in lens])).to(DEV),
            torch.from_numpy(np.cumsum(lens) - 1).to(DEV))


def _exact_prefill_llama(case, seed):
    lens, ids, pos, last = _packed(_prompts(case, seed))
    D = _decoder_cfg(case["model"]).head_dim
    return {"logits": _exact_llama(case["model"], ids, pos, lambda li, q, k, v: _attend(q, k, v, lens, D ** -0.5, True), last), "cache": None}


def _retention(q, k, v, decay, lens):
    """S <- a S + k v^T, o = S^T q per head and sequence -> (o [T, H, Dv], final S [n, H, D, Dv])."""
    out, states, at = [], [], 0
    la = torch.log(torch.tensor(decay, dtype=F64, device=DEV))
    for n in lens:
        qs, ks, vs = (t[at:at + n].transpose(0, 1) for t in (q, k, v))
        at += n
        i = torch.arange(n, device=DEV, dtype=F64)
        gap = (i[:, None] - i[None, :]).clamp(min=0)
        w = torch.exp(la[:, None, None] * gap).tril()
        out.append(((qs @ ks.transpose(1, 2)) * w @ vs).transpose(0, 1))
        states.append((ks * torch.exp(la[:, None] * (n - 1 - i))[..., None]).transpose(1, 2) @ vs)
    return torch.cat(out), torch.stack(states)


def _exact_limatar(toks):
    c, W = _layer_list_config("limatar"), _layer_list_weights("limatar")
    w = lambda k: W[k].to(F64)  # noqa: E731
    lens, ids, pos, last = _packed(toks)
    eps, T = c["norm"]["eps"], ids.numel()
    norm = lambda x, k: _unit(x, eps) * (1.0 + w(k))  # noqa: E731
    x, S = norm(w("embed")[ids], "embed.norm"), None
    for i, L in enumerate(c["layers"]):
        m, p = L["mixer"], f"l{i}."
        H, D, Dv = m["heads"], m["dim"], m["vdim"]
        h = norm(x, p + "norm1")
        gate = h @ w(p + "mix.g").T
        if L["type"] == "latent_attention":
            C, R, rot = m["kv_rank"], m["rot_dim"], m["rot"]
            q = ((_unit(h @ w(p + "mix.dq").T, eps) * w(p + "mix.dq.norm")) @ w(p + "mix.uq").T).view(T, H, D + R)
            dkv = h @ w(p + "mix.dkv").T
            lat = _unit(dkv[:, :C], eps) * w(p + "mix.dkv.norm")
            turn = lambda t: _rope(t, pos, rot["base"], R, rot["scaling"], "adjacent")  # noqa: E731
            q = torch.cat([q[..., :D], turn(q[..., D:])], -1)
            k = torch.cat([(lat @ w(p + "mix.uk").T).view(T, H, D), turn(dkv[:, C:])[:, None].expand(T, H, R)], -1)
            a = _attend(q, k, (lat @ w(p + "mix.uv").T).view(T, H, Dv), lens, m["scale"], True, w(p + "mix.sink")).reshape(T, -1) * torch.sigmoid(gate)
        else:
            q, k, v = ((h @ w(p + "mix." + n).T).view(T, H, -1) for n in "qkv")
            q, k = (_rope(t, pos, m["rot"]["base"], m["rot"]["dims"]) for t in (q, k))
            o, S = _retention(q, k * D ** -0.5, v, m["decay"], lens)
            a = _unit(o, eps).reshape(T, -1) * _silu(gate)
        x = x + norm(a @ w(p + "mix.o").T, p + "norm1b")
        if i + 1 == len(c["layers"]):
            x = x[last]
        h, e = norm(x, p + "norm2"), L["mlp"]
        if e["kind"] == "dense":
            g, u = (h @ w(p + "mlp.gate").T).clamp(max=e["limit"]), (h @ w(p + "mlp.up").T).clamp(-e["limit"], e["limit"])
            y = (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "mlp.down").T
        else:
            top = torch.topk(h @ w(p + "mlp.router").T + w(p + "mlp.router.b"), e["router"]["top"], -1)
            names = [[f"{p}mlp.e{j}.{n}" for n in ("gate", "up", "down")] for j in range(e["router"]["experts"])]
            y = _experts(h, top.indices, torch.softmax(top.values, -1), [tuple((lambda n=n: w(n)) for n in t) for t in names])
            y = y + (_silu(h @ w(p + "mlp.shared.gate").T) * (h @ w(p + "mlp.shared.up").T)) @ w(p + "mlp.shared.down").T
        x = x + norm(y, p + "norm2b")
    return {"logits": norm(x, "final.norm") @ w("embed").T, "cache": None, "S": S}


def _conv(x, wt, pos):
    """Causal convolution along each packed sequence: y_t = sum_j w[:, j] x_(t - taps + 1 + j)."""
    taps, y = wt.shape[1], x * wt[:, -1]
    for back in range(1, taps):
        y[back:] += torch.where((pos[back:] >= back)[:, None], x[:-back], torch.zeros((), dtype=F64, device=DEV)) * wt[:, taps - 1 - back]
    return y


def _delta(q, k, v, beta, g, lens):
    """Gated delta rule of packed sequences, all of them walked together -> (o [T, H, Dv], final S [n, H, D, Dv])."""
    n, L, H, D, Dv = len(lens), max(lens), v.shape[1], q.shape[2], v.shape[2]
    start = torch.tensor([0] + list(np.cumsum(lens)[:-1]), device=DEV)
    ln = torch.tensor(lens, device=DEV)
    S = torch.zeros(n, H, D, Dv, dtype=F64, device=DEV)
    o = torch.zeros_like(v)
    order = torch.argsort(ln, descending=True, stable=True)      # the sequences still running are always the first ones
    start, counts = start[order], [sum(1 for x in lens if x > t) for t in range(L)]
    for t in range(L):
        i = start[:counts[t]] + t
        s = S[:counts[t]]
        s *= g[i][:, :, None, None]
        u = beta[i][:, :, None] * (v[i] - (s.transpose(2, 3) @ k[i][..., None])[..., 0])
        s += k[i][..., None] * u[:, :, None, :]
        o[i] = (s.transpose(2, 3) @ q[i][..., None])[..., 0]
    back = torch.empty_like(S)
    back[order] = S
    return o, back


def _exact_merudra(toks):
    c, W = _layer_list_config("merudra"), _layer_list_weights("merudra")
    w = lambda k: W[k].to(F64)  # noqa: E731
    lens, ids, pos, last = _packed(toks)
    eps, T, sd, S = c["norm"]["eps"], ids.numel(), c["token_side"]["dim"], None
    x = w("embed")[ids]
    X = [x]
    for i, L in enumerate(c["layers"]):
        m, p, e = L["mixer"], f"l{i}.", L["mlp"]
        H, G, D, Dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        h = x + _conv(x, w(p + "canon1"), pos)
        gate = h @ w(p + "mix.g").T
        if L["type"] == "attention":
            q = (h @ w(p + "mix.q").T + w(p + "mix.q.b")).view(T, H, D)
            k = (h @ w(p + "mix.k").T + w(p + "mix.k.b")).view(T, G, D)
            t = m["q_temp"]
            temp = 1.0 + t["coef"] * torch.log(((pos + 1) // t["every"] + 1).to(F64))
            a = _attend(_unit(q, eps) * temp[:, None, None], _unit(k, eps), k, lens, m["scale"], True).reshape(T, -1) * torch.sigmoid(gate)
        else:
            q, k, v = (_silu(_conv(h @ w(p + f"mix.{n}").T, w(p + f"mix.{n}.conv"), pos)) for n in "qkv")
            q, k, v = q.view(T, G, D), k.view(T, G, D), v.view(T, H, Dv)
            q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            q, k = (t.repeat_interleave(H // G, 1) for t in (q * D ** -0.5, k))
            beta = torch.sigmoid(h @ w(p + "mix.b").T)
            g = torch.exp(-torch.exp(w(p + "mix.A_log")) * torch.nn.functional.softplus(h @ w(p + "mix.a").T + w(p + "mix.dt_bias")))
            o, S = _delta(q, k, v, beta, g, lens)
            a = (_unit(o, eps) * w(p + "mix.norm")).reshape(T, -1) * _silu(gate)
        y = (a @ w(p + "mix.o").T) * torch.sigmoid(x @ w(p + "rg1").T + w(p + "rg1.b"))
        x = x + _unit(y, eps) * w(p + "norm1")
        h, tok = x + _conv(x, w(p + "canon2"), pos), ids
        if i + 1 == len(c["layers"]):
            x, h, tok, X = x[last], h[last], ids[last], [t[last] for t in X]
        s = torch.softmax(h @ w(p + "mlp.router").T, -1)
        r = e["router"]
        top = torch.topk(s + w(p + "mlp.correction"), r["top"], -1).indices
        wt = torch.gather(s, 1, top)
        names = [[f"{p}mlp.e{j}.{n}" for n in ("gate", "up", "down")] for j in range(r["experts"])]
        y = _experts(h, top, wt, [tuple((lambda n=n: w(n)) for n in t) for t in names])
        y = y + h * (wt * (top >= r["experts"])).sum(-1, keepdim=True)
        y = y * torch.sigmoid(x @ w(p + "rg2").T + w(p + "rg2.b"))
        x = x + _unit(y, eps) * w(p + "norm2")
        z = x @ w(p + "side.gate").T
        z = 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))
        y = (z * w("side.embed")[tok, i * sd:(i + 1) * sd]) @ w(p + "side.proj").T
        x = x + _unit(y, eps) * w(p + "side.norm")
        X.append(x)
        x = sum(w(p + "dwa")[j] * X[j] for j in range(i + 2))
    return {"logits": (_unit(x, eps) * w("final.norm")) @ w("head").T, "cache": None, "S": S}


def _exact_bert(name, texts):
    c = encoder_config(ENCODERS[name])
    g = torch.Generator(device=DEV).manual_seed(WEIGHT_SEED + 7)
    d, f, H = c.hidden, c.ffn, c.heads
    rnd = lambda *s: (torch.randn(*s, generator=g, device=DEV) * 0.02).to(BF16)  # noqa: E731
    word, posw, typ = rnd(c.vocab_size, d), rnd(c.max_position, d), rnd(c.type_vocab, d)
    layers = [[rnd(3 * d, d), rnd(d, d), rnd(f, d), rnd(d, f)] for _ in range(c.layers)]
    pt = (posw.float() + typ[0].float()).to(BF16).to(F64)
    ln = lambda x: torch.nn.functional.layer_norm(x, (d,), eps=c.ln_eps)  # noqa: E731
    out = []
    for a in range(0, len(texts), 512):
        lens, ids, pos, last = _packed([np.asarray(t[:512], np.int64) for t in texts[a:a + 512]])
        x = ln(word.to(F64)[ids] + pt[pos])
        for wqkv, wo, w1, w2 in layers:
            q, k, v = ((x @ t.to(F64).T).view(-1, H, d // H) for t in wqkv.split(d))
            x = ln(x + _attend(q, k, v, lens, (d // H) ** -0.5, False).reshape(-1, d) @ wo.to(F64).T)
            x = ln(x + torch.nn.functional.gelu(x @ w1.to(F64).T) @ w2.to(F64).T)
        first = x[torch.cat([last.new_zeros(1), last[:-1] + 1])]
        out.append(torch.nn.functional.normalize(first, dim=-1))
    return torch.cat(out)


def exact(case, seed):
    path, name = case["path"], case.get("model")
    if path == "sample":
        if not case["logprobs"]:
            return None     # whole numbers only
        x = _logits_for(case, seed)
        top = torch.stack([torch.log_softmax(x[a:a + 1].to(F64), -1)[0].topk(case["logprobs"]).values for a in range(x.shape[0])])
        return {"token": None, "logprob": None, "top_ids": None, "top_logprobs": top}
    if path in ("embed", "consensus"):
        texts = _texts(case, seed)
        if name == "e5":
            lens, ids, pos, last = _packed([np.asarray(t, np.int64) for t in texts[0]])
            h = _exact_llama("e5", ids, pos, lambda li, q, k, v: _attend(q, k, v, lens, 128 ** -0.5, True), last, logits=False)
            return {"embedding": torch.nn.functional.normalize(h, dim=-1)}
        E = _exact_bert(name, [t for r in texts for t in r])
        if path == "embed":
            return {"embedding": E}
        E = E.view(case["requests"], case["n"], -1)
        sim = E @ E.transpose(1, 2)
        cen = (sim.sum(-1) - sim.diagonal(dim1=1, dim2=2)) / max(1, case["n"] - 1)
        return {"similarity": sim, "centrality": cen, "weights": torch.softmax(cen / 0.05, -1)}
    if name in ("limatar", "merudra"):
        if path == "prefill":
            toks = _prompts(case, seed)
        else:
            b = _Batch(case, seed)
            toks = [np.append(t, b.tokens[r]) for r, t in enumerate(_context_tokens(case, seed, b))]
        return (_exact_limatar if name == "limatar" else _exact_merudra)(toks)
    return (_exact_decode_llama if path == "decode" else _exact_prefill_llama)(case, seed)
