"""Per-shape GEMM backend choice for the decoder projections (K6).

Backends computing ``A . W^T`` for the dense projections:

* ``blas``   — hipBLASLt through ``torch.nn.functional.linear`` (its own stream-K kernels);
* ``g8``     — the hand-written MFMA GEMM in persistent 256-row tiles with a stream-K tail (``csrc/kernels/gemm8p.hip``);
* ``g4``     — the hand-written 4-wave interleaved MFMA GEMM, 256 x 256 tiles (``csrc/kernels/gemm4w.hip``);
* ``g4n192`` — the same core with 256 x 192 tiles (the qkv projection at decode batch 4096: 512 tiles =
  two whole rounds of 256 CUs, where 256 x 256 tiles leave half of the second round idle);
* ``g4p``    — gemm4w 256 x 256 with the VAR 64 schedule: each persistent workgroup DMAs its next tile's
  first two K tiles inside its last two main-loop iterations and runs the wave-local epilogue on the
  transposed accumulator layout (``profiles/gemm4w_stamps_r5.md``).
* ``gv``     — the skinny weight-stream GEMM for few rows (M <= 256; plain, residual, SwiGLU and bias (+ GELU)
  epilogues; ``csrc/kernels/skinny.hip``): the serving path's small decode steps, the encoders' few short texts.
* ``g2``     — tiles for two workgroups per CU (``csrc/kernels/gemm2w.hip``), 64 x 64 with K ranges up to 192 x 128 by the
  sizes: up to 8192 rows (above, the 256 x 256 tiles of ``g8`` and of the library are always faster: 65536 rows x 3072 x
  1024 418 us against 387 and 322), from a few dozen rows on.
* ``g4s``    — gemm4w VAR 64 with split-K (``ops.split_plan``): shapes whose tiles leave CUs idle (the
  serving path's mid-size row counts: o / down at M = 2048 are 128 tiles for 256 CUs) run every tile as 2-4
  K-range units, a ragged last round (lm_head) splits only that round's tiles.

The gemm4w backends (``g4*``) are left out of every choice while ``ops.GEMM4W`` is off.

The hand-written cores also fuse the SwiGLU of the gate|up projection, or the residual add of the o /
down projections (:func:`linear_add_`), into their epilogue.  None wins everywhere
(``profiles/gemm4w.md``), so the choice is made per (M, N, K, epilogue) by timing every applicable
backend on the device, once, before a decode bucket's hipGraph is captured (:meth:`LlamaModel.tune_gemms`);
a hand-written core is taken when it is at least as fast as the library (``OWN_MARGIN``, 0); for a decode bucket
the engine then A/Bs whole captured steps (planner / all-library / all-own, ``LlamaModel.step_plans``).  Untuned shapes (prefill)
use hipBLASLt, but where :func:`_untuned` names a core.  ``LWC_GEMM=blas|g8|g4|g4n192`` forces one backend (``auto`` = measured, the default).
"""
from __future__ import annotations

import logging
import os
from typing import Dict, Optional, Tuple

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import GEMM4W, gemm2w, gemm2w_ok, gemm4w, gemm8p, silu_mul, skinny_gemm, skinny_ok, split_plan

MODE = os.environ.get("LWC_GEMM", "auto")
BACKENDS = ("blas", "g8", "g4", "g4n192", "g4p", "gv", "g2", "g4s")
G2_ROWS = 8192
# a hand-written core is chosen when it is at least as fast as the library in the isolated timings (no
# bias either way: the decode step's plan is then settled by the engine's in-step A/B of whole captured steps,
# engine.LLMEngine._step_ab, which sees the step's clock and cache state)
OWN_MARGIN = float(os.environ.get("LWC_GEMM_OWN_MARGIN", "0"))
EXCLUDE = {b for b in os.environ.get("LWC_GEMM_NO", "").split(",") if b}
G4 = ("g4", "g4n192", "g4p", "g4s")   # the gemm4w backends: left out of every choice while ops.GEMM4W is off
if not GEMM4W:
    EXCLUDE.update(G4)
# LWC_GEMM_SKINNY=0 leaves the skinny decode GEMM out of the timing (A/B knob)
SKINNY = os.environ.get("LWC_GEMM_SKINNY", "1") != "0"
_CHOICE: Dict[Tuple[int, int, int, str], str] = {}
TIMINGS: Dict[Tuple[int, int, int, str], Dict[str, float]] = {}
WARM: set = set()  # keys that :func:`tune` had to time on weights in the caches (those of the encoders' first calls always are)
log = logging.getLogger(__name__)


# row-count buckets (mixed chunked-prefill steps: decode rows + prompt-chunk rows vary every step): per
# (N, K, epilogue) a sorted list of (M bucket, choice); a call takes the smallest tuned bucket >= its M
_BUCKETS: Dict[Tuple[int, int, str], list] = {}


def choice(M: int, N: int, K: int, epi: str) -> str:
    if MODE in BACKENDS:
        return MODE
    c = _CHOICE.get((M, N, K, epi))
    if c is not None:
        return c
    bl = _BUCKETS.get((N, K, epi))
    if bl:
        for mb, cb in bl:
            if M <= mb:
                return cb
        return bl[-1][1]
    return "blas"


def _g8_fill(M: int, N: int, K: int) -> float:
    """How full gemm8p's rounds of 256 CUs are at a call's sizes: the product's share of a time in us per K iteration and round of
    256, 224 and 192 rows and for the hand-off of cut tiles.  The costs are those at which :func:`_untuned` was measured; the
    kernel's own (``row_tile`` and ``call_cost`` in csrc/kernels/gemm8p.hip) have fallen since, 0.79 to 1.0 of the time that these
    give, so that the calls which they let pass are the faster for it."""
    KT, least = K // 64, float("inf")
    for bm, cost in ((256, 1.0), (224, 0.89), (192, 0.83)):
        tiles = -(-M // bm) * -(-N // 256)
        G = 256 if tiles * KT >= 2048 else 8 * max(1, tiles * KT // 64)
        rest = tiles % G
        cut = 0.0 if rest == 0 else 10 + 45.0 * rest / G if tiles > G else 10.0 if G % tiles == 0 else 15.0 * G / tiles
        least = min(least, 1.56 * cost * KT * tiles / G + cut)
    return 1.56 * KT * (M / 256) * (N / 256) / 256 / least


def _untuned(M: int, N: int, K: int, epi: str) -> str:
    """The backend of a shape that no one tuned: a core of its own where it was as fast as the library or faster over a range of
    sizes (times relative to the library, weights from memory), else the library.

    Many rows of a gate|up projection: the library needs a SwiGLU pass over its [M, N] result, gemm8p none. Beyond 8192
    rows, N x K 8192 x 1024 to 27648 x 5120: 0.65 to 1.02; from 4609 rows on N decides how full the last round of tiles is:
    14336 x 2048, 8192 and 16384 x 1024, 16384 x 2048, 22016 and 28672 x 4096, 27648 x 5120 0.72 to 1.01, but 8192 x 4096
    0.65 to 1.09, 11264 x 4096 0.76 to 1.07, 9216 x 1152 up to 1.09, 4096 x 2048 up to 1.24. 32768 x 8192: 0.90 to 1.05.

    Hundreds of rows, where gemm8p's row tile fits them (90 counts of 545 to 3600): gate|up 22016, 24576 and 28672 x 4096, 24576 x
    4608, 25600 and 27648 x 5120 0.63 to 1.06 from 545 to 1900 rows and 0.76 to 1.04 from 2401 to 3600 where its tiles fill their
    rounds (:func:`_g8_fill`), else up to 1.16 (25600 x 5120, 913 rows); between the two up to 1.10, fewer columns either way
    (14336 x 4096 0.74 to 1.17, 8192 x 4096 0.88 to 1.20), 32768 x 4096 up to 1.11. Down into 16 column tiles, 3968 x 12288, 4096 x
    11008, 12800 and 14336: 0.49 to 1.03 from 545 to 1900 rows but for 897 to 960 at the narrower K (0.97 to
    1.08; 0.94 to 0.99 at 14336); 2048 x 14336 up to 1.15, 5120 x 13824 1.10, 8192 x 14336 1.11, 4096 x 8192 1.14.

    Down into the same 16 column tiles by other counts (94 counts at 3968 x 12288, 4096 x 11008, 12800 and 14336): 385 to 544 rows
    0.79 to 1.00, 321 to 384 up to 1.02. Beyond 4096 rows it is the library that changes: 4096 rows x 14336 take it 309 us, 4097
    722, gemm8p 319 and 347, whose tail of tiles is cut over all CUs. 4097 to 4608 rows 0.47 to 0.52, 6145 to 7424 0.60 to 0.90,
    8193 to 12032 0.64 to 0.92, 12289 to 13824 0.82 to 0.92; between them the library's tiles fit again: 4609 to 5120 0.90 to 1.04,
    5121 to 5632 0.60 to 1.09, 5633 to 6144 up to 1.06, 7425 to 8192 to 1.06, 12033 to 12288 to 1.04.

    Few rows (prefill: a batch of prompts' last layer runs on their last tokens only, and short prompts on few rows
    everywhere): the weight's read bounds them. gate|up, which saves its SwiGLU pass, up to 64 rows on gemm2w: 11264, 14336
    and 28672 x 4096, 16384 x 2048, 12288 x 3072, 32768 x 4096 0.74 to 0.98, 22016 x 4096 0.77 to 1.05, 8192 x 4096 0.94 to
    1.06, but 4096 x 8192 to 1.13, 16384 x 8192 to 1.07. The others on the weight stream up to 16 rows: 2048 x 2048 to 8192
    x 2048, 1024 x 4096 to 4096 x 4096 0.54 to 0.99, but 16384 x 1024 1.06 to 1.25, 6144 x 4096 0.90 to 1.23; on gemm2w from
    33 to 64: 2048 to 6144 x 4096 to 14336 0.56 to 0.99, 8192 x 2048 and 16384 x 1024 0.70 to 0.90, but 8192 and 14336 x
    4096 1.04 to 1.09. From 17 to 32 rows the library keeps all: both cores gain on some weights (4096 x 2048 0.72 and 0.91,
    4096 x 14336 1.2 and 0.87) and lose on others (8192 x 4096 1.27 and 1.18). Down from 65 to 128 on gemm2w, whose K ranges fill
    the CUs that a few column tiles leave idle: 14 weights of 2048 to 4096 x 8192 to 18688 0.30 to 0.95, but 4608 x 12288,
    5120 x 8192 and 13824 0.92 to 1.37; 129 to 144 rows, a third row tile, up to 1.40.

    With the weights past the caches (``weights_pass``, csrc/kernels/common.h) gemm2w also leads at up to 32 rows of a head, 32000 to
    151936 x 4096, 50304 and 151936 x 2048, 32768 x 5120, 65536 x 8192 0.46 to 1.00 (128256 x 4096, 5 rows 183 us -> 152; 33 to 64 rows
    up to 1.07; 30522 x 1024 is 16 us on either).

    Down at up to 24 rows, 12 widths and 16 depths of 4096 to 5120 x 11008 to 14336: 0.49 to 1.02, 0.57 at 4096 and 5120 x 11008, but for
    the multiples of 512 below 14336, for which the library has its best kernels: 4096 up to 16 rows 0.98 to 1.04, below 8 rows 4160 to
    4672 0.94 to 1.06 and the wider 13824 0.99 to 1.03. (4096 x 8192 up to 1.08.)"""
    size = N * K
    if epi == "swiglu":
        if M > 4608:  # (M * N: 32-bit byte offsets)
            wide = N >= (8192 if M > 8192 or K <= 1024 else 14336)
            return "g8" if wide and 1 << 23 <= size < 1 << 28 and M * N < 1 << 30 else "blas"
        if 22016 <= N <= 28672 and 4096 <= K <= 5120 and (544 < M <= 1900 or 2400 < M <= 3600) and _g8_fill(M, N, K) >= 0.8:
            return "g8"
        return "g2" if M <= 64 and N >= 8192 and K <= 4096 and 1 << 25 <= size <= 1 << 27 else "blas"
    if epi == "residual" and 3840 < N <= 4096 and 11008 <= K <= 14336 and (
            384 < M <= 1900 and not (896 < M <= 960 and K <= 12800) or  # (a fifth row tile, of 192 or 224, has little to do)
            4096 < M <= 4608 or 6144 < M <= 7424 or 8192 < M <= 12032 or 12288 < M <= 13824):
        return "g8"
    if epi == "residual" and 64 < M <= 128 and 2048 <= N <= 4096 and K >= 8192 and size <= 1 << 26:
        return "g2"
    if epi == "plain" and M <= 32 and N >= 32000 and 2048 <= K <= 8192 and 3 << 25 <= size < 1 << 30:
        return "g2"
    if epi == "residual" and M <= 24 and 4096 <= N <= 5120 and 11008 <= K <= 14336 and (
            K % 512 or K > 13824 or M > 16 or N > 4096 and (M >= 8 or N >= 4736 and K < 13824)):
        return "g2"
    if M <= 16 and K <= 4096 and N <= 8 * K and 1 << 22 <= size <= 1 << 24:
        return "gv"
    return "g2" if 32 < M <= 64 and (N < 8192 or K <= 2048) and 1 << 24 <= size <= 1 << 26 else "blas"


def _unseen(*ts: torch.Tensor) -> bool:
    """Whether no one but autograd could see or transform a torch call of these tensors: no forward-mode duals, vmap or other function
    transforms, fake and other subclasses, dispatch modes, tracing."""
    if not set(map(type, ts)) <= {torch.Tensor, torch.nn.Parameter}:
        return False
    if torch._C._functorch.peek_interpreter_stack() is not None or torch._C._len_torch_dispatch_stack() or \
            torch.jit.is_tracing() or torch.compiler.is_compiling():
        return False
    return forward_ad._current_level < 0 or all(forward_ad.unpack_dual(t).tangent is None for t in ts)


def _plain(*ts: torch.Tensor) -> bool:
    """Whether a raw kernel may take these tensors' place in a torch call: nothing records, transforms or watches it."""
    return not (torch.is_grad_enabled() and any(t.requires_grad for t in ts)) and _unseen(*ts)


def _backend(x: torch.Tensor, w: torch.Tensor, epi: str, ws, acc: Optional[torch.Tensor] = None):
    """(backend, its workspace) of a call: as tuned or forced with the caller's, else :func:`_untuned` with the current
    stream's own (a model's workspace belongs to the stream of its steps).  The library keeps what only it takes
    (:func:`_plain`; operands off 16 bytes, a strided weight) and, untuned, what is captured."""
    (M, K), N = x.shape, w.shape[0]
    b = choice(M, N, K, epi)
    if b != "blas" or MODE != "auto" or (M, N, K, epi) in _CHOICE or (N, K, epi) in _BUCKETS:
        return b, ws
    own = _untuned(M, N, K, epi)
    if own == "blas" or not (x.is_cuda and w.is_cuda and x.dtype == w.dtype == torch.bfloat16
                             and _plain(*(t for t in (x, w, acc) if t is not None)) and w.is_contiguous()
                             and x.stride(0) % 8 == 0 and M * x.stride(0) < 1 << 30
                             and (x.data_ptr() | w.data_ptr()) % 16 == 0) or torch.cuda.is_current_stream_capturing():
        return b, ws
    return own, None


def _g8_ok(N: int, K: int, epi: str) -> bool:
    return K % 64 == 0 and N % (64 if epi == "swiglu" else 8) == 0


def _own_ok(b: str, x: torch.Tensor, N: int, K: int, epi: str) -> bool:
    """Whether hand-written backend ``b`` takes this call (layout and the cores' shape rules; ``LWC_GEMM_NO``:
    a comma list of backends the planner leaves out, for A/B runs)."""
    if b == "blas" or not _g8_ok(N, K, epi) or x.stride(1) != 1 or x.stride(0) < K or b in EXCLUDE:
        return False  # (rows that overlap, or an expanded row: the cores bound x by rows * stride, or refuse it)
    if b == "gv":
        return SKINNY and skinny_ok(x.shape[0], N, K, swiglu=epi == "swiglu")
    if b == "g2":
        return x.is_cuda and x.shape[0] <= G2_ROWS and gemm2w_ok(N, K, x, swiglu=epi == "swiglu")
    if b == "g4s":  # VAR 64, split-K wherever split_plan splits this M (else unsplit: a bucket's M varies)
        return x.is_cuda
    return not (b == "g4n192" and epi == "swiglu")


def _own(b: str, x: torch.Tensor, w: torch.Tensor, ws=None, **kw) -> torch.Tensor:
    if b == "g8":
        return gemm8p(x, w, ws=ws, **kw)
    if b == "gv":
        return skinny_gemm(x, w, **kw)
    if b == "g2":
        return gemm2w(x, w, ws=ws, **kw)
    if b == "g4s":
        s_, f_ = split_plan(x.shape[0], w.shape[0], x.shape[1])
        return gemm4w(x, w, var=64, splits=s_, split_from=f_, **kw)
    return gemm4w(x, w, bn=192 if b == "g4n192" else 256, var=64 if b == "g4p" else 0, **kw)


def linear(x: torch.Tensor, w: torch.Tensor, ws=None) -> torch.Tensor:
    """x [M, K] . w[N, K]^T -> [M, N] bf16 on the chosen backend."""
    M, K = x.shape
    N = w.shape[0]
    b, ws = _backend(x, w, "plain", ws)
    if _own_ok(b, x, N, K, "plain"):
        return _own(b, x, w, ws)
    return F.linear(x, w)


def linear_add_(x: torch.Tensor, w: torch.Tensor, acc: torch.Tensor, ws=None) -> torch.Tensor:
    """acc += x [M, K] . w[N, K]^T in place (the residual-stream update of the o / down projections):
    hipBLASLt with beta = 1 (C = D = acc, one fp32 sum and one rounding), or gemm8p's residual
    epilogue writing over its residual operand (every output element is read and written by the same
    lane).  Saves the separate residual add's read and write of the [M, N] projection output."""
    M, K = x.shape
    N = w.shape[0]
    b, ws = _backend(x, w, "residual", ws, acc)
    if _own_ok(b, x, N, K, "residual") and acc.is_contiguous() and (b not in ("g2", "gv") or acc.data_ptr() % 16 == 0):
        return _own(b, x, w, ws, residual=acc, out=acc)
    return acc.addmm_(x, w.t())


def swiglu(x: torch.Tensor, w_gu: torch.Tensor, block: int, ws=None) -> torch.Tensor:
    """silu(x Wg^T) * (x Wu^T) [M, F] for a fused gate|up weight [2F, K] whose rows are [gate; up]
    (block 0) or interleaved in blocks of ``block`` (ops.swiglu_interleave; required by g8)."""
    M, K = x.shape
    N = w_gu.shape[0]
    b, ws = _backend(x, w_gu, "swiglu", ws)
    if block == 32 and _own_ok(b, x, N, K, "swiglu"):
        return _own(b, x, w_gu, ws, swiglu=True)
    return silu_mul(F.linear(x, w_gu), block=block)


STEP_ROWS = 64


def step_core(x: torch.Tensor, w: torch.Tensor, epi: str) -> int:
    """The core of a decode step's projection as ``ops.step_project`` and ``ops.step_qkv`` number them, 0 where the choice at
    these sizes is another one (the library; a shape no one tuned)."""
    M, N = x.shape[0], w.shape[0]
    b = choice(M, N, x.shape[1], epi)
    return _NATIVE.get(b, 0) if M <= STEP_ROWS and _own_ok(b, x, N, x.shape[1], epi) else 0


def _m_bucket(M: int) -> int:
    """Encoder token counts vary per call: tune per power-of-two bucket (everything >= 64k tokens is one)."""
    return min(1 << max(M - 1, 1).bit_length(), 1 << 16)


def linear_bias(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor, gelu: bool = False, ws=None) -> torch.Tensor:
    """x . w^T + b (optionally GELU) — the encoder projections.  g8 applies the bias / exact-erf GELU in
    its epilogue on the fp32 accumulators; blas is hipBLASLt with the bias, and for GELU its bias+GELU
    epilogue (``torch._addmm_activation``: the tanh form of GELU on the fp32 accumulator, max 8.1e-3 from
    the fp32 erf-GELU at the bge-large FFN1 shape — the bf16 output's own rounding, 7.8e-3 for gemm8p's
    exact erf — where GEMM + the K9b bias_gelu pass rounds twice, 1.6e-2, and runs 657 vs 510 us at
    65536 tokens: scripts/gelu_epilogue_probe.py).  The backend is chosen per (token bucket, N, K,
    epilogue) by timing the library and the hand-written cores (:data:`ENC_BACKENDS`: gemm8p, gemm2w, the weight
    stream, ...) that take the call, on the first one."""
    M, K = x.shape
    N = w.shape[0]
    epi = "bias_gelu" if gelu else "bias"
    key = (_m_bucket(M), N, K, epi)
    c = MODE if MODE in ENC_BACKENDS else _CHOICE.get(key)
    blas = (lambda: torch._addmm_activation(b, x, w.t(), use_gelu=True)) if gelu else (lambda: F.linear(x, w, b))
    if c is None:
        if not (x.is_cuda and x.stride(1) == 1 and _g8_ok(N, K, epi)) or torch.cuda.is_current_stream_capturing():
            c = "blas"
        else:
            runs = {"blas": blas}
            runs.update({n: (lambda n=n: _own(n, x, w, ws, bias=b, gelu=gelu)) for n in ENC_BACKENDS[1:] if _enc_ok(n, x, w, epi, b)})
            c = _pick(key, runs, x)
        _CHOICE[key] = c
    # (a choice made for the token bucket may name a core that does not take this call: a 2 GiB A, an odd alignment)
    return _own(c, x, w, ws, bias=b, gelu=gelu) if c != "blas" and _enc_ok(c, x, w, epi, b) else blas()


ENC_BACKENDS = ("blas", "g4", "g4p", "g8", "gv", "g2")
_NATIVE = {"gv": 1, "g2": 2}
_ENC_NATIVE = {**_NATIVE, "g8": 3}


def encoder_cores(M: int, projections) -> Optional[list]:
    """The cores of an encoder layer's projections ((weight, its bias or None where it adds into the stream, epilogue
    name) each) at M rows as ``ops.encoder_layers`` numbers them, 0 the library (``ops.encoder_layers_mixed``); None until all are
    timed, or if one's choice is another core or does not take the call."""
    out = []
    for w, b, epi in projections:
        N, K = w.shape
        c = MODE if MODE in ENC_BACKENDS else _CHOICE.get((_m_bucket(M), N, K, epi))
        if c == "blas":
            out.append(0)
            continue
        n = _ENC_NATIVE.get(c)
        if n is None or not _g8_ok(N, K, epi) or c in EXCLUDE:
            return None
        if not (SKINNY and skinny_ok(M, N, K) if n == 1 else M * K < 1 << 30 if n == 3 else M <= G2_ROWS and gemm2w_ok(N, K, w, b)):
            return None
        out.append(n)
    return out


def _enc_ok(n: str, x: torch.Tensor, w: torch.Tensor, epi: str, other: torch.Tensor) -> bool:
    """Whether core ``n`` takes an encoder projection (``other``: its bias, or the stream it adds into)."""
    N, K = w.shape
    if not x.is_cuda or not _own_ok(n, x, N, K, epi):
        return False
    if n == "g8":  # addresses A through one 32-bit buffer range (gemm4w runs an A of 2 GiB or more as row blocks)
        return x.shape[0] * x.stride(0) * 2 < (1 << 31)
    return n != "g2" or gemm2w_ok(N, K, w, other)


# gemm8p is taken for an encoder's projection where it leads by this much: a stack runs at the clock that its power leaves, where gemm8p
# falls 2 to 5 % behind what :func:`_time_between` gives.  Its time there over the library's (in medians of 20 calls and more; in the
# few calls of now up to 0.05 less), and what a pass changes by with gemm8p for that projection alone, at 32 projections of stacks of 9600 to 102400 tokens: up to 0.92 (9 projections) -0.5 to -6.5 % of the pass; 0.95 to
# 1.00 (7) -1.4 to +2.7 %, four of them slower; above 1.00 +0.5 to +8.3 %, but two.  (Seven samples a core, in one round, gave 0.88 to 0.92
# for three projections that slow the pass by 1.5 to 2.7 %: bge-large on 38400 tokens 23.4 -> 24.4 ms.)
# FFN1 with its GELU asks for none: the library's is the tanh form (:func:`linear_bias`), the exact one is taken where it is as fast.
# With gemm8p's at 0.95 to 1.00 of the library's time a pass takes 0.98 to 0.995 of it (bge-base on 10145, 16384, 101197 and 524288 tokens,
# bge-large on 98705), 1.00 (7132) and 1.016 (38400).
G8_LEAD = 0.9


def _pick(key, runs, x: torch.Tensor) -> str:
    # (twice round: the first that a process times runs slow, the library's 233 us a call that takes 201 the next time)
    t = {name: _time_between(fn, x) for name, fn in runs.items()}
    t = {name: min(t[name], _time_between(fn, x)) for name, fn in runs.items()}
    TIMINGS[key] = t
    lead = 1.0 if key[-1] == "bias_gelu" else G8_LEAD
    if "g8" in t and t["g8"] > lead * min(t[n] for n in t if n != "g8"):
        t = {n: v for n, v in t.items() if n != "g8"}
    # (a tie goes to an own core that is launched from native code: bge-large on 7156 tokens with qkv at 52 us on the library and 53 on
    # gemm2w: 6.31 ms with the library's, 6.08 with gemm2w's.  Where the layer is not launched so, choose_encoder takes it back)
    return min((n for n in t if n != "blas" and t[n] <= t["blas"] * ((1.03 if n in _ENC_NATIVE else 1.0) + OWN_MARGIN)),
               key=lambda n: t[n], default="blas")


def choose_encoder(x: torch.Tensor, projections) -> None:
    """Choose the cores of an encoder layer's projections (as :func:`encoder_cores` takes them) for rows like ``x`` before the first
    of them runs, each by its time; a core that is no faster than the library is kept only if all four are launched from native code, or
    for its exact GELU."""
    keys = [(_m_bucket(x.shape[0]), *w.shape, epi) for w, _, epi in projections]
    if MODE in ENC_BACKENDS or all(k in _CHOICE for k in keys) or not x.is_cuda or torch.cuda.is_current_stream_capturing():
        return
    y = x
    for i, (w, b, epi) in enumerate(projections):
        a = y if i == 3 else x   # (down reads what up gives)
        y = linear_residual_(a, w, x.clone()) if b is None else linear_bias(a, w, b, gelu=epi == "bias_gelu")
    if not all(_CHOICE[k] in _ENC_NATIVE for k in keys):
        for k in keys:
            t = TIMINGS.get(k)
            if t and k[-1] != "bias_gelu" and t.get(_CHOICE[k], 0) > t["blas"] * (1 + OWN_MARGIN):
                _CHOICE[k] = "blas"


def linear_residual_(x: torch.Tensor, w: torch.Tensor, acc: torch.Tensor, ws=None) -> torch.Tensor:
    """acc += x . w^T in place — the post-LN encoder's o / FFN2 projections with the residual stream added in
    the GEMM epilogue (their bias then enters the LayerNorm that follows as its pre-norm bias, so that norm
    reads one [M, d] tensor instead of two).  Backend per (token bucket, N, K), timed on the first call on a
    copy of acc: hipBLASLt with beta = 1 (``addmm_``), gemm4w's residual epilogue (VAR 32 / 64) or gemm8p's."""
    M, K = x.shape
    N = w.shape[0]
    key = (_m_bucket(M), N, K, "enc_residual")
    c = MODE if MODE in ENC_BACKENDS else _CHOICE.get(key)
    takes = lambda n: acc.is_contiguous() and _enc_ok(n, x, w, "residual", acc)
    if c is None:
        if not (x.is_cuda and x.stride(1) == 1 and _g8_ok(N, K, "residual") and acc.is_contiguous()) or \
                torch.cuda.is_current_stream_capturing():
            c = "blas"
        else:
            a = acc.clone()  # the timing runs add into a copy, never into the stream
            runs = {"blas": lambda: a.addmm_(x, w.t())}
            runs.update({n: (lambda n=n: _own(n, x, w, ws, residual=a, out=a)) for n in ENC_BACKENDS[1:] if takes(n)})
            c = _pick(key, runs, x)
            del a, runs
        _CHOICE[key] = c
    return _own(c, x, w, ws, residual=acc, out=acc) if c != "blas" and takes(c) else acc.addmm_(x, w.t())


def _time(fn, iters: int = 5, rounds: int = 3) -> float:
    fn()
    torch.cuda.synchronize()
    ts = []
    for _ in range(rounds):
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for _ in range(iters):
            fn()
        e.record()
        torch.cuda.synchronize()
        ts.append(s.elapsed_time(e) / iters * 1e3)
    return sorted(ts)[len(ts) // 2]


def _time_between(fn, x: torch.Tensor, n: int = 7) -> float:
    """Median time of ``fn`` with a pass over its rows ``x`` before each call, as in a stack, where another kernel comes between
    any two of them: calls of one kernel in a row run on each other's heels (FFN1 of bge-base on 16391 rows, gemm8p and the
    library: 87 and 93 us a call in a row, 105 and 105 with a pass between them, 107 and 95 in the stack).  Of ``n`` calls behind
    the first, 3 where that takes a millisecond: a request waits for them (with 7 to 40, behind four: the first pass of bge-large on 38400
    tokens 176 ms, so 60, of bge-base on 524288 429 and 227, of bge-small on 1661 45 and 10; gemm8p's time over the library's up to 0.05 higher)."""
    def calls(n: int) -> list:
        marks = []
        for _ in range(n):
            x.sum()
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            fn()
            e.record()
            marks.append((s, e))
        torch.cuda.synchronize()
        return sorted(s.elapsed_time(e) for s, e in marks)
    times = calls(3 if calls(1)[0] > 1 else n)
    return times[len(times) // 2] * 1e3


def _evict_buffer(device) -> Optional[torch.Tensor]:
    """Twice the last-level cache to read between timed calls; None where the device has no room for it.  (Its block stays with
    torch's allocator for the next shape, or whatever else is allocated.)"""
    try:
        return torch.ones(1 << 27, device=device)
    except torch.cuda.OutOfMemoryError:
        return None


def _time_step(fn, x: torch.Tensor, evict: torch.Tensor, iters: int = 5) -> float:
    """Mean time of ``fn`` as a step finds its operands: the weights passed through by a read of ``evict``, the rows ``x`` just
    touched.  (The read also keeps the device busy while the host enqueues the call.)"""
    marks = []
    for _ in range(iters):
        evict.sum()
        x.clone()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        fn()
        e.record()
        marks.append((s, e))
    torch.cuda.synchronize()
    return sum(s.elapsed_time(e) for s, e in marks) / iters * 1e3


def tune(x: torch.Tensor, w: torch.Tensor, epi: str = "plain", block: int = 0, ws=None,
         bucket: bool = False) -> Optional[str]:
    """Time every applicable backend for this (M, N, K, epi) and record the choice (no-op under graph
    capture, off the GPU, for an already tuned shape, or when a backend is forced).  Rounds interleave the
    backends (one process, one device: their clock and cache states match).  ``bucket``: also the choice of
    every row count up to M not tuned exactly (down to the next smaller bucket)."""
    M, K = x.shape
    N = w.shape[0]
    key = (M, N, K, epi)
    if MODE != "auto" or not x.is_cuda or torch.cuda.is_current_stream_capturing():
        return _CHOICE.get(key)
    if key in _CHOICE:
        if bucket:
            _add_bucket(M, N, K, epi, _CHOICE[key])
        return _CHOICE[key]
    lo = None
    if bucket:
        # a bucket's choice serves every row count down to the next smaller bucket: time at its top and at the
        # middle of its range (256-row-tile cores cost in whole m-tiles, the library more smoothly; a choice
        # timed at the top alone took a split-K core that lost at the bucket's smaller row counts)
        prev = max((mb for mb, _ in _BUCKETS.get((N, K, epi), []) if mb < M), default=M // 2)
        lo = max(1, (prev + M) // 2)
        lo = lo if lo < M else None
    c = _tune(x, w, epi, block, ws, M, N, K, key, lo)
    if bucket:
        _add_bucket(M, N, K, epi, c)
    return c


def _add_bucket(M: int, N: int, K: int, epi: str, c: str) -> None:
    bl = _BUCKETS.setdefault((N, K, epi), [])
    if all(mb != M for mb, _ in bl):
        bl.append((M, c))
        bl.sort()


def _tune(x, w, epi, block, ws, M, N, K, key, lo=None) -> str:
    """``lo``: also time every backend at that row count (the bucket's middle); the choice minimises the sum."""
    if not _g8_ok(N, K, epi) or (epi == "swiglu" and block != 32):
        _CHOICE[key] = "blas"
        return "blas"
    acc = torch.zeros(M, N, dtype=x.dtype, device=x.device) if epi == "residual" else None

    def run(b, xx):
        aa = acc[:xx.shape[0]] if acc is not None else None
        if epi == "swiglu":
            return (lambda: silu_mul(F.linear(xx, w), block=block)) if b == "blas" else \
                (lambda: _own(b, xx, w, ws, swiglu=True))
        if epi == "residual":
            return (lambda: aa.addmm_(xx, w.t())) if b == "blas" else \
                (lambda: _own(b, xx, w, ws, residual=aa, out=aa))
        return (lambda: F.linear(xx, w)) if b == "blas" else (lambda: _own(b, xx, w, ws))

    runs = {}
    for b in BACKENDS:
        if b != "blas" and not _own_ok(b, x, N, K, epi):
            continue
        if b == "g4s" and (M < 256 or split_plan(M, N, K)[0] == 1 or lo is not None):
            # (unsplit at the top it is g4p.)  Not for the mixed steps' row-count buckets: timed 3-7 % ahead of
            # g4p at the buckets' rows, it ran the serving load's mixed steps 0.6-2 % slower (profiles/round6_ab.md)
            continue
        fns = [run(b, x)]
        if lo is not None:
            if b != "blas" and not _own_ok(b, x[:lo], N, K, epi):
                continue  # a backend must take the whole bucket
            fns.append(run(b, x[:lo]))
        runs[b] = fns
    # A decode step reads each layer's weight from memory (the last-level cache holds 256 MB, a step's weights are more);
    # repeated calls find it cached, and that favours the cores that read it more often: 4096 rows x 6144 x 4096 took
    # gemm2w 164 us against 169 of gemm8p there, and 180 against 172 in the step.
    evict = _evict_buffer(x.device)
    if evict is None:
        WARM.add(key)
        log.warning("no room for 512 MB: GEMM %dx%dx%d:%s timed on cached weights", M, N, K, epi)
    rows = (x, x if lo is None else x[:lo])
    ts = {b: [] for b in runs}
    # 5 interleaved rounds of 5 calls: o and gate|up are within 1-3 % between backends, and 3 x 3 calls
    # flipped the choice from run to run (profiles/bench_r64_round3.md); runs before graph capture only
    for _ in range(5):
        for b, fns in runs.items():
            ts[b].append(sum(_time(fn, iters=5, rounds=1) if evict is None else _time_step(fn, r, evict) for fn, r in zip(fns, rows)))
    med = {b: sorted(t)[len(t) // 2] for b, t in ts.items()}
    TIMINGS[key] = med
    own = min((b for b in med if b != "blas"), key=lambda b: med[b], default=None)
    _CHOICE[key] = own if own is not None and med[own] <= med["blas"] * (1 + OWN_MARGIN) else "blas"
    return _CHOICE[key]


def table() -> Dict[str, Dict[str, float]]:
    """Measured shapes -> {backend: us, 'choice': ..., 'weights': 'cached' where the timing found them in the caches for want of
    room} (for logs and /metrics)."""
    return {f"{M}x{N}x{K}:{e}": dict(TIMINGS.get((M, N, K, e), {}), choice=c, **({"weights": "cached"} if (M, N, K, e) in WARM else {}))
            for (M, N, K, e), c in _CHOICE.items()}
