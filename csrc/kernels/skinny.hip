// K6 skinny projection GEMM for small row counts: C[M, N] = A[M, K] . W[N, K]^T (+ residual, + bias, + bias and
// exact-erf GELU, or SwiGLU), bf16 in / out, fp32 accumulation.
//
// At a serving decode step (a few to 64 sequences) every projection is a weight stream: o (N = K = 4096)
// reads 33.5 MB of W for 0.5 MFLOP per weight row.  The 256 x 256-tile cores (gemm4w / gemm8p) leave all
// but M / 256 of their tile idle and run one tile per 256 W rows (16 workgroups for o: 10x the library's
// time), and hipBLASLt's kernels at these shapes read W at 1.7-2.5 TB/s (o / qkv at M <= 64,
// `scripts/serve_load.py` planner table).  Here the weight stream is the whole design:
//
//   * one workgroup per 16 W rows (N / 16 workgroups: 256 for o, 384 for qkv), 8 waves each owning 1/8 of K
//     (split-K inside the workgroup: no atomics, no second pass, a fixed summation order);
//   * per wave, batches of U k-steps of 32: U 16-byte W loads (lane (r16, g): row r16, k 8g..8g+7 of the
//     step) and U x MT activation loads (A is a few KB-MB, L2-resident) issued back to back, then U x MT
//     `v_mfma_f32_16x16x32_bf16` with W as the A operand and the activations as the B operand, so the
//     accumulator of lane (r16, q) holds output row 16 mt + r16, columns n0 + 4q .. 4q + 3 (4 consecutive
//     output columns: one 8-byte store, one 8-byte residual load);
//   * the 8 waves' partial tiles meet in LDS (8 x MT x 1 KiB) and MT waves finish: sum in wave order,
//     + residual / bias (GELU) (or SwiGLU of the gate and up tiles, EPI 2), bf16, store.
// Rows past M read zeros (buffer offsets past the activation resource's end) and are not stored.  Rows past 64 go in
// chunks of 64 over grid y (encoders: a few texts, whose weights stay in the caches).
//
// K is cut into steps of 32, ceil(K / 256) of them per wave; the FULL build (K % 2048 == 0, every wave the same even
// number of whole batches) has no masks, the other sends the steps past a wave's share to offsets past the resources'
// ends, which load zeros without a memory request.  A bge-small text of 12 tokens (K 384 / 1536, N 384 .. 1536): the
// 256-row tiles ran 8 workgroups, 14.3 us plain and 22.1 us with GELU; here 3.3 and
// 3.4 us (hipBLASLt 3.8, with 2-3 times the host time per call); from 64 rows on the library catches up (activations
// are read once per 16 columns), which the planners' timings see.
//
// Requires K % 32 == 0, N % 16 == 0, lda / ldc % 4 == 0; the planners (ops/gemm_plan.py, backend "gv") time it against
// hipBLASLt per decode bucket and per encoder token bucket.
#include "common.h"
#include "step_fuse.h"

namespace lwc {
namespace skinny {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int KS = 8;  // waves per workgroup (split-K)

LWC_DEVICE float4v mfma(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

struct Params {
  const bf16_t* A;
  const bf16_t* W;
  bf16_t* C;
  const bf16_t* R;  // residual [M, ldc] (EPI 1) — may alias C; bias [N] (EPI 3, 4)
  int M, N, K, lda, ldc;
  RowSumsq ss;  // NORM: read by EPI 0, 2, 5, written by EPI 1
  RopeKV kv;    // EPI 5
};

// NW weight tiles of 16 rows per workgroup, on the same activation fragments: EPI 2 (SwiGLU, W = [gate; up]
// interleaved in blocks of 32 rows, ops.swiglu_interleave) takes its 16 output columns' gate rows 64 (x / 2) +
// 16 (x % 2) + [0, 16) and the up rows 32 further (NW = 2); the plain / residual forms take 16 (NW = 1) or 32
// adjacent output columns (NW = 2: half the workgroups, so half the activation re-reads from L2 — past 16
// rows those loads, M / 16 times the weight bytes, are what limits the NW = 1 form)
// EPI 5 (the qkv projection of a decode step, step_fuse.h): the two tiles are the halves of a head that rotate together.
// NORM: the folded RMSNorm of step_fuse.h.
template <int MT, int EPI, int NW, bool FULL, bool NORM>
__global__ void __launch_bounds__(512) skinny_kernel(Params p) {
  constexpr int U = 4;  // k-steps per load batch (FULL: nb = K / 1024 batches, even for K % 2048 == 0)
  static_assert((EPI != 2 && EPI != 5) || NW == 2, "SwiGLU pairs a gate and an up tile, RoPE the halves of a head");
  const int TS = EPI == 2 ? 32 : EPI == 5 ? p.kv.D / 2 : 16;  // W rows between the NW tiles
  __shared__ float4v red[KS][NW][MT][64];
  __shared__ float rowscale[NORM ? MT * 16 : 1];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int strips = EPI == 5 ? p.kv.D / 32 : 1;  // (EPI 5: workgroups per head)
  const int n0 = EPI == 5 ? blockIdx.x / strips * p.kv.D + blockIdx.x % strips * 16
                          : blockIdx.x * (EPI == 2 ? 16 : 16 * NW);  // first output column
  const int wrow = EPI == 2 ? 64 * (blockIdx.x >> 1) + 16 * (blockIdx.x & 1) : n0;  // first W row
  const int m0 = blockIdx.y * 64;   // this chunk's first row
  const int M = min(p.M - m0, 64);
  const int steps = p.K / 32, per = (steps + KS - 1) / KS;   // this wave's k-steps: [w per, w per + cnt)
  const int cnt = max(0, min(per, steps - w * per));
  const int nb = FULL ? per / U : ((per + U - 1) / U + 1) & ~1;   // load batches, an even number
  const int k0 = w * per * 32;
  const __amdgpu_buffer_rsrc_t rW = uniform_rsrc(p.W + (size_t)wrow * p.K, (16 + TS * (NW - 1)) * p.K * 2);
  const __amdgpu_buffer_rsrc_t rA = uniform_rsrc(p.A + (size_t)m0 * p.lda, M * p.lda * 2);
  constexpr uint32_t kPast = 0x7ffffff0u;  // past every resource: loads zeros
  uint32_t voW[NW];
#pragma unroll
  for (int t = 0; t < NW; ++t) voW[t] = (uint32_t)(((r16 + TS * t) * p.K + k0 + 8 * g) * 2);
  // (rows past M of the last row's stride would reach past the rows' own end when lda > K: sent past the resource too)
  uint32_t voA[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) voA[mt] = mt * 16 + r16 < M ? (uint32_t)(((mt * 16 + r16) * p.lda + k0 + 8 * g) * 2) : kPast;

  float4v acc[NW][MT];
#pragma unroll
  for (int t = 0; t < NW; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = float4v{0.f, 0.f, 0.f, 0.f};
  // two register sets: batch b + 1's loads go out before batch b's MFMAs (sched_barrier keeps the compiler
  // from interleaving them into load / wait / MFMA triples, which drained the queue every batch)
  uint4v wf[2][U][NW], af[2][U][MT];
  auto load = [&](int b, uint4v(&wb)[U][NW], uint4v(&ab)[U][MT]) {
#pragma unroll
    for (int s = 0; s < U; ++s) {
      const bool in = FULL || b * U + s < cnt;    // wave-uniform
      const int so = in ? (b * U + s) * 64 : 0;   // 32 k of bf16 per step (soffset)
#pragma unroll
      for (int t = 0; t < NW; ++t)
        wb[s][t] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(rW, in ? voW[t] : kPast, so, 0));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        ab[s][mt] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(rA, in ? voA[mt] : kPast, so, 0));
    }
  };
  auto compute = [&](const uint4v(&wb)[U][NW], const uint4v(&ab)[U][MT]) {
#pragma unroll
    for (int s = 0; s < U; ++s)
#pragma unroll
      for (int t = 0; t < NW; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = mfma(wb[s][t], ab[s][mt], acc[t][mt]);
  };
  // the rows' partial sums of squares go out ahead of the first weights and are added up while those are on their way
  constexpr bool kScale = NORM && EPI != 1;
  constexpr int NR = 2 * MT;  // rows per wave
  float4v ssv[NR];
  if constexpr (kScale) {
    const __amdgpu_buffer_rsrc_t rS = uniform_rsrc(p.ss.ss + (size_t)m0 * p.ss.P, M * p.ss.P * 4);
#pragma unroll
    for (int i = 0; i < NR; ++i)
      ssv[i] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
                                               rS, 4 * lane < p.ss.P ? ((w + 8 * i) * p.ss.P + 4 * lane) * 4 : kPast, 0, 0));
  }
  RopeAhead<4> ahead;  // (waves past the m tiles and rows past M: row m0's, unused)
  if constexpr (EPI == 5) rope_kv_row(p.kv, ahead, m0 + (w < MT && w * 16 + r16 < M ? w * 16 + r16 : 0), blockIdx.x / strips);
  // straight-line pairs (no conditional loads: a load under a branch made the wait before every compute a
  // vmcnt(0)); nb is even
  load(0, wf[0], af[0]);
  if constexpr (EPI == 5) rope_kv_angles(p.kv, ahead, blockIdx.x / strips, blockIdx.x % strips * 16 + 4 * g);
  if constexpr (kScale) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const float t = wave_sum((ssv[i][0] + ssv[i][1]) + (ssv[i][2] + ssv[i][3]));
      if (lane == 0) rowscale[w + 8 * i] = rsqrtf(t / p.K + p.ss.eps);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int b = 0; b + 2 < nb; b += 2) {
    load(b + 1, wf[1], af[1]);
    __builtin_amdgcn_sched_barrier(0);
    compute(wf[0], af[0]);
    __builtin_amdgcn_sched_barrier(0);
    load(b + 2, wf[0], af[0]);
    __builtin_amdgcn_sched_barrier(0);
    compute(wf[1], af[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  load(nb - 1, wf[1], af[1]);
  __builtin_amdgcn_sched_barrier(0);
  compute(wf[0], af[0]);
  __builtin_amdgcn_sched_barrier(0);
  compute(wf[1], af[1]);
#pragma unroll
  for (int t = 0; t < NW; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[w][t][mt][lane] = acc[t][mt];
  __syncthreads();
  if (w < MT) {  // wave w finishes m-tile w: the 8 partials in wave order
    float4v sum[NW];
#pragma unroll
    for (int t = 0; t < NW; ++t) {
      sum[t] = red[0][t][w][lane];
#pragma unroll
      for (int k = 1; k < KS; ++k) sum[t] += red[k][t][w][lane];
    }
    constexpr int NO = EPI == 2 ? 1 : NW;  // 16-column output groups
    if constexpr (kScale) {
#pragma unroll
      for (int t = 0; t < NW; ++t) sum[t] *= rowscale[w * 16 + r16];
    }
    if constexpr (EPI == 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[0][e] = sum[0][e] * __builtin_amdgcn_rcpf(1.f + __expf(-sum[0][e])) * sum[1][e];
    }
    const int m = w * 16 + r16;
    if constexpr (EPI == 5) {
      if (m < M) {
        const float x[4] = {sum[0][0], sum[0][1], sum[0][2], sum[0][3]}, y[4] = {sum[1][0], sum[1][1], sum[1][2], sum[1][3]};
        rope_kv_store<4>(p.kv, ahead, p.C, p.ldc, m0 + m, blockIdx.x / strips, blockIdx.x % strips * 16 + 4 * g, x, y);
      }
    } else if (m < M) {
#pragma unroll
      for (int t = 0; t < NO; ++t) {
        const size_t off = (size_t)(m0 + m) * p.ldc + n0 + 16 * t + 4 * g;
        float v[4] = {sum[t][0], sum[t][1], sum[t][2], sum[t][3]};
        if constexpr (EPI == 3 || EPI == 4) {
          const bf16_t* b = p.R + n0 + 16 * t + 4 * g;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] += bf2f(b[e]);
            if constexpr (EPI == 4) v[e] = gelu_erf(v[e]);
          }
        }
        if constexpr (EPI == 1) {
          const uint2 rr = *reinterpret_cast<const uint2*>(p.R + off);
          v[0] += __uint_as_float(rr.x << 16);
          v[1] += __uint_as_float(rr.x & 0xffff0000u);
          v[2] += __uint_as_float(rr.y << 16);
          v[3] += __uint_as_float(rr.y & 0xffff0000u);
        }
        uint2 o;
        o.x = pack_bf16x2(v[0], v[1]);
        o.y = pack_bf16x2(v[2], v[3]);
        *reinterpret_cast<uint2*>(p.C + off) = o;
        if constexpr (EPI == 1 && NORM) {  // of the row as stored: one partial per 16 columns
          const float a = __uint_as_float(o.x << 16), b = __uint_as_float(o.x & 0xffff0000u), c = __uint_as_float(o.y << 16),
                      d = __uint_as_float(o.y & 0xffff0000u);
          const float t2 = row_sum4((a * a + b * b) + (c * c + d * d));
          if (g == 0) p.ss.ss[(size_t)(m0 + m) * p.ss.P + n0 / 16 + t] = t2;
        }
      }
    }
  }
}

template <int EPI, int NW, bool FULL, bool NORM>
int launch_full(const Params& p, hipStream_t s) {
  const int mt = (min(p.M, 64) + 15) / 16;
  const dim3 grid(EPI == 2 ? p.N / 32 : p.N / (16 * NW), (p.M + 63) / 64);  // SwiGLU: N / 2 output columns, 16 per workgroup
  switch (mt) {
    case 1: skinny_kernel<1, EPI, NW, FULL, NORM><<<grid, 512, 0, s>>>(p); break;
    case 2: skinny_kernel<2, EPI, NW, FULL, NORM><<<grid, 512, 0, s>>>(p); break;
    case 3:
    case 4: skinny_kernel<4, EPI, NW, FULL, NORM><<<grid, 512, 0, s>>>(p); break;
    default: return -1;
  }
  return (int)hipGetLastError();
}

template <int EPI, int NW, bool NORM>
int launch_nw(const Params& p, hipStream_t s) {
  return p.K % 2048 == 0 ? launch_full<EPI, NW, true, NORM>(p, s) : launch_full<EPI, NW, false, NORM>(p, s);
}

// plain / residual: 32 output columns per workgroup past 16 rows when that still leaves >= 192 workgroups
// (M / 16 activation re-reads halved: qkv at M = 32 23.9 -> 17.9 us), else 16 (o, N = 4096: 128 workgroups
// of 32 columns ran 17.6 us against 13.8 with 256 of 16 — too little of the weight stream in flight)
template <int EPI, bool NORM = false>
int launch(const Params& p, hipStream_t s) {
  if constexpr (EPI == 2 || EPI == 5) {
    return launch_nw<EPI, 2, NORM>(p, s);
  } else {
    if (p.M > 16 && p.N % 32 == 0 && p.N / 32 >= 192) return launch_nw<EPI, 2, NORM>(p, s);
    return launch_nw<EPI, 1, NORM>(p, s);
  }
}

}  // namespace skinny
}  // namespace lwc

// C = A . W^T (epi 0), R + A . W^T (epi 1; R may be C), silu(A . Wg^T) * (A . Wu^T) over a 32-row gate/up interleaved
// W [N, K] (epi 2, C [M, N / 2]), A . W^T + bias (epi 3; R = bias [N]) or gelu(A . W^T + bias) (epi 4) for M <= 256 rows;
// epi 5: the qkv projection with k and v written into the paged cache (kv).  ss: the folded RMSNorm (epi 0, 2 and 5 scale
// their rows by it, epi 5 always; epi 1 writes N / 16 partials per row).  -1: shape not taken.
extern "C" int lwc_skinny_gemm(const void* A, const void* W, void* C, const void* R, int M, int N, int K, int lda,
                               int ldc, int epi, const lwc::RowSumsq* ss, const lwc::RopeKV* kv, hipStream_t s) {
  using namespace lwc::skinny;
  const int NC = epi == 2 ? N / 2 : epi == 5 && kv != nullptr ? kv->Hq * kv->D : N;
  if (M < 0 || M > 256 || K < 32 || K % 32 != 0 || N % (epi == 2 ? 64 : 16) != 0 || lda % 4 != 0 || ldc % 4 != 0 ||
      lda < K || ldc < NC)
    return -1;
  if (epi < 0 || epi > 5) return -1;
  if ((epi == 1 || epi == 3 || epi == 4) && R == nullptr) return -1;
  if (ss != nullptr && (epi == 3 || epi == 4 || ss->P < 4 || ss->P % 4 != 0 || ss->P > 256 || (epi == 1 && ss->P != N / 16))) return -1;
  if (epi == 5 && (ss == nullptr || kv == nullptr || !lwc::rope_kv_ok(*kv, N))) return -1;
  if ((long long)(16 + (epi == 5 ? kv->D / 2 : 32)) * K * 2 >= 0x7ffffff0LL || (long long)64 * lda * 2 >= 0x7ffffff0LL) return -1;
  if (M == 0 || N == 0) return 0;
  Params p{(const lwc::bf16_t*)A, (const lwc::bf16_t*)W, (lwc::bf16_t*)C, (const lwc::bf16_t*)R, M, N, K, lda, ldc,
           ss != nullptr ? *ss : lwc::RowSumsq{}, kv != nullptr ? *kv : lwc::RopeKV{}};
  if (ss != nullptr) switch (epi) {
    case 0: return launch<0, true>(p, s);
    case 1: return launch<1, true>(p, s);
    case 2: return launch<2, true>(p, s);
    default: return launch<5, true>(p, s);
  }
  switch (epi) {
    case 0: return launch<0>(p, s);
    case 1: return launch<1>(p, s);
    case 2: return launch<2>(p, s);
    case 3: return launch<3>(p, s);
  }
  return launch<4>(p, s);
}
