// Layers of a post-norm encoder over few packed rows (a search query, a handful of short texts), four or five kernels a layer.
//
// A text of 12 tokens through bge-small is 12 layers of 7 dependent kernels of 3 to 5 us each over 42 MB of weights: what
// counts is how many there are, and what each waits for.  Here the rows' LayerNorm is computed again by every workgroup of the
// projection that reads them, under the wait for its weights (1 to 2 us, a kernel of its own 2.7), and in the narrow stack a
// head's projection and its attention are one workgroup's:
//
//   qkv_attn   x = LN(pre) (first layer: LN(word[ids] + pos[positions])); q, k, v of head h = x . W^T + b; a_h = softmax(q k^T) v
//              (wider than 384: project and the packed attention; a head's 400 KB of weights are 20 us for one compute unit)
//   project    o = a . Wo^T
//   project    y = LN(o + bo + x); h = gelu(y . W1^T + b1)
//   project    PF parts of h . W2^T, a range of K each; pre = their sum + b2 + y, fp32, is formed by the norm that reads it
//
// and a last LN.  One MI355X, a call of `embed`, us, the general layers against these: bge-small 12 tokens 400 / 266, 32 tokens
// 446 / 332; bge-base 449 / 331, 527 / 412; bge-large 931 / 742, 1172 / 980.  A part of the sum read more is 0.3 to 1 us for
// every workgroup, the halves of a long K 1 us less: two parts at 384, four at 768 and at 1024 up to 16 rows (742 against 785),
// two beyond (980 against 1412, whose rows in registers spill).
//
// project: one workgroup per 16 output columns, 8 waves over K in steps of 32 (wave w: steps w, w + 8, ..), W the A operand
// and the rows the B operand of mfma_f32_16x16x32_bf16, so that a lane holds four consecutive columns of one row.  qkv_attn: one
// workgroup per head, 24 (16 columns, part of K) units over 8 waves.  Sums over waves, units and parts in a fixed order.  Rows
// go in MT tiles of 16; rows past T are zeros and are not stored.
#include "common.h"

extern "C" int lwc_prefill_attention(const void* q, const void* k, const void* v, void* out, const int* cu_q, const int* cu_k, int nseq,
                                     int rows, int max_seqlen, int ldq, int ldk, int ldv, int ldo, int Hq, int Hkv, int D,
                                     float scale, int causal, hipStream_t s);

namespace lwc {
namespace efew {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

constexpr int kT = 512, kW = kT / 64;

LWC_DEVICE float4v mfma(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

struct Norm {
  const float* part;     // [P, T, D]: the parts of what the last projection gave
  const bf16_t* res;     // [T, D] and
  const bf16_t* rbias;   // [D]: the stream and the projection's bias, added to them
  const bf16_t* word;    // [V, D]: the embeddings where part is null
  const bf16_t* pos;     // [NP, D]
  const int* ids;        // [T]
  const int* positions;  // [T]
  int V, NP;
  const bf16_t* g;       // [D]
  const bf16_t* b;
  float eps;
  bf16_t* out;           // [T, D], written by workgroup 0 (not res: others may still read it)
};

LWC_DEVICE float4v widen4(const uint2v& v) {
  return float4v{__uint_as_float(v[0] << 16), __uint_as_float(v[0] & 0xffff0000u), __uint_as_float(v[1] << 16),
                 __uint_as_float(v[1] & 0xffff0000u)};
}
LWC_DEVICE uint2v narrow4(const float4v& v) { return uint2v{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}; }

// The rows' LayerNorm into LDS, [16 MT][D + 8] (the pad spreads 16 rows' fragments over the banks), one wave per row.  Its loads
// come first, in one trip where P * RPW * C allows; `weights` issues the caller's behind them, whose data come later (loads
// return in order: ahead of the rows', the weights from memory would be what the norm waits for).
template <int MT, int D, int P, class F>
LWC_DEVICE void norm_rows(const Norm& n, int T, bf16_t* xs, const F& weights) {
  constexpr int RPW = 16 * MT / kW, C = (D / 4 + 63) / 64, PB = RPW * C * P <= 32 ? P : RPW * C * 2 <= 32 ? 2 : 1;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float4v v[RPW][C];
  uint2v g[C], b[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int at = min((c * 64 + lane) * 4, D - 4);
    g[c] = *reinterpret_cast<const uint2v*>(n.g + at);
    b[c] = *reinterpret_cast<const uint2v*>(n.b + at);
  }
  if (n.part) {
    uint2v r[RPW][C], rb[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int at = min((c * 64 + lane) * 4, D - 4);
      rb[c] = *reinterpret_cast<const uint2v*>(n.rbias + at);
#pragma unroll
      for (int i = 0; i < RPW; ++i)
        r[i][c] = *reinterpret_cast<const uint2v*>(n.res + (size_t)min(w + i * kW, T - 1) * D + at);
    }
#pragma unroll
    for (int p0 = 0; p0 < P; p0 += PB) {
      float4v t[PB][RPW][C];
#pragma unroll
      for (int q = 0; q < PB; ++q)
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
          for (int c = 0; c < C; ++c)
            if (w + i * kW < T)
              t[q][i][c] = *reinterpret_cast<const float4v*>(n.part + ((size_t)min(p0 + q, P - 1) * T + w + i * kW) * D + min((c * 64 + lane) * 4, D - 4));
            else
              t[q][i][c] = float4v{0.f, 0.f, 0.f, 0.f};
      if (p0 + PB >= P) {
        __builtin_amdgcn_sched_barrier(0);
        weights();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < PB; ++q)
#pragma unroll
        for (int i = 0; i < RPW; ++i)
#pragma unroll
          for (int c = 0; c < C; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][c][j] = p0 + q == 0 ? t[q][i][c][j] : p0 + q < P ? v[i][c][j] + t[q][i][c][j] : v[i][c][j];
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const float4v q = widen4(rb[c]);
#pragma unroll
      for (int i = 0; i < RPW; ++i) {
        const float4v x = widen4(r[i][c]);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][c][j] += q[j] + x[j];
      }
    }
  } else {
    weights();
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int row = min(w + i * kW, T - 1);
      const int id = min(max(n.ids[row], 0), n.V - 1), at_p = min(max(n.positions[row], 0), n.NP - 1);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int at = min((c * 64 + lane) * 4, D - 4);
        const float4v x = widen4(*reinterpret_cast<const uint2v*>(n.word + (size_t)id * D + at));
        const float4v e = widen4(*reinterpret_cast<const uint2v*>(n.pos + (size_t)at_p * D + at));
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i][c][j] = x[j] + e[j];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const int row = w + i * kW;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
      if ((c * 64 + lane) * 4 < D) s += (v[i][c][0] + v[i][c][1]) + (v[i][c][2] + v[i][c][3]);
    const float mean = row_sum4(row16_sum(s)) * (1.f / D);
    float s2 = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
      if ((c * 64 + lane) * 4 < D)
#pragma unroll
        for (int j = 0; j < 4; ++j) s2 += (v[i][c][j] - mean) * (v[i][c][j] - mean);
    const float inv = rsqrtf(row_sum4(row16_sum(s2)) * (1.f / D) + n.eps);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int at = (c * 64 + lane) * 4;
      if (at >= D) continue;
      const float4v gf = widen4(g[c]), bf = widen4(b[c]);
      float4v y;
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = row < T ? (v[i][c][j] - mean) * inv * gf[j] + bf[j] : 0.f;
      const uint2v o = narrow4(y);
      if (xs) *reinterpret_cast<uint2v*>(xs + row * (D + 8) + at) = o;
      if (n.out && blockIdx.x == 0 && blockIdx.y == 0 && row < T) *reinterpret_cast<uint2v*>(n.out + (size_t)row * D + at) = o;
    }
  }
}

template <int MT, int D, int P>
__global__ void __launch_bounds__(kT) norm_kernel(Norm n, int T) {
  norm_rows<MT, D, P>(n, T, nullptr, [] {});
}

struct Attn {
  Norm n;
  const bf16_t* W;  // [3 D, D]
  const bf16_t* bias;
  const int* cu;  // [nseq + 1]
  bf16_t* a;      // [T, D]
  int T, nseq;
  float scale;
};

template <int MT, int D, int DH>
struct AttnLds {
  static constexpr int TK = MT == 1 ? 32 : 16 * MT;          // keys, a multiple of the MFMA's 32
  static constexpr int kX = 16 * MT * (D + 8) * 2;
  static constexpr int kRed = 24 * MT * 1024;                // the units' partials, over the rows that they are done with
  static constexpr int kQ = kX > kRed ? kX : kRed;           // q, k [16 MT][DH + 8]; v [DH][TK + 8]; p [16 MT][TK + 8]
  static constexpr int kK = kQ + 16 * MT * (DH + 8) * 2;
  static constexpr int kV = kK + 16 * MT * (DH + 8) * 2;
  static constexpr int kP = kV + DH * (TK + 8) * 2;
  static constexpr int kBytes = kP + 16 * MT * (TK + 8) * 2;
};

template <int MT, int D, int DH, int P>
__global__ void __launch_bounds__(kT) qkv_attn_kernel(Attn p) {
  using L = AttnLds<MT, D, DH>;
  constexpr int NT = 3 * DH / 16, SPLIT = 24 / NT, KU = D / 32 / SPLIT, TK = L::TK;
  static_assert(NT * SPLIT == 24 && KU * 32 * SPLIT == D, "24 units of whole K steps");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  bf16_t* xs = reinterpret_cast<bf16_t*>(smem);
  float4v* red = reinterpret_cast<float4v*>(smem);
  bf16_t* qs = reinterpret_cast<bf16_t*>(smem + L::kQ);
  bf16_t* ks = reinterpret_cast<bf16_t*>(smem + L::kK);
  bf16_t* vs = reinterpret_cast<bf16_t*>(smem + L::kV);
  bf16_t* ps = reinterpret_cast<bf16_t*>(smem + L::kP);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, h = blockIdx.x;

  // unit u of 24: 16 columns (q, k or v's) tt = u / SPLIT, K part u % SPLIT
  auto wptr = [&](int i) {
    const int u = w * 3 + i, tt = u / SPLIT;
    const int row = tt / (DH / 16) * D + h * DH + tt % (DH / 16) * 16 + r16;
    return p.W + (size_t)row * D + u % SPLIT * KU * 32 + 8 * g;
  };
  uint4v wf[3][KU];
  uint2v bias[(NT * MT * 64 + kT - 1) / kT];
#pragma unroll
  for (int i = 0; i < (NT * MT * 64 + kT - 1) / kT; ++i) {
    const int o = min(tid + i * kT, NT * MT * 64 - 1), tt = o / 64 / MT;
    bias[i] = *reinterpret_cast<const uint2v*>(p.bias + tt / (DH / 16) * D + h * DH + tt % (DH / 16) * 16 + 4 * ((o & 63) >> 4));
  }
  const int bounds = p.cu[min(lane, p.nseq)];
  norm_rows<MT, D, P>(p.n, p.T, xs, [&] {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int s = 0; s < KU; ++s) wf[i][s] = *reinterpret_cast<const uint4v*>(wptr(i) + s * 32);
  });
  __syncthreads();
  float4v acc[3][MT];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[i][m] = float4v{0.f, 0.f, 0.f, 0.f};
    const bf16_t* xr = xs + (w * 3 + i) % SPLIT * KU * 32 + 8 * g;
#pragma unroll
    for (int s = 0; s < KU; ++s)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[i][m] = mfma(wf[i][s], *reinterpret_cast<const uint4v*>(xr + (16 * m + r16) * (D + 8) + s * 32), acc[i][m]);
  }
  __syncthreads();  // every wave is done with the rows
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((w * 3 + i) * MT + m) * 64 + lane] = acc[i][m];
  if (TK > 16 * MT)  // (MT 1) the keys past the tile: v's are zeros, and so are their probabilities
    for (int i = tid; i < DH * 16; i += kT) vs[i / 16 * (TK + 8) + 16 + i % 16] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (NT * MT * 64 + kT - 1) / kT; ++i) {
    const int o = tid + i * kT;
    if (o >= NT * MT * 64) break;
    const int ln = o & 63, m = o / 64 % MT, tt = o / 64 / MT;
    float4v y = red[((tt * SPLIT) * MT + m) * 64 + ln];
#pragma unroll
    for (int s = 1; s < SPLIT; ++s) {
      const float4v z = red[((tt * SPLIT + s) * MT + m) * 64 + ln];
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] += z[j];
    }
    const int which = tt / (DH / 16), col = tt % (DH / 16) * 16 + 4 * (ln >> 4), row = 16 * m + (ln & 15);
    const float4v b = widen4(bias[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] += b[j];
    const uint2v v = narrow4(y);
    if (which < 2) {
      *reinterpret_cast<uint2v*>((which ? ks : qs) + row * (DH + 8) + col) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) vs[(col + j) * (TK + 8) + row] = (bf16_t)(v[j >> 1] >> (16 * (j & 1)));
    }
  }
  __syncthreads();
  // Scores, transposed, a wave per 16 queries: lane (r16, g) holds query r16's keys 16 j + 4 g ..
  if (w >= MT) return;
  const int qi = 16 * w + r16;
  int lo = 0, hi = 0;  // the keys of the query's text
  for (int s = 0; s < p.nseq; ++s) {
    const int a = __builtin_amdgcn_readlane(bounds, s), b = __builtin_amdgcn_readlane(bounds, s + 1);
    if (a <= qi && qi < b) lo = a, hi = b;
  }
  float4v sc[MT];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    sc[j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DH / 32; ++s)
      sc[j] = mfma(*reinterpret_cast<const uint4v*>(ks + (16 * j + r16) * (DH + 8) + s * 32 + 8 * g),
                   *reinterpret_cast<const uint4v*>(qs + qi * (DH + 8) + s * 32 + 8 * g), sc[j]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = 16 * j + 4 * g + r;
      sc[j][r] = key >= lo && key < hi ? sc[j][r] * p.scale : -INFINITY;
      mx = fmaxf(mx, sc[j][r]);
    }
  }
  mx = row_max4(mx);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[j][r] = mx > -INFINITY ? __expf(sc[j][r] - mx) : 0.f;
      sum += sc[j][r];
    }
    *reinterpret_cast<uint2v*>(ps + qi * (TK + 8) + 16 * j + 4 * g) = narrow4(sc[j]);
  }
  if (TK > 16 * MT) *reinterpret_cast<uint2v*>(ps + qi * (TK + 8) + 16 + 4 * g) = uint2v{0u, 0u};
  sum = row_sum4(sum);
  const float inv = sum > 0.f ? 1.f / sum : 0.f;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // the wave's own rows of p
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  float4v o[DH / 16];
  float all = 0.f;
#pragma unroll
  for (int c = 0; c < DH / 16; ++c) {
    o[c] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < TK / 32; ++s)
      o[c] = mfma(*reinterpret_cast<const uint4v*>(vs + (16 * c + r16) * (TK + 8) + s * 32 + 8 * g),
                  *reinterpret_cast<const uint4v*>(ps + qi * (TK + 8) + s * 32 + 8 * g), o[c]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[c][r] *= inv;
      all = fmaf(o[c][r], 0.f, all);  // 0, or NaN
    }
  }
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(all != 0.f) != 0, 0)) {
    // an infinity or NaN among the values: a weight of zero does not keep it to its own text, so each query's keys alone
#pragma unroll
    for (int c = 0; c < DH / 16; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float t = 0.f;
        for (int key = lo; key < hi; ++key) t += bf2f(ps[qi * (TK + 8) + key]) * bf2f(vs[(16 * c + 4 * g + r) * (TK + 8) + key]);
        o[c][r] = t * inv;
      }
  }
#pragma unroll
  for (int c = 0; c < DH / 16; ++c)
    if (qi < p.T) *reinterpret_cast<uint2v*>(p.a + (size_t)qi * D + h * DH + 16 * c + 4 * g) = narrow4(o[c]);
}

enum Out { OUT_PART = 0, OUT_BIAS = 1, OUT_GELU = 2 };

struct Proj {
  Norm n;           // LN: the rows
  const bf16_t* A;  // !LN: the rows [T, lda]
  const bf16_t* W;  // [N, lda]
  const bf16_t* bias;
  float* part;      // OUT_PART: [grid y, T, N]
  bf16_t* h;        // else: [T, N]
  int T, N, lda;
};

// 16 columns of the product of K of the lda columns (the blockIdx.y-th K of them).  P > 0: the rows are normalised here, from P parts
template <int MT, int K, int P, int OUT>
__global__ void __launch_bounds__(kT) project_kernel(Proj p) {
  constexpr int S = K / 32, PER = (S + kW - 1) / kW;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float4v* red = reinterpret_cast<float4v*>(smem);
  bf16_t* xs = reinterpret_cast<bf16_t*>(smem + kW * MT * 1024);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, n0 = blockIdx.x * 16, k0 = blockIdx.y * K;
  const bf16_t* wr = p.W + (size_t)(n0 + r16) * p.lda + k0 + 8 * g;
  uint4v wf[PER];
  auto weights = [&] {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int s = w + i * kW;
      wf[i] = s < S ? *reinterpret_cast<const uint4v*>(wr + s * 32) : uint4v{0u, 0u, 0u, 0u};
    }
  };
  const int row = 16 * w + r16, col = n0 + 4 * g;  // MT of the waves finish
  uint2v bias = {0u, 0u};
  if (OUT != OUT_PART && w < MT) bias = *reinterpret_cast<const uint2v*>(p.bias + col);
  float4v acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = float4v{0.f, 0.f, 0.f, 0.f};
  if constexpr (P > 0) {
    norm_rows<MT, K, P>(p.n, p.T, xs, weights);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int s = w + i * kW;
      if (s < S)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m] = mfma(wf[i], *reinterpret_cast<const uint4v*>(xs + (16 * m + r16) * (K + 8) + s * 32 + 8 * g), acc[m]);
    }
  } else {
    weights();
    uint4v af[MT][PER];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int s = w + i * kW;
        af[m][i] = s < S && 16 * m + r16 < p.T
                       ? *reinterpret_cast<const uint4v*>(p.A + (size_t)(16 * m + r16) * p.lda + k0 + s * 32 + 8 * g)
                       : uint4v{0u, 0u, 0u, 0u};
      }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < PER; ++i) acc[m] = mfma(wf[i], af[m][i], acc[m]);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) red[(w * MT + m) * 64 + lane] = acc[m];
  __syncthreads();
  if (w >= MT) return;
  float4v y = red[w * 64 + lane];
#pragma unroll
  for (int i = 1; i < kW; ++i) {
    const float4v z = red[(i * MT + w) * 64 + lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] += z[j];
  }
  if (row >= p.T) return;
  if constexpr (OUT == OUT_PART) {
    *reinterpret_cast<float4v*>(p.part + ((size_t)blockIdx.y * p.T + row) * p.N + col) = y;
  } else {
    const float4v b = widen4(bias);
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = OUT == OUT_GELU ? gelu_erf(y[j] + b[j]) : y[j] + b[j];
    *reinterpret_cast<uint2v*>(p.h + (size_t)row * p.N + col) = narrow4(y);
  }
}

template <auto Kernel>
void lds(int bytes) {
  static const hipError_t once = hipFuncSetAttribute((const void*)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  (void)once;
}

struct Call {
  const void* const* w;
  int layers;
  const int* cu;
  int nseq, T;
  float scale;
  float* part;  // [4, T, D] (no kernel both reads and writes it)
  bf16_t *x, *y, *a, *h;
  hipStream_t s;
};

// The whole stack
template <int MT, int D, int DH>
int run(Norm n, const Call& c) {
  constexpr int F = 4 * D, H = D / DH, PF = D <= 384 || D * MT > 1536 ? 2 : 4, kRed = kW * MT * 1024, kLn = kRed + 16 * MT * (D + 8) * 2;
  static_assert(kLn <= 160 * 1024, "a compute unit's LDS");
  const int T = c.T;
  const void* const* w = c.w;
  lds<project_kernel<MT, D, 1, OUT_GELU>>(kLn);
  for (int l = 0; l < c.layers; ++l, w += 12) {
    auto t = [&](int i) { return (const bf16_t*)w[i]; };
    n.out = c.x;
    if constexpr (D <= 384) {
      constexpr int kAttn = AttnLds<MT, D, DH>::kBytes;
      static_assert(kAttn <= 160 * 1024, "a compute unit's LDS");
      lds<qkv_attn_kernel<MT, D, DH, PF>>(kAttn);
      qkv_attn_kernel<MT, D, DH, PF><<<H, kT, kAttn, c.s>>>(Attn{n, t(0), t(1), c.cu, c.a, T, c.nseq, c.scale});
    } else {
      lds<project_kernel<MT, D, PF, OUT_BIAS>>(kLn);
      project_kernel<MT, D, PF, OUT_BIAS><<<3 * D / 16, kT, kLn, c.s>>>(Proj{n, nullptr, t(0), t(1), nullptr, c.h, T, 3 * D, D});
      const int rc = lwc_prefill_attention(c.h, c.h + D, c.h + 2 * D, c.a, c.cu, c.cu, c.nseq, T, T, 3 * D, 3 * D, 3 * D, D, H, H, DH,
                                           c.scale, 0, c.s);
      if (rc != 0) return rc;
    }
    project_kernel<MT, D, 0, OUT_PART><<<D / 16, kT, kRed, c.s>>>(Proj{n, c.a, t(2), nullptr, c.part, nullptr, T, D, D});
    n.part = c.part;
    n.res = c.x;
    n.rbias = t(3);
    n.g = t(4);
    n.b = t(5);
    n.out = c.y;
    project_kernel<MT, D, 1, OUT_GELU><<<F / 16, kT, kLn, c.s>>>(Proj{n, nullptr, t(6), t(7), nullptr, c.h, T, F, D});
    project_kernel<MT, F / PF, 0, OUT_PART><<<dim3(D / 16, PF), kT, kRed, c.s>>>(Proj{n, c.h, t(8), nullptr, c.part, nullptr, T, D, F});
    n.res = c.y;
    n.rbias = t(9);
    n.g = t(10);
    n.b = t(11);
  }
  n.out = c.x;
  norm_kernel<MT, D, PF><<<1, kT, 0, c.s>>>(n, T);
  return (int)hipGetLastError();
}

}  // namespace efew
}  // namespace lwc

// Whether lwc_encoder_few takes T rows of a stack of width d, H heads and f FFN columns.
extern "C" int lwc_encoder_few_ok(int T, int d, int H, int f) {
  return T > 0 && T <= 32 && f == 4 * d && ((d == 384 && H == 12) || (d == 768 && H == 12) || (d == 1024 && H == 16));
}

// x [T, d] = the last hidden rows of `layers` layers over word[ids] + pos[positions].  w: 12 pointers a layer (qkv, its bias, o,
// its bias, norm 1 gain and bias, FFN up and bias, FFN down and bias, norm 2 gain and bias), all contiguous and 16-byte aligned.
// part [4, T, d] fp32, y and a [T, d], h [T, f]: scratch.
extern "C" int lwc_encoder_few(const void* word, const void* pos, const int* ids, const int* positions, int V, int P, const void* g,
                               const void* b, float eps, const void* const* w, int layers, const int* cu, int nseq, int T, int d,
                               int H, int f, float scale, float* part, void* x, void* y, void* a, void* h, hipStream_t s) {
  using namespace lwc::efew;
  using lwc::bf16_t;
  if (!lwc_encoder_few_ok(T, d, H, f) || nseq < 1 || nseq > 63) return -1;
  const Norm n{nullptr, nullptr, nullptr, (const bf16_t*)word, (const bf16_t*)pos, ids, positions, V, P, (const bf16_t*)g,
               (const bf16_t*)b, eps, nullptr};
  const Call c{w, layers, cu, nseq, T, scale, part, (bf16_t*)x, (bf16_t*)y, (bf16_t*)a, (bf16_t*)h, s};
#define LWC_FEW(MT, D, DH) return run<MT, D, DH>(n, c)
  if (T <= 16) {
    if (d == 384) LWC_FEW(1, 384, 32);
    if (d == 768) LWC_FEW(1, 768, 64);
    LWC_FEW(1, 1024, 64);
  }
  if (d == 384) LWC_FEW(2, 384, 32);
  if (d == 768) LWC_FEW(2, 768, 64);
  LWC_FEW(2, 1024, 64);
#undef LWC_FEW
}
