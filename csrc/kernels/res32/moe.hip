// Mixture-of-experts routing with a softmax or sigmoid router over real and identity experts (gfx950, wave64).
//
//   router_topk     s = softmax(z) over all NE router outputs (fp32); the k largest of s + correction are chosen
//                   (ties: the lower index); the weights are the chosen s, not renormalised.  Outputs beyond the
//                   first E are IDENTITY experts (their output is the token's input itself).  Counts the rows of
//                   every real expert and hands each (token, choice) its rank within its expert.
//                   Sigmoid scores instead of the softmax, and groups of neighbouring outputs of which only the best
//                   few (by the sum of their two largest scores) are open to the choice: RouterRule.
//   router_offsets  exclusive scan of the counts -> row_off [E + 1]
//   router_scatter  expert-major rows: src[row] = token, row_expert[row], inv[t*k + j] = row (-1: identity)
//   expert_rows     one workgroup per expert-major row: y = W_down act(W_gate h, W_up h), any sizes, fp32 sums; act =
//                   silu(g) u or the clamped unit g' sigmoid(alpha g') (u' + 1), g' = min(g, L), u' = clamp(u, -L, L)
//   moe_combine     out[t] = sum_j w[t][j] * (inv >= 0 ? Y[inv] : h[t]) (+ sigmoid(gate[t]) * add[t])   (fp32)
#include "elem.h"

namespace lwc {
namespace {

constexpr int kMaxPerLane = 8;  // router outputs per lane: NE <= 512
constexpr int kOneGroup = 512;   // tokens that one workgroup routes (router_one_group_kernel)

// How scores become choices and weights.
struct RouterRule {
  int sigmoid;       // scores = sigmoid(z), else the softmax over all outputs
  int renorm;        // weights = chosen scores / (their sum + floor) * scale, else chosen scores * scale
  float floor, scale;
  int groups, keep;  // groups > 1: NE / groups neighbours each; only the `keep` best groups are open
};

template <int PER>
__global__ void router_topk_kernel(const float* __restrict__ z, const float* __restrict__ corr,
                                   const float* __restrict__ bias, int ldz, RouterRule rule, int NE, int E, int k,
                                   int* __restrict__ ids, float* __restrict__ wts, int* __restrict__ counts,
                                   int* __restrict__ rank, int T) {
  const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (t >= T) return;
  const int lane = threadIdx.x & 63;
  const float* zr = z + (size_t)t * ldz;
  float v[PER], c[PER];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i;
    v[i] = e < NE ? zr[e] + (bias ? bias[e] : 0.f) : -INFINITY;
    m = fmaxf(m, v[i]);
  }
  if (rule.sigmoid) {
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = lane + 64 * i < NE ? sigmoid_f(v[i]) : 0.f;
  } else {
    m = wave_max(m);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + 64 * i;
      v[i] = e < NE ? expf(v[i] - m) : 0.f;
      sum += v[i];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = v[i] / sum;
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i;
    c[i] = e < NE ? v[i] + (corr ? corr[e] : 0.f) : -INFINITY;
  }
  if (rule.groups > 1) {  // groups' scores: group g's lives in lane g & 63, slot g >> 6
    const int size = NE / rule.groups;
    float gs[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) gs[i] = -INFINITY;
    for (int g = 0; g < rule.groups; ++g) {
      float a = -INFINITY, b = -INFINITY;  // this lane's two largest of the group, then the wave's
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        if (e >= g * size && e < (g + 1) * size) {
          b = fmaxf(b, fminf(a, c[i]));
          a = fmaxf(a, c[i]);
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float oa = __shfl_xor(a, o, 64), ob = __shfl_xor(b, o, 64);
        b = fmaxf(fmaxf(b, ob), fminf(a, oa));
        a = fmaxf(a, oa);
      }
      const float score = size > 1 ? a + b : a;
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (lane + 64 * i == g) gs[i] = score;
    }
    unsigned open = 0;  // bit i: this lane's output lane + 64 i may be chosen
    for (int j = 0; j < rule.keep; ++j) {
      float best = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (gs[i] > best) best = gs[i], bi = lane + 64 * i;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) best = ob, bi = oi;
      }
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        if (e == bi) gs[i] = -INFINITY;
        if (e >= bi * size && e < (bi + 1) * size) open |= 1u << i;
      }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (!((open >> i) & 1u)) c[i] = -INFINITY;
  }
  float chosen = 0.f;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY;
    int bi = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + 64 * i;
      if (e < NE && (c[i] > best || (c[i] == best && e < bi))) best = c[i], bi = e;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ob > best || (ob == best && oi < bi)) best = ob, bi = oi;
    }
    // the winner's lane removes it and reports its score
    float sc = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (lane + 64 * i == bi) sc = v[i], c[i] = -INFINITY;
    sc = wave_sum(sc);
    chosen += sc;
    if (lane == 0) {
      ids[(size_t)t * k + j] = bi;
      wts[(size_t)t * k + j] = sc;
      rank[(size_t)t * k + j] = bi < E ? atomicAdd(counts + bi, 1) : -1;
    }
  }
  if (lane == 0 && (rule.renorm || rule.scale != 1.0f))  // softmax, floor 0: the softmax over the chosen outputs only
    for (int j = 0; j < k; ++j) wts[(size_t)t * k + j] *= rule.scale / (rule.renorm ? chosen + rule.floor : 1.0f);
}

// This lane's rank within expert x, for a wave whose lanes hold one choice each: lane e's `next` is the rank that the first
// of them to choose expert e takes, and moves past them all.  -1 where x is no real expert or the lane is not live.
__device__ __forceinline__ int expert_rank(int x, bool live, int E, int& next) {
  const int lane = threadIdx.x & 63;
  int r = -1;
  for (int e = 0; e < E; ++e) {
    const unsigned long long m = __ballot(live && x == e);
    if (m == 0ull) continue;
    const int first = __builtin_amdgcn_readlane(next, e);
    if (live && x == e) r = first + __popcll(m & ((1ull << lane) - 1ull));
    if (lane == e) next += __popcll(m);
  }
  return r;
}

// Few router outputs (NE <= NMAX): one THREAD per token t0, the scores in registers.  Writes ids and weights and returns
// the k choices, four bits each.  mine, in lane e < E: how many choices of this wave's tokens are expert e.
template <int NMAX>
__device__ __forceinline__ unsigned long long route_token(const float* __restrict__ z, const float* __restrict__ corr,
                                                          const float* __restrict__ bias, int ldz, RouterRule rule, int NE,
                                                          int E, int k, int* __restrict__ ids, float* __restrict__ wts,
                                                          int t0, int T, int& mine) {
  static_assert(NMAX <= 16, "a choice takes four bits");
  const bool live = t0 < T;  // lanes past the last token go along (wave-wide votes below) and write nothing
  const int t = live ? t0 : T - 1;
  const float* zr = z + (size_t)t * ldz;
  float v[NMAX], c[NMAX];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < NMAX; ++i) {
    v[i] = i < NE ? zr[i] + (bias ? bias[i] : 0.f) : -INFINITY;
    m = fmaxf(m, v[i]);
  }
  if (rule.sigmoid) {
#pragma unroll
    for (int i = 0; i < NMAX; ++i) v[i] = i < NE ? sigmoid_f(v[i]) : 0.f;
  } else {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NMAX; ++i) {
      v[i] = i < NE ? expf(v[i] - m) : 0.f;
      sum += v[i];
    }
#pragma unroll
    for (int i = 0; i < NMAX; ++i) v[i] = v[i] / sum;
  }
#pragma unroll
  for (int i = 0; i < NMAX; ++i) c[i] = i < NE ? v[i] + (corr ? corr[i] : 0.f) : -INFINITY;
  if (rule.groups > 1) {
    const int size = NE / rule.groups;
    float gs[NMAX];
#pragma unroll
    for (int g = 0; g < NMAX; ++g) {
      float a = -INFINITY, b = -INFINITY;  // the group's two largest
#pragma unroll
      for (int i = 0; i < NMAX; ++i)
        if (i >= g * size && i < (g + 1) * size) {
          b = fmaxf(b, fminf(a, c[i]));
          a = fmaxf(a, c[i]);
        }
      gs[g] = g < rule.groups ? (size > 1 ? a + b : a) : -INFINITY;
    }
    unsigned open = 0;  // bit i: output i may be chosen
    for (int j = 0; j < rule.keep; ++j) {
      float best = -INFINITY;
      int bg = 0;
#pragma unroll
      for (int g = 0; g < NMAX; ++g)
        if (gs[g] > best) best = gs[g], bg = g;
#pragma unroll
      for (int g = 0; g < NMAX; ++g)
        if (g == bg) gs[g] = -INFINITY;
      open |= ((1u << size) - 1u) << (bg * size);
    }
#pragma unroll
    for (int i = 0; i < NMAX; ++i)
      if (!((open >> i) & 1u)) c[i] = -INFINITY;
  }
  float chosen = 0.f;
  unsigned long long picks = 0;
  mine = 0;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY, sc = 0.f;
    int bi = 0;
#pragma unroll
    for (int i = 0; i < NMAX; ++i)
      if (i < NE && c[i] > best) best = c[i], bi = i, sc = v[i];
#pragma unroll
    for (int i = 0; i < NMAX; ++i)
      if (i == bi) c[i] = -INFINITY;
    chosen += sc;
    picks |= (unsigned long long)bi << (4 * j);
    expert_rank(bi, live, E, mine);
    if (live) {
      ids[(size_t)t * k + j] = bi;
      wts[(size_t)t * k + j] = sc;
    }
  }
  if (live && (rule.renorm || rule.scale != 1.0f))
    for (int j = 0; j < k; ++j) wts[(size_t)t * k + j] *= rule.scale / (rule.renorm ? chosen + rule.floor : 1.0f);
  return picks;
}

// One atomic per (wave, expert): lane e takes as many ranks of expert e as its wave's tokens have chosen it, and the
// tokens take them choice by choice, in lane order.  (An atomic per wave, choice AND expert, each waited for: 16.8 us for
// 1024 tokens, top 2 of 8; 73 us for top 8 of 16.  So: 12.3 and 32 us, with the fill, offsets and scatter.)
template <int NMAX>
__global__ void router_topk_thread_kernel(const float* __restrict__ z, const float* __restrict__ corr,
                                          const float* __restrict__ bias, int ldz, RouterRule rule, int NE, int E, int k,
                                          int* __restrict__ ids, float* __restrict__ wts, int* __restrict__ counts,
                                          int* __restrict__ rank, int T) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
  int next;
  const unsigned long long picks = route_token<NMAX>(z, corr, bias, ldz, rule, NE, E, k, ids, wts, t, T, next);
  next = lane < E && next ? atomicAdd(counts + lane, next) : 0;
  for (int j = 0; j < k; ++j) {
    const int r = expert_rank((int)(picks >> (4 * j)) & 15, t < T, E, next);
    if (t < T) rank[(size_t)t * k + j] = r;
  }
}

// The whole routing of at most kOneGroup tokens in ONE workgroup: choice, counts, offsets and expert-major rows.
// Few tokens are all latency: apart, a fill, the choice, the offsets and the scatter cost 14.3 us (64 tokens, 8 of 10 outputs
// real, top 2), most of it launches and one dependent atomic in memory per choice and expert; here 6.9 us, the counts in LDS.
// kOneGroup: 512 tokens take 8.4 us here and 12.3 in three kernels, 1024 take 11.7 to 13.1 and 11.9 (16 outputs, top 8:
// 30 and 32, 41 and 29): beyond it one CU has too many waves to run one after the other.
template <int NMAX>
__global__ void __launch_bounds__(kOneGroup) router_one_group_kernel(const float* __restrict__ z, const float* __restrict__ corr,
                                                                     const float* __restrict__ bias, int ldz, RouterRule rule,
                                                                     int NE, int E, int k, int* __restrict__ ids,
                                                                     float* __restrict__ wts, int* __restrict__ row_off,
                                                                     int* __restrict__ src, int* __restrict__ row_expert,
                                                                     int* __restrict__ inv, int T) {
  __shared__ int counts[NMAX];
  const int t = threadIdx.x, lane = t & 63;
  if (t < NMAX) counts[t] = 0;
  __syncthreads();
  int next;
  const unsigned long long picks = route_token<NMAX>(z, corr, bias, ldz, rule, NE, E, k, ids, wts, t, T, next);
  next = lane < E && next ? atomicAdd(counts + lane, next) : 0;
  __syncthreads();
  const int c = lane < E ? counts[lane] : 0;
  int off = c;  // lane e < NMAX: where expert e's rows end
#pragma unroll
  for (int o = 1; o < NMAX; o <<= 1) {
    const int before = __shfl_up(off, o, 64);
    if (lane >= o) off += before;
  }
  const int rows = __shfl(off, NMAX - 1, 64);
  next += off - c;
  if (t <= E) row_off[t] = t == E ? rows : off - c;
  for (int j = 0; j < k; ++j) {
    const int x = (int)(picks >> (4 * j)) & 15, row = expert_rank(x, t < T, E, next);
    if (t < T) inv[t * k + j] = row;
    if (t < T && row >= 0) src[row] = t, row_expert[row] = x;
  }
  for (int r = rows + t; r < T * k; r += blockDim.x) src[r] = 0, row_expert[r] = 0;  // rows of no expert
}

__global__ void router_offsets_kernel(const int* __restrict__ counts, int E, int* __restrict__ row_off) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int o = 0;
    for (int e = 0; e < E; ++e) {
      row_off[e] = o;
      o += counts[e];
    }
    row_off[E] = o;
  }
}

__global__ void router_scatter_kernel(const int* __restrict__ ids, const int* __restrict__ rank,
                                      const int* __restrict__ row_off, int E, int k, int* __restrict__ src,
                                      int* __restrict__ row_expert, int* __restrict__ inv, int total) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int x = ids[e];
  if (x < E) {
    const int row = row_off[x] + rank[e];
    src[row] = e / k;
    row_expert[row] = x;
    inv[e] = row;
  } else {
    inv[e] = -1;
  }
}

// W_gu [E][2 ff][d]: gate rows then up rows; W_down [E][d][ff]
template <typename AT>
__global__ void __launch_bounds__(256) expert_rows_kernel(const AT* __restrict__ h, int ldh, const int* __restrict__ src,
                                                           const int* __restrict__ row_expert,
                                                           const int* __restrict__ row_off, int E,
                                                           const AT* __restrict__ w_gu, const AT* __restrict__ w_down,
                                                           float* __restrict__ Y, int d, int ff, int clamped, float alpha,
                                                           float limit) {
  extern __shared__ float smem[];  // h [d] | act [ff]
  const int row = blockIdx.x;
  if (row >= row_off[E]) return;
  float* hs = smem;
  float* act = smem + d;
  const int t = src[row], e = row_expert[row];
  for (int i = threadIdx.x; i < d; i += blockDim.x) hs[i] = Elem<AT>::ld(h + (size_t)t * ldh + i);
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const AT* wg = w_gu + (size_t)e * 2 * ff * d;
  for (int f = wv; f < ff; f += nw) {
    const AT* g = wg + (size_t)f * d;
    const AT* u = wg + (size_t)(ff + f) * d;
    float sg = 0.f, su = 0.f;
    for (int i = lane; i < d; i += 64) {
      sg += Elem<AT>::ld(g + i) * hs[i];
      su += Elem<AT>::ld(u + i) * hs[i];
    }
    sg = wave_sum(sg);
    su = wave_sum(su);
    if (lane == 0) {
      if (clamped) {
        const float gc = fminf(sg, limit);
        act[f] = gc * sigmoid_f(alpha * gc) * (fminf(fmaxf(su, -limit), limit) + 1.0f);
      } else {
        act[f] = silu_f(sg) * su;
      }
    }
  }
  __syncthreads();
  const AT* wd = w_down + (size_t)e * d * ff;
  for (int c = wv; c < d; c += nw) {
    const AT* r = wd + (size_t)c * ff;
    float s = 0.f;
    for (int i = lane; i < ff; i += 64) s += Elem<AT>::ld(r + i) * act[i];
    s = wave_sum(s);
    if (lane == 0) Y[(size_t)row * d + c] = s;
  }
}

template <typename AT, typename YT>
__global__ void moe_combine_kernel(const YT* __restrict__ Y, const int* __restrict__ inv, const float* __restrict__ wts,
                                   const AT* __restrict__ h, int ldh, int k, float* __restrict__ out, int d,
                                   const AT* __restrict__ add, int lda, const float* __restrict__ gate, int ldg) {
  const int t = blockIdx.x;
  const float ga = gate ? sigmoid_f(gate[(size_t)t * ldg]) : 1.0f;
  for (int c = threadIdx.x; c < d; c += blockDim.x) {
    float s = add ? Elem<AT>::ld(add + (size_t)t * lda + c) * ga : 0.f;
    for (int j = 0; j < k; ++j) {
      const int r = inv[(size_t)t * k + j];
      const float v = r >= 0 ? Elem<YT>::ld(Y + (size_t)r * d + c) : Elem<AT>::ld(h + (size_t)t * ldh + c);
      s += wts[(size_t)t * k + j] * v;
    }
    out[(size_t)t * d + c] = s;
  }
}

// 4 NCH columns per thread (d a multiple of four, aligned bases), 1024 NCH a workgroup: the loads of a choice's row, and of the
// next choice's, are on their way at once.  64 tokens of 4096, top 2: 6.4 -> 4.8 us (a loop over the columns and the
// choices, a load at a time); 16384 tokens (0.6 GB) 119 -> 109.
template <typename AT, typename YT, int NCH>
__global__ void __launch_bounds__(256) moe_combine_vec_kernel(const YT* __restrict__ Y, const int* __restrict__ inv,
                                                               const float* __restrict__ wts, const AT* __restrict__ h, int ldh,
                                                               int k, float* __restrict__ out, int d, const AT* __restrict__ add,
                                                               int lda, const float* __restrict__ gate, int ldg) {
  const int t = blockIdx.x, c0 = (blockIdx.y * 256 * NCH + threadIdx.x) * 4;
  if (c0 >= d) return;
  const float ga = gate ? sigmoid_f(gate[(size_t)t * ldg]) : 1.0f;
  float4v s[NCH];
#pragma unroll
  for (int u = 0; u < NCH; ++u) {
    const int c = c0 + 1024 * u;
    s[u] = add && c < d ? Vec4<AT>::ld(add + (size_t)t * lda + c) * ga : float4v{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll 2
  for (int j = 0; j < k; ++j) {
    const int r = inv[(size_t)t * k + j];
    const float wt = wts[(size_t)t * k + j];
    float4v v[NCH];
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int c = c0 + 1024 * u, at = c < d ? c : 0;
      v[u] = r >= 0 ? Vec4<YT>::ld(Y + (size_t)r * d + at) : Vec4<AT>::ld(h + (size_t)t * ldh + at);
    }
#pragma unroll
    for (int u = 0; u < NCH; ++u) s[u] += v[u] * wt;
  }
#pragma unroll
  for (int u = 0; u < NCH; ++u) {
    const int c = c0 + 1024 * u;
    if (c < d) Vec4<float>::st(out + (size_t)t * d + c, s[u]);
  }
}

}  // namespace
}  // namespace lwc

using namespace lwc;

extern "C" int r32_router_max_outputs() { return 64 * kMaxPerLane; }

// Whether a router of these sizes runs in one workgroup: counts is not used then, and src and row_expert need no clearing.
extern "C" int r32_router_one_group(int T, int NE) { return T <= kOneGroup && NE <= 16; }

// counts, src and row_expert must be zero on entry (E, T k, T k ints) unless r32_router_one_group(T, NE)
// z rows have leading dimension ldz; corr (added to the scores for the choice only) and bias (added to the logits) may be
// null; sigmoid, renorm, floor, scale, groups, keep: RouterRule
extern "C" int r32_router(const float* z, int ldz, const float* corr, const float* bias, int sigmoid, int renorm, float floor,
                          float scale, int groups, int keep, int T, int NE, int E, int k,
                          int* ids, float* wts, int* counts, int* rank, int* row_off, int* src, int* row_expert, int* inv,
                          hipStream_t s) {
  if (T <= 0) return 0;
  if (NE > 64 * kMaxPerLane || k < 1 || k > NE || E > NE) return -1;
  if (groups > 1 && (NE % groups != 0 || keep < 1 || keep > groups || k > keep * (NE / groups))) return -1;
  const RouterRule rule{sigmoid, renorm, floor, scale, groups, keep};
  if (r32_router_one_group(T, NE)) {
    router_one_group_kernel<16><<<1, (T + 63) / 64 * 64, 0, s>>>(z, corr, bias, ldz, rule, NE, E, k, ids, wts, row_off, src, row_expert,
                                                                inv, T);
    LWC_CHECK_LAUNCH();
    return 0;
  }
  if (NE <= 16) router_topk_thread_kernel<16><<<(T + 63) / 64, 64, 0, s>>>(z, corr, bias, ldz, rule, NE, E, k, ids, wts, counts, rank, T);
  else if (NE <= 64) router_topk_kernel<1><<<(T + 3) / 4, 256, 0, s>>>(z, corr, bias, ldz, rule, NE, E, k, ids, wts, counts, rank, T);
  else router_topk_kernel<kMaxPerLane><<<(T + 3) / 4, 256, 0, s>>>(z, corr, bias, ldz, rule, NE, E, k, ids, wts, counts, rank, T);
  router_offsets_kernel<<<1, 64, 0, s>>>(counts, E, row_off);
  const int total = T * k;
  router_scatter_kernel<<<(total + 255) / 256, 256, 0, s>>>(ids, rank, row_off, E, k, src, row_expert, inv, total);
  LWC_CHECK_LAUNCH();
  return 0;
}

extern "C" int r32_expert_rows(const void* h, int ldh, const int* src, const int* row_expert, const int* row_off, int E,
                               const void* w_gu, const void* w_down, float* Y, int rows, int d, int ff, int clamped, float alpha,
                               float limit, int f32, hipStream_t s) {
  if (rows <= 0) return 0;
  const size_t shm = (size_t)(d + ff) * sizeof(float);
  if (shm > 60000) return -1;
  if (f32)
    expert_rows_kernel<float><<<rows, 256, shm, s>>>((const float*)h, ldh, src, row_expert, row_off, E, (const float*)w_gu,
                                                      (const float*)w_down, Y, d, ff, clamped, alpha, limit);
  else
    expert_rows_kernel<bf16_t><<<rows, 256, shm, s>>>((const bf16_t*)h, ldh, src, row_expert, row_off, E, (const bf16_t*)w_gu,
                                                       (const bf16_t*)w_down, Y, d, ff, clamped, alpha, limit);
  LWC_CHECK_LAUNCH();
  return 0;
}

// add: rows of the activation type added to every token's sum (a shared expert), or null; gate: fp32 logits, one per
// token (stride ldg), whose sigmoid multiplies the added row, or null
extern "C" int r32_moe_combine(const void* Y, int y_f32, const int* inv, const float* wts, const void* h, int ldh, int T,
                               int k, float* out, int d, const void* add, int lda, const float* gate, int ldg, int f32,
                               hipStream_t s) {
  if (T <= 0) return 0;
  if (d > 0 && d % 4 == 0 && ldh % 4 == 0 && lda % 4 == 0 && aligned_to(add, f32 ? 16 : 8) && aligned_to(Y, y_f32 ? 16 : 8) && aligned_to(h, f32 ? 16 : 8) && aligned_to(out, 16)) {
#define LWC_COMBINE(AT, YT, NCH)                                                                                              \
  moe_combine_vec_kernel<AT, YT, NCH><<<dim3(T, (d + 1024 * NCH - 1) / (1024 * NCH)), 256, 0, s>>>(                            \
      (const YT*)Y, inv, wts, (const AT*)h, ldh, k, out, d, (const AT*)add, lda, gate, ldg)
    // as few workgroups a row as hold it in 4096 columns each, of as few columns as that leaves (5120: two of 3072)
    const int groups = (d + 4095) / 4096, nch = (d + 1024 * groups - 1) / (1024 * groups);
#define LWC_COMBINE_N(AT, YT)                  \
  if (nch == 1) LWC_COMBINE(AT, YT, 1);        \
  else if (nch == 2) LWC_COMBINE(AT, YT, 2);   \
  else if (nch == 3) LWC_COMBINE(AT, YT, 3);   \
  else LWC_COMBINE(AT, YT, 4)
    if (f32 && y_f32) {
      LWC_COMBINE_N(float, float);
    } else if (!f32 && y_f32) {
      LWC_COMBINE_N(bf16_t, float);
    } else if (!f32 && !y_f32) {
      LWC_COMBINE_N(bf16_t, bf16_t);
    } else {
      return -1;
    }
#undef LWC_COMBINE_N
#undef LWC_COMBINE
    LWC_CHECK_LAUNCH();
    return 0;
  }
  if (f32 && y_f32)
    moe_combine_kernel<float, float><<<T, 256, 0, s>>>((const float*)Y, inv, wts, (const float*)h, ldh, k, out, d, (const float*)add, lda, gate, ldg);
  else if (!f32 && y_f32)
    moe_combine_kernel<bf16_t, float><<<T, 256, 0, s>>>((const float*)Y, inv, wts, (const bf16_t*)h, ldh, k, out, d, (const bf16_t*)add, lda, gate, ldg);
  else if (!f32 && !y_f32)
    moe_combine_kernel<bf16_t, bf16_t><<<T, 256, 0, s>>>((const bf16_t*)Y, inv, wts, (const bf16_t*)h, ldh, k, out, d, (const bf16_t*)add, lda, gate, ldg);
  else
    return -1;
  LWC_CHECK_LAUNCH();
  return 0;
}
