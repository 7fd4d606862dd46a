// Retention: linear attention with a fixed decay per head and no softmax (gfx950, wave64).
//
//   S_t = a_h S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t          S fp32 [D, Dv] per head and sequence
// q and k are rotated by position on their first `rd` entries ("rotate half": entry i pairs with i + rd / 2, angle
// p * f_i as an fp32 product), k is then multiplied by D^-1/2.  Everything that enters the recurrence is fp32.
// Lightning form: q, k and v go through silu first, no rotation (rd = 0), no scale.
//
//   retention_prep   q, k of a step's rows (activation type) -> activated, rotated, scaled fp32 rows [T, 2, H, D]
//   retention        the recurrence over a step's items (rows of one sequence at consecutive positions + the
//                    sequence's state slot; a decode row is an item of one row).  One workgroup of NW waves per (item,
//                    head, 16 NW value columns): a lane keeps a quarter of one state column in registers (lane =
//                    quarter * 16 + column), the q / k / v of TT tokens are staged through LDS at once (one barrier
//                    pair per TT tokens), the four partial dots of a column meet by two half-wave swaps.  The state is
//                    read from the slot unless the item starts at position 0, and written back at the end.
#include <type_traits>
#include "elem.h"

namespace lwc {
namespace {

template <typename AT, bool ACT>
__global__ void __launch_bounds__(256)
retention_prep_kernel(const AT* __restrict__ proj, int ldp, int k_off, const float* __restrict__ freq, float mult,
                      const int* __restrict__ positions, float* __restrict__ qk, int H, int D, int rd, float k_scale) {
  const int t = blockIdx.x;
  auto ld = [](const AT* p) {
    const float z = Elem<AT>::ld(p);
    return ACT ? silu_f(z) : z;
  };
  const float p = (float)positions[t];
  const AT* pr = proj + (size_t)t * ldp;
  float* o = qk + (size_t)t * 2 * H * D;
  const int half = rd / 2;
  for (int i = threadIdx.x; i < half; i += blockDim.x) {  // one angle serves every head, q and k
    float sn, cs;
    sincosf(p * freq[i], &sn, &cs);
    sn *= mult, cs *= mult;
    for (int h = 0; h < H; ++h) {
      const int c = h * D + i;
      const float qu = ld(pr + c), qv = ld(pr + c + half);
      const float ku = ld(pr + k_off + c), kv = ld(pr + k_off + c + half);
      o[c] = qu * cs - qv * sn;
      o[c + half] = qv * cs + qu * sn;
      o[H * D + c] = (ku * cs - kv * sn) * k_scale;
      o[H * D + c + half] = (kv * cs + ku * sn) * k_scale;
    }
  }
  const int rest = D - rd;
  for (int e = threadIdx.x; e < H * rest; e += blockDim.x) {
    const int h = e / rest, c = h * D + rd + (e - h * rest);
    o[c] = ld(pr + c);
    o[H * D + c] = ld(pr + k_off + c) * k_scale;
  }
}

// Activated rows without a rotation (k_scale on the second half), four entries per thread: n = H D a multiple of four
template <typename AT>
__global__ void __launch_bounds__(256)
lightning_prep_vec_kernel(const AT* __restrict__ proj, int ldp, int k_off, float* __restrict__ qk, int n, float k_scale) {
  const int t = blockIdx.x;
  const AT* pr = proj + (size_t)t * ldp;
  float* o = qk + (size_t)t * 2 * n;
#pragma unroll 4
  for (int e = threadIdx.x * 4; e < 2 * n; e += 1024) {
    const bool isk = e >= n;
    const float4v z = Vec4<AT>::ld(pr + (isk ? k_off + e - n : e));
    const float4v a = float4v{silu_f(z[0]), silu_f(z[1]), silu_f(z[2]), silu_f(z[3])};
    Vec4<float>::st(o + e, isk ? a * k_scale : a);
  }
}

constexpr int kTT = 16;  // tokens staged at once

template <typename AT, int DPL, int NW>
__global__ void __launch_bounds__(64 * NW)
retention_kernel(const float* __restrict__ qk, const AT* __restrict__ v, int ldv, const float* __restrict__ decay,
                 float* __restrict__ state, long long slot_stride, const int* __restrict__ cu,
                 const int* __restrict__ item_slot, const int* __restrict__ positions, float* __restrict__ out, int ldo,
                 int H, int D, int Dv, int col_tiles, int act) {
  constexpr int QLD = DPL + 4;   // a quarter's stride in LDS: the four quarters start in different banks
  constexpr int VT = 16 * NW;    // value columns of a workgroup
  __shared__ __attribute__((aligned(16))) float q_s[kTT][4 * QLD];
  __shared__ __attribute__((aligned(16))) float k_s[kTT][4 * QLD];
  __shared__ float v_s[kTT][VT];
  const int item = blockIdx.y;
  const int h = blockIdx.x / col_tiles, col0 = (blockIdx.x % col_tiles) * VT;
  const int r0 = cu[item], r1 = cu[item + 1];
  if (r0 >= r1) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int r = lane >> 4, cl = wv * 16 + (lane & 15), col = col0 + cl;
  const bool live = col < Dv;
  const int i0 = r * DPL;
  const float a = decay[h];
  float* Sg = state + (long long)item_slot[item] * slot_stride + ((size_t)h * D + i0) * Dv + (live ? col : 0);
  float S[DPL];
  const bool fresh = positions[r0] == 0;
#pragma unroll
  for (int j = 0; j < DPL; ++j) S[j] = (!fresh && live && i0 + j < D) ? Sg[(size_t)j * Dv] : 0.f;
  for (int t0 = r0; t0 < r1; t0 += kTT) {
    const int nt = min(kTT, r1 - t0);
    __syncthreads();  // the previous tile has been read
    for (int e = tid; e < nt * 4 * DPL; e += 64 * NW) {
      const int tt = e / (4 * DPL), i = e - tt * (4 * DPL);
      const float* row = qk + (size_t)(t0 + tt) * 2 * H * D + (size_t)h * D;
      const int at = (i / DPL) * QLD + (i % DPL);
      q_s[tt][at] = i < D ? row[i] : 0.f;
      k_s[tt][at] = i < D ? row[H * D + i] : 0.f;
    }
    for (int e = tid; e < nt * VT; e += 64 * NW) {
      const int tt = e / VT, c = e - tt * VT;
      const float z = col0 + c < Dv ? Elem<AT>::ld(v + (size_t)(t0 + tt) * ldv + (size_t)h * Dv + col0 + c) : 0.f;
      v_s[tt][c] = act ? silu_f(z) : z;
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float4v* ks = reinterpret_cast<const float4v*>(&k_s[tt][r * QLD]);
      const float4v* qs = reinterpret_cast<const float4v*>(&q_s[tt][r * QLD]);
      const float vv = v_s[tt][cl];
      float4v acc = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < DPL / 4; ++j) {
        const float4v k4 = ks[j], q4 = qs[j];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[4 * j + e] = a * S[4 * j + e] + k4[e] * vv;
          acc[e] += S[4 * j + e] * q4[e];
        }
      }
      const float o = row_sum4((acc[0] + acc[1]) + (acc[2] + acc[3]));
      if (live && r == 0) out[(size_t)(t0 + tt) * ldo + (size_t)h * Dv + col] = o;
    }
  }
  if (live) {
#pragma unroll
    for (int j = 0; j < DPL; ++j)
      if (i0 + j < D) Sg[(size_t)j * Dv] = S[j];
  }
}

// The same recurrence over whole portions, a chunk of kC = 32 tokens at a time on the fp32 matrix cores.  With S the state
// before the chunk and i, j its tokens:
//   o_i = a^(i+1) S^T q_i + sum_(j <= i) a^(i-j) (q_i . k_j) v_j,     S <- a^n S + sum_j a^(n-1-j) k_j v_j^T
// One workgroup of four waves per (item, head, 64 value columns), a wave owns 16 columns and all D rows of the state: the
// accumulators of v_mfma_f32_16x16x4, whose layout (row 4 g + r, column c) is the B operand's as well when the contraction
// runs over d = 16 n + 4 g + r, so the state never leaves its registers; A is then four consecutive floats of a q row.  The
// 32 x 32 products q_i . k_j are formed once per workgroup (k on the row side, so that a lane holds four consecutive j of
// one i: the A operand of their product with v), the next chunk's rows are in flight meanwhile.
typedef float float4a __attribute__((ext_vector_type(4)));
LWC_DEVICE float4a mfma4(float a, float b, const float4a& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int kC = 32;

template <typename AT, int ND>  // D <= 16 ND
__global__ void __launch_bounds__(256, ND <= 8 ? 2 : 1)
retention_chunk_kernel(const float* __restrict__ qk, const AT* __restrict__ v, int ldv, const float* __restrict__ decay,
                       float* __restrict__ state, long long slot_stride, const int* __restrict__ cu,
                       const int* __restrict__ item_slot, const int* __restrict__ positions, float* __restrict__ out, int ldo,
                       int H, int D, int Dv, int col_tiles, int act) {
  constexpr int DP = 16 * ND, LD = DP + 4;     // LD: a row's and the next row's entries start four banks apart
  __shared__ __attribute__((aligned(16))) float qk_s[2][kC * LD];  // q | k rows
  __shared__ __attribute__((aligned(16))) float p_s[kC * (kC + 4)];
  __shared__ float pw[kC + 1], pw_lo[kC + 1];  // a^n, and what its rounding left out
  const int item = blockIdx.y, h = blockIdx.x / col_tiles;
  const int r0 = cu[item], r1 = cu[item + 1];
  if (r0 >= r1) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, g = lane >> 4;
  const int col0 = (blockIdx.x % col_tiles) * 64 + wv * 16, col = col0 + c16;
  const bool wlive = col0 < Dv, live = col < Dv;  // (a wave without columns still stages and multiplies q by k)
  if (tid <= kC) {
    double x = 1.0, b = (double)decay[h];
    for (int n = tid; n; n >>= 1, b *= b)
      if (n & 1) x *= b;
    pw[tid] = (float)x;
    pw_lo[tid] = (float)(x - (double)(float)x);
  }
  float* Sg = state + (long long)item_slot[item] * slot_stride + (size_t)h * D * Dv + (live ? col : 0);
  const bool fresh = positions[r0] == 0;
  float4a S[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * n + 4 * g + r;
      S[n][r] = (!fresh && live && d < D) ? Sg[(size_t)d * Dv] : 0.f;
    }
  if (D < DP)  // entries past D stay zero
    for (int e = tid; e < 2 * kC * LD; e += 256) qk_s[0][e] = 0.f;
  // A chunk's rows on their way to LDS, and the wave's values: loaded a chunk ahead, as they lie.  A thread's groups of four
  // floats lie TPU tokens apart: a uniform base per load and one lane offset for all of them (the address arithmetic of 24
  // loads and stores per chunk would otherwise be as long as a third of its MFMAs).
  constexpr int PER = kC * DP / 512, TPU = 1024 / DP;  // groups per thread: the first half of q, the second of k
  float4a st[PER];
  AT vr[8];
  const int i4 = tid % (DP / 4) * 4, tt0 = tid / (DP / 4);
  const unsigned row = 2u * H * D, qk_off = tt0 * row + min(i4, D - 4);
  const unsigned v_off = 4u * g * ldv + min(col, Dv - 1), o_off = 4u * g * ldo + col;
  auto fetch_qk = [&](int t0, int u) {  // group u of the chunk at t0, all of whose rows are there
    st[u] = *reinterpret_cast<const float4a*>(qk + (size_t)(t0 + u % (PER / 2) * TPU) * row + (size_t)(u / (PER / 2)) * H * D + (size_t)h * D + qk_off);
  };
  auto fetch_v = [&](int t0, int u) { vr[u] = (v + (size_t)(t0 + 16 * (u >> 2) + (u & 3)) * ldv + (size_t)h * Dv)[v_off]; };
  auto fetch_tail = [&](int t0) {  // fewer rows: the last one stands in for those past the end
#pragma unroll
    for (int u = 0; u < PER; ++u)
      st[u] = *reinterpret_cast<const float4a*>(qk + (size_t)min(t0 + u % (PER / 2) * TPU + tt0, r1 - 1) * row + (size_t)(u / (PER / 2)) * H * D + (size_t)h * D + min(i4, D - 4));
#pragma unroll
    for (int u = 0; u < 8; ++u)
      vr[u] = v[(size_t)min(t0 + 16 * (u >> 2) + 4 * g + (u & 3), r1 - 1) * ldv + (size_t)h * Dv + min(col, Dv - 1)];
  };
  __syncthreads();  // the powers are in LDS
  const int ib = wv > 0, jb = wv > 1;  // the first three waves form the blocks (i, j) = (0, 0), (1, 0), (1, 1) of the products
  float pij[4];                        // a^(i-j) of the lane's products
#pragma unroll
  for (int r = 0; r < 4; ++r) pij[r] = pw[max(16 * (ib - jb) + c16 - 4 * g - r, 0)];
  auto chunk = [&](int t0, auto whole) {
    constexpr bool W = decltype(whole)::value;
    const int nt = W ? kC : r1 - t0;
    // the rows that the loads inside the loop below fetch: the next whole chunk's (there is none: this one's again, unused)
    const int tn = t0 + 2 * kC <= r1 ? t0 + kC : t0;
    __syncthreads();  // the previous chunk has been read
    if (i4 < D) {
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int tt = tt0 + u % (PER / 2) * TPU;
        const float4a zero = {0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<float4a*>(&qk_s[u / (PER / 2)][tt * LD + i4]) = W || tt < nt ? st[u] : zero;
      }
    }
    float vc[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float z = Elem<AT>::ld(&vr[u]);
      vc[u] = W || 16 * (u >> 2) + 4 * g + (u & 3) < nt ? z : 0.f;
    }
    if (act) {
#pragma unroll
      for (int u = 0; u < 8; ++u) vc[u] = silu_f(vc[u]);
    }
    __syncthreads();
    if (wv < 3) {
      const float4a* kr = reinterpret_cast<const float4a*>(&qk_s[1][(16 * jb + c16) * LD + 4 * g]);
      const float4a* qr = reinterpret_cast<const float4a*>(&qk_s[0][(16 * ib + c16) * LD + 4 * g]);
      float4a x[4] = {};
      float4a k4 = kr[0], q4 = qr[0];
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const int nn = n + 1 < ND ? n + 1 : n;
        const float4a kn = kr[4 * nn], qn = qr[4 * nn];  // (LDS reads one step ahead)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = mfma4(k4[r], q4[r], x[r]);
        __builtin_amdgcn_sched_barrier(0);
        k4 = kn, q4 = qn;
      }
      float4a y = (x[0] + x[1]) + (x[2] + x[3]);
      const int i = 16 * ib + c16, j = 16 * jb + 4 * g;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = j + r <= i ? y[r] * pij[r] : 0.f;
      *reinterpret_cast<float4a*>(&p_s[i * (kC + 4) + j]) = y;
    }
    float4a O[2];
    {
      const float4a* qr = reinterpret_cast<const float4a*>(&qk_s[0][c16 * LD + 4 * g]);
      float4a x[4] = {}, y[4] = {};
      float4a q0 = qr[0], q1 = qr[4 * LD];
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const int nn = n + 1 < ND ? n + 1 : n;
        const float4a n0 = qr[4 * nn], n1 = qr[4 * LD + 4 * nn];
        if (W) {  // the next chunk's loads, spread over the MFMAs
#pragma unroll
          for (int u = n * PER / ND; u < (n + 1) * PER / ND; ++u) fetch_qk(tn, u);
#pragma unroll
          for (int u = n * 8 / ND; u < (n + 1) * 8 / ND; ++u) fetch_v(tn, u);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (wlive) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            x[r] = mfma4(q0[r], S[n][r], x[r]);
            y[r] = mfma4(q1[r], S[n][r], y[r]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        q0 = n0, q1 = n1;
      }
      O[0] = (x[0] + x[1]) + (x[2] + x[3]);
      O[1] = (y[0] + y[1]) + (y[2] + y[3]);
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) O[b][r] *= pw[16 * b + 4 * g + r + 1];
    }
    if (W && t0 + 2 * kC > r1) fetch_tail(t0 + kC);
    __syncthreads();  // the products are in LDS
    if (!wlive) return;
    const float4a* pr = reinterpret_cast<const float4a*>(&p_s[c16 * (kC + 4) + 4 * g]);
    const float4a p00 = pr[0], p10 = pr[4 * (kC + 4)], p11 = pr[4 * (kC + 4) + 4];
    float finite = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) finite = fmaf(vc[u], 0.f, finite);
    if (__all(finite == 0.f)) {
      float4a x = {0.f, 0.f, 0.f, 0.f}, y = x, z = x;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x = mfma4(p00[r], vc[r], x);
        y = mfma4(p10[r], vc[r], y);
        z = mfma4(p11[r], vc[4 + r], z);
      }
      O[0] += x;
      O[1] += y + z;
    } else {  // an infinity or NaN must not reach the tokens before it (as 0 x it): row by row over its own tokens
      for (int i = 0; i < nt; ++i) {
        float4a x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 4 * g + r;
          x = mfma4(i < 16 ? p00[r] : p10[r], j <= i ? vc[r] : 0.f, x);
          if (i >= 16) x = mfma4(p11[r], 16 + j <= i ? vc[4 + r] : 0.f, x);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (i == 4 * g + r) O[0][r] += x[r];
          if (i == 16 + 4 * g + r) O[1][r] += x[r];
        }
      }
    }
    if (live) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int t = 16 * (u >> 2) + (u & 3);
        if (W || t + 4 * g < nt) (out + (size_t)(t0 + t) * ldo + (size_t)h * Dv)[o_off] = O[u >> 2][u & 3];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int t = 16 * (u >> 2) + 4 * g + (u & 3);
      if (W) vc[u] *= pw[kC - 1 - t];
      else vc[u] = t < nt ? vc[u] * pw[max(nt - 1 - t, 0)] : 0.f;
    }
    const float an = pw[nt], an_lo = pw_lo[nt];  // (the same factor chunk after chunk: its rounding would add up)
    const float* kc = &qk_s[1][4 * g * LD + c16];
    float ka[8], kb[8];
    auto load = [&](float (&d)[8], int n) {
#pragma unroll
      for (int u = 0; u < 8; ++u) d[u] = kc[(16 * (u >> 2) + (u & 3)) * LD + 16 * n];
    };
    load(ka, 0);
    load(kb, 1);
#pragma unroll
    for (int n = 0; n < ND; n += 2) {
      float na[8], nb[8];
      if (n + 2 < ND) {
        load(na, n + 2);
        load(nb, n + 3);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        S[n][r] = fmaf(S[n][r], an, S[n][r] * an_lo);
        S[n + 1][r] = fmaf(S[n + 1][r], an, S[n + 1][r] * an_lo);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        S[n] = mfma4(ka[u], vc[u], S[n]);
        S[n + 1] = mfma4(kb[u], vc[u], S[n + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (n + 2 < ND) {
#pragma unroll
        for (int u = 0; u < 8; ++u) ka[u] = na[u], kb[u] = nb[u];
      }
    }
  };
  int t0 = r0;
  if (t0 + kC <= r1) {
#pragma unroll
    for (int u = 0; u < PER; ++u) fetch_qk(t0, u);
#pragma unroll
    for (int u = 0; u < 8; ++u) fetch_v(t0, u);
  } else {
    fetch_tail(t0);
  }
  for (; t0 + kC <= r1; t0 += kC) chunk(t0, std::true_type{});
  if (t0 < r1) chunk(t0, std::false_type{});
  if (live) {
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * n + 4 * g + r;
        if (d < D) Sg[(size_t)d * Dv] = S[n][r];
      }
  }
}

}  // namespace
}  // namespace lwc

using namespace lwc;

// Rows per item from which the chunk kernel takes a step.  Measured with 32 items (32 heads of 128 x 128, prep included): 16
// rows each 62 us token by token and 67 in chunks, 32 rows 86 and 73.
constexpr int kChunkFrom = 32;

extern "C" int r32_retention_max_dim() { return 256; }

extern "C" int r32_retention_prep(const void* proj, int ldp, int k_off, const float* freq, float mult, const int* positions,
                                  float* qk, int T, int H, int D, int rd, float k_scale, int act, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (rd % 2 != 0 || rd > D || rd < 0) return -1;
  const int ab = f32 ? 16 : 8;
  if (act && rd == 0 && H * D % 4 == 0 && ldp % 4 == 0 && k_off % 4 == 0 && aligned_to(proj, ab) && aligned_to(qk, 16)) {
    if (f32) lightning_prep_vec_kernel<float><<<T, 256, 0, s>>>((const float*)proj, ldp, k_off, qk, H * D, k_scale);
    else lightning_prep_vec_kernel<bf16_t><<<T, 256, 0, s>>>((const bf16_t*)proj, ldp, k_off, qk, H * D, k_scale);
    LWC_CHECK_LAUNCH();
    return 0;
  }
#define LWC_PREP(AT, ACT) \
  retention_prep_kernel<AT, ACT><<<T, 256, 0, s>>>((const AT*)proj, ldp, k_off, freq, mult, positions, qk, H, D, rd, k_scale)
  if (f32 && act) LWC_PREP(float, true);
  else if (f32) LWC_PREP(float, false);
  else if (act) LWC_PREP(bf16_t, true);
  else LWC_PREP(bf16_t, false);
#undef LWC_PREP
  LWC_CHECK_LAUNCH();
  return 0;
}

// qk fp32 [T, 2, H, D] from retention_prep; v rows of the activation type (leading dimension ldv), head h at columns
// h Dv ..; state fp32 [slots, H, D, Dv]; out fp32 rows (leading dimension ldo); act != 0: v goes through silu
extern "C" int r32_retention(const float* qk, const void* v, int ldv, const float* decay, float* state, long long slot_stride,
                             const int* cu, const int* item_slot, const int* positions, float* out, int ldo, int items,
                             int T, int H, int D, int Dv, int act, int f32, hipStream_t s) {
  if (items <= 0) return 0;
  if (D < 1 || D > 256 || Dv < 1) return -1;
  if (T >= kChunkFrom * items && D % 4 == 0 && D >= 4) {
    const int tiles = (Dv + 63) / 64;
#define LWC_RETC2(AT, ND)                                                                                       \
  retention_chunk_kernel<AT, ND><<<dim3(H * tiles, items), 256, 0, s>>>(qk, (const AT*)v, ldv, decay, state, slot_stride, cu, \
                                                                        item_slot, positions, out, ldo, H, D, Dv, tiles, act)
#define LWC_RETC(ND)       \
  if (f32) {               \
    LWC_RETC2(float, ND);  \
  } else {                 \
    LWC_RETC2(bf16_t, ND); \
  }
    if (D <= 32) {
      LWC_RETC(2)
    } else if (D <= 64) {
      LWC_RETC(4)
    } else if (D <= 128) {
      LWC_RETC(8)
    } else {
      LWC_RETC(16)
    }
#undef LWC_RETC
#undef LWC_RETC2
    LWC_CHECK_LAUNCH();
    return 0;
  }
  const int tiles = (Dv + 15) / 16;
#define LWC_RET2(AT, DPL, NW)                                                                                             \
  retention_kernel<AT, DPL, NW><<<dim3(H * ((tiles + NW - 1) / NW), items), 64 * NW, 0, s>>>(                            \
      qk, (const AT*)v, ldv, decay, state, slot_stride, cu, item_slot, positions, out, ldo, H, D, Dv, (tiles + NW - 1) / NW, act)
#define LWC_RET(DPL, NW)       \
  if (f32) {                   \
    LWC_RET2(float, DPL, NW);  \
  } else {                     \
    LWC_RET2(bf16_t, DPL, NW); \
  }
#define LWC_RET_NW(DPL)    \
  if (tiles >= 4) {        \
    LWC_RET(DPL, 4)        \
  } else if (tiles >= 2) { \
    LWC_RET(DPL, 2)        \
  } else {                 \
    LWC_RET(DPL, 1)        \
  }
  if (D <= 32) {
    LWC_RET_NW(8)
  } else if (D <= 64) {
    LWC_RET_NW(16)
  } else if (D <= 128) {
    LWC_RET_NW(32)
  } else {
    LWC_RET_NW(64)
  }
#undef LWC_RET_NW
#undef LWC_RET
#undef LWC_RET2
  LWC_CHECK_LAUNCH();
  return 0;
}
