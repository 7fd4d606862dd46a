// Sliding-window attention with a logarithmic distance bias over a paged K/V cache (gfx950, wave64).
//
//   score(i, j) = q_i . k_j - r1_h * ln(1 + r2_h * (i - j))        for 0 <= i - j < window
//   out_i       = softmax_j(score) . v_j
// With a sink (fp32 per head) the softmax's denominator also holds exp(sink_h): a share of the weight that belongs
// to no key and adds no value.  With a cap c > 0 a score q . k becomes c tanh(q . k / c) (before the distance bias).
// q arrives in fp32 already multiplied by the head's softmax scale; K rows have D elements, V rows Dv (any sizes,
// D != Dv allowed), G key/value heads serve H query heads (head h reads group h / (H / G)).  Scores, the softmax
// and the weighted sum are fp32 whatever the cache's element type (bf16 or fp32).
//
// Cache layout (one layer): K [num_blocks, block_size, G * D] token rows; V [num_blocks, block_size / 4, G * Dv, 4],
// 4-token interleaved: the four tokens 4t .. 4t+3 of one value column are one 8-byte word (bf16), which is the
// matrix cores' B operand for P V as it lies in memory.  Block strides are given separately (the layers of a model
// share one pool).
//
// Rows are query tokens.  Row t belongs to table row `item`: t itself when cu_q is null (decode: one token
// per sequence), else the item with cu_q[item] <= t < cu_q[item + 1] (a portion of a prompt); its position in
// the sequence is positions[t], and every key it may see is already in the cache.
//
// window_attn_kernel: one wave per (row, head); lanes over 64 keys for the scores, an online softmax per
// 64-key step, then lanes over the value dimension (several keys side by side when Dv < 64).
#include <algorithm>

#include "elem.h"

namespace lwc {
namespace {

template <typename CT> struct KLoad;
template <> struct KLoad<bf16_t> {
  static constexpr int kVec = 8;
  static LWC_DEVICE float dot(const bf16_t* k, const float* q, int D) {
    float acc = 0.f;
    if ((D & 7) == 0 && ((uintptr_t)k & 15) == 0) {
      for (int d = 0; d < D; d += 8) {
        const uint4v kv = *reinterpret_cast<const uint4v*>(k + d);
        float f[8];
        unpack8(kv, f);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += q[d + e] * f[e];
      }
    } else {
      for (int d = 0; d < D; ++d) acc += q[d] * bf2f(k[d]);
    }
    return acc;
  }
  static LWC_DEVICE float ld(const bf16_t* p) { return bf2f(*p); }
  static LWC_DEVICE void st(bf16_t* p, float v) { *p = f2bf(v); }
};
template <> struct KLoad<float> {
  static LWC_DEVICE float dot(const float* k, const float* q, int D) {
    float acc = 0.f;
    if ((D & 3) == 0 && ((uintptr_t)k & 15) == 0) {
      for (int d = 0; d < D; d += 4) {
        const float4v kv = *reinterpret_cast<const float4v*>(k + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc += q[d + e] * kv[e];
      }
    } else {
      for (int d = 0; d < D; ++d) acc += q[d] * k[d];
    }
    return acc;
  }
  static LWC_DEVICE float ld(const float* p) { return *p; }
  static LWC_DEVICE void st(float* p, float v) { *p = v; }
};

constexpr int kMaxSlots = 8;  // value dimension <= 512

template <typename CT>
__global__ void __launch_bounds__(64)
window_attn_kernel(const float* __restrict__ q, const CT* __restrict__ k_cache, const CT* __restrict__ v_cache,
                   long long kb_stride, long long vb_stride, int block_size, const int* __restrict__ positions,
                   const int* __restrict__ cu_q, int n_items, const int* __restrict__ block_tables, int bt_width,
                   const float* __restrict__ r1, const float* __restrict__ r2, const float* __restrict__ sink, int window,
                   int chunk, float cap, CT* __restrict__ out, int ldo, int H, int G, int D, int Dv) {
  extern __shared__ float q_s[];  // [D]
  __shared__ float p_s[64];
  __shared__ long long vo_s[64];
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  int item = t;
  if (cu_q) {
    int lo = 0, hi = n_items - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (cu_q[mid] <= t) lo = mid; else hi = mid - 1;
    }
    item = lo;
  }
  const int* table = block_tables + (size_t)item * bt_width;
  const int i = positions[t];
  const int g = h / (H / G);
  for (int d = lane; d < D; d += 64) q_s[d] = q[((size_t)t * H + h) * D + d];
  __syncthreads();
  const float r1h = r1[h], r2h = r2[h];
  int DvP = 64;
  if (Dv < 64) {
    DvP = 1;
    while (DvP < Dv) DvP <<= 1;
  }
  const int kpar = 64 / DvP, dvl = lane % DvP, kp = lane / DvP;
  float o[kMaxSlots];
#pragma unroll
  for (int ns = 0; ns < kMaxSlots; ++ns) o[ns] = 0.f;
  float m = -INFINITY, l = 0.f;
  const int j_lo = max(max(0, i - window + 1), chunk > 0 ? i - i % chunk : 0);  // the window's and the chunk's first key
  for (int j0 = j_lo; j0 <= i; j0 += 64) {
    const int j = j0 + lane;
    const bool valid = j <= i;
    float s = -INFINITY;
    long long vo = 0;
    if (valid) {
      const long long blk = table[j / block_size];
      const long long off = j % block_size;
      const CT* kr = k_cache + blk * kb_stride + (off * G + g) * D;
      s = KLoad<CT>::dot(kr, q_s, D);
      if (cap > 0.f) s = cap * tanhf(s / cap);
      s -= r1h * log1pf(r2h * (float)(i - j));
      vo = blk * vb_stride + (off >> 2) * (4LL * G * Dv) + 4LL * g * Dv + (off & 3);
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);
    l = l * alpha + wave_sum(p);
    m = m_new;
    __syncthreads();
    p_s[lane] = p;
    vo_s[lane] = vo;
    __syncthreads();
    const int nkeys = min(64, i - j0 + 1);
#pragma unroll
    for (int ns = 0; ns < kMaxSlots; ++ns) o[ns] *= alpha;
    for (int jj = kp; jj < nkeys; jj += kpar) {
      const float pj = p_s[jj];
      const CT* vr = v_cache + vo_s[jj];
#pragma unroll
      for (int ns = 0; ns < kMaxSlots; ++ns) {
        const int dv = ns * 64 + dvl;
        if (dv < Dv) o[ns] += pj * KLoad<CT>::ld(vr + 4 * dv);
      }
    }
  }
  for (int off = DvP; off < 64; off <<= 1) o[0] += __shfl_xor(o[0], off, 64);
  if (sink) {  // a sink: exp(sink_h) joins the denominator; it has no key and no value
    const float sk = sink[h], mf = fmaxf(m, sk), a = expf(m - mf);
    l = l * a + expf(sk - mf);
#pragma unroll
    for (int ns = 0; ns < kMaxSlots; ++ns) o[ns] *= a;
  }
  if (kp == 0) {
    const float inv = 1.0f / l;
    CT* orow = out + (size_t)t * ldo + (size_t)h * Dv;
#pragma unroll
    for (int ns = 0; ns < kMaxSlots; ++ns) {
      const int dv = ns * 64 + dvl;
      if (dv < Dv) KLoad<CT>::st(orow + dv, o[ns] * inv);
    }
  }
}

}  // namespace
}  // namespace lwc

using namespace lwc;

extern "C" int r32_window_attn(const float* q, const void* k_cache, const void* v_cache, long long kb_stride,
                               long long vb_stride, int block_size, const int* positions, const int* cu_q, int n_items,
                               const int* block_tables, int bt_width, const float* r1, const float* r2, const float* sink,
                               int window, int chunk, float cap, void* out, int ldo, int T, int H, int G, int D, int Dv, int f32,
                               hipStream_t s) {
  if (T <= 0) return 0;
  if (Dv > 64 * kMaxSlots || D > 8192 || H % G != 0) return -1;
  const dim3 grid(T, H);
  const size_t shm = (size_t)D * sizeof(float);
  if (f32)
    window_attn_kernel<float><<<grid, 64, shm, s>>>(q, (const float*)k_cache, (const float*)v_cache, kb_stride, vb_stride,
                                                    block_size, positions, cu_q, n_items, block_tables, bt_width, r1, r2,
                                                    sink, window, chunk, cap, (float*)out, ldo, H, G, D, Dv);
  else
    window_attn_kernel<bf16_t><<<grid, 64, shm, s>>>(q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, kb_stride,
                                                     vb_stride, block_size, positions, cu_q, n_items, block_tables,
                                                     bt_width, r1, r2, sink, window, chunk, cap, (bf16_t*)out, ldo, H, G, D, Dv);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------
// window_attn_mfma_kernel: prompt portions on the matrix cores (bf16 cache, D = 32 ND, Dv = 16 NV).
//
// Workgroup = 4 waves = 64 QS consecutive query rows of one (item, head); wave w owns rows 16 QS w .. in QS blocks of 16
// and all four walk the 32-key tiles of the rows' windows, staged through LDS (K row-major; V transposed with the keys
// permuted so that a lane's eight k-slots of one value column are one 16-byte read).  mfma_f32_16x16x32_bf16, lane l:
// r16 = l & 15, g = l >> 4:
//   S^T = K Q^T : A = K rows from LDS, B = Q^T in registers; C reg r = S^T[key 4g + r][query r16], two 16-key
//                 subtiles.  q is fp32: it enters as hi + lo bf16 halves (two MFMAs), so the scores keep fp32's
//                 precision against the cache's bf16 keys.
//   O  += P V   : A = the lane's own softmax weights (k slots 8g+e <-> keys {4g+e, 16+4g+e-4}), again as hi + lo
//                 halves; B = V^T from LDS with the same key permutation; C reg r = O[query 4g + r][dv 16n + r16].
// The distance bias comes from a table bias[h][i - j] (fp32, built once from r1, r2).  Online softmax in fp32;
// masked scores never enter it (weights forced to 0), rows are finite-initialised.
// Positions ascend by one along an item's rows (a portion of a prompt).
//
// Bound by the matrix cores and the LDS reads that feed them: the two halves of q and of the weights double the products,
// and with one 16-row block per wave every product reads its own 1 KiB fragment, which two blocks (QS 2, kWideFrom) share.  The
// row sums stay in their lanes until the end, the reference maximum moves only past 2^8, the four lanes of a row meet by lane
// swaps, and without a distance bias none is read.  8 x 2048 tokens, 32 heads, one MI355X: 192 / 128 entries, 32 key heads 2270
// -> 890 us; 128 / 128, 8 key heads 1462 -> 750 us; 2 x 512 tokens 52 -> 38 us and 44 -> 35 us.

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

LWC_DEVICE float4v mfma16(const short8& a, const short8& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

struct WAttnMfmaParams {
  const float* q;
  const bf16_t* k_cache;
  const bf16_t* v_cache;
  long long kb_stride, vb_stride;
  int block_size, bs_shift;  // block_size = 1 << bs_shift (the matrix-core kernels take power-of-two pages)
  const int* positions;
  const int* cu_q;
  const int* k_lens;
  int tiles_per_item;
  int unit;           // neighbouring heads that run on one XCD (H / G or 1), 0: workgroups in plain order
  const int* block_tables;
  int bt_width;
  const float* bias;  // [H, window], or null: no distance bias
  const float* sink;  // [H], or null: exp(sink_h) joins the softmax denominator of head h (no key, no value)
  int window;
  int chunk;          // > 0: row i sees only keys of its own chunk, j >= i - i % chunk (besides the window)
  float cap;          // > 0: scores become cap tanh(score / cap)
  bf16_t* out;
  int ldo, H, G;
};

constexpr float kLog2e = 1.4426950408889634f;
// Two row blocks per wave from as many rows times heads as make this many workgroups of 128 rows, with 192 key entries (whose
// score products read the most LDS), and portions of more than 64 rows on average (shorter ones leave waves without rows).  us,
// one / two blocks, 32 heads of 192 / 128: 8 x 2048 tokens 1072 / 890, 8 x 512 (1024) 116 / 105, 64 x 200 259 / 222, 64 x 65 68 / 65,
// 24 x 130 (780) 56 / 64, 16 x (300 and 30) 105 / 114.  128 / 128: 8 x 2048 750 / 750, 8 x 512 89 / 90, 64 x 100 63 / 67, 24 x 20 8.2 /
// 13.8; 64 / 64, 16 heads: 8 x 2048 230 / 242, 64 x 100 22 / 27.
constexpr long long kWideFrom = 1024;
constexpr int kVPad = 40;  // keys per V^T row in LDS (32 + 8: rows stay 16-byte aligned, banks spread)

template <int ND, int NV, int QS, bool BIAS>
__global__ void __launch_bounds__(256, 2) window_attn_mfma_kernel(const WAttnMfmaParams p) {
  constexpr int D = 32 * ND, DV = 16 * NV, KLD = D + 8, ROWS = 64 * QS, NB = ROWS + 32;
  constexpr int KCH = (32 * (D / 8) + 255) / 256, VCH = (8 * (DV / 2) + 255) / 256;  // 16-byte words per thread and tile
  constexpr float kLazy = 8.0f;  // a row's reference maximum moves only when a score passes it by 2^8 (weights stay <= 256)
  // two images of every staged tile: tile kt + 1 is written while tile kt is read (one barrier per tile)
  __shared__ __attribute__((aligned(16))) bf16_t K_s2[2][32 * KLD];
  __shared__ __attribute__((aligned(16))) bf16_t Vt_s2[2][DV * kVPad];
  __shared__ float bias_s2[2][BIAS ? NB : 1];  // the tile's bias by (row - key + 31): the workgroup's rows, keys 0..31 of the tile
  extern __shared__ int pages_s[];  // the item's block table over this workgroup's key range (dynamic size)
  // workgroup -> (item, head, row tile).  XCD x (workgroups x, x + 8, ...) takes the units x, x + 8, ... of p.unit neighbouring
  // heads of an item, all row tiles of a head in a row, so a head's keys and values pass through one L2; of these the last
  // rows see the most keys: they start first.  (Whole heads in turn, not a run of items each: items of unequal length would
  // leave XCDs idle.)
  const int tiles = p.tiles_per_item;
  int it, h, tile;
  if (p.unit) {
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
    const int pair = (local / (p.unit * tiles) * 8 + xcd) * p.unit + local / tiles % p.unit;
    it = pair / p.H, h = pair % p.H, tile = tiles - 1 - local % tiles;
  } else {
    const int per_head = gridDim.x / p.H, at = blockIdx.x % per_head;
    it = at / tiles, h = blockIdx.x / per_head, tile = tiles - 1 - at % tiles;
  }
  const int q_begin = p.cu_q[it], q_end = p.cu_q[it + 1];
  const int row0 = q_begin + tile * ROWS;
  if (row0 >= q_end) return;
  const int H = p.H, g = h / (H / p.G), G = p.G;
  const int nrows = min(ROWS, q_end - row0);
  const int k_len = p.k_lens[it];
  const int pos0 = p.positions[row0], pos_last = pos0 + nrows - 1;  // positions ascend by one along the rows
  // first visible key of the row at position i: the later of its window's and its chunk's start (ascends with i)
  auto lo_of = [&](int i) { return max(max(0, i - p.window + 1), p.chunk > 0 ? i - i % p.chunk : 0); };
  const int j_lo = lo_of(pos0), j_hi = min(pos_last, k_len - 1);
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, g4 = lane >> 4;
  const int* table = p.block_tables + (size_t)it * p.bt_width;
  const int BS = p.block_size, bsh = p.bs_shift;
  // page and offset of key j (a runtime division would cost tens of instructions per load)
  auto page_ix = [&](int j) { return j >> bsh; };
  auto page_off = [&](int j) { return j & (BS - 1); };
  typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

  const int wrow = 16 * QS * w;  // this wave's first row; lane r16 of row block qs: row wrow + 16 qs + r16
  short8 qhi[QS][ND], qlo[QS][ND];
#pragma unroll
  for (int qs = 0; qs < QS; ++qs)
#pragma unroll
    for (int kd = 0; kd < ND; ++kd) {
      float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      const int qrow = wrow + 16 * qs + r16;
      if (qrow < nrows) {
        const float* qp = p.q + ((size_t)(row0 + qrow) * H + h) * D + kd * 32 + 8 * g4;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = qp[e];
      }
      split8(x, qhi[qs][kd], qlo[qs][kd]);
    }
  const int w_min = pos0 + wrow, w_max = min(w_min + 16 * QS - 1, pos_last);  // this wave's positions
  const int w_lo_min = lo_of(w_min), w_lo_max = lo_of(max(w_max, w_min));     // and their first visible keys
  const bool wave_live = wrow < nrows, wave_full = w_max - w_min == 16 * QS - 1;
  const float cap_k = p.cap > 0.f ? 2.0f * kLog2e / p.cap : 0.f;

  float4v O[QS][NV];
  float m[QS], l[QS];  // l: this lane's share of the row's sum (its keys only; the four lanes of a row meet at the end)
#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    m[qs] = -1e30f;
    l[qs] = 0.f;
#pragma unroll
    for (int n = 0; n < NV; ++n) O[qs][n] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  const float* bias_h = BIAS ? p.bias + (size_t)h * p.window : nullptr;

  const int pg0 = page_ix((j_lo / 32) * 32);  // first page of the workgroup's key range
  // a tile's words are fetched into registers one tile ahead (the loads fly while the previous tile is computed)
  uint4v kreg[KCH], vreg[VCH];
  float breg = 0.f;
  auto fetch = [&](int kt) {
#pragma unroll
    for (int u = 0; u < KCH; ++u) {
      const int c = tid + 256 * u;
      const int key = c / (D / 8), dc = c % (D / 8);
      const int j = kt * 32 + key;
      kreg[u] = uint4v{0u, 0u, 0u, 0u};
      if (c < 32 * (D / 8) && j <= j_hi) {
        const long long page = pages_s[page_ix(j) - pg0];
        kreg[u] = *reinterpret_cast<const uint4v*>(p.k_cache + page * p.kb_stride + ((long long)page_off(j) * G + g) * D + dc * 8);
      }
    }
    // V: 8 groups of 4 keys; a 16-byte word = 2 value columns x 4 keys
#pragma unroll
    for (int u = 0; u < VCH; ++u) {
      const int c = tid + 256 * u;
      const int kg = c / (DV / 2), dc = c % (DV / 2);
      const int j = kt * 32 + 4 * kg;
      vreg[u] = uint4v{0u, 0u, 0u, 0u};
      if (c < 8 * (DV / 2) && j <= j_hi) {
        const long long page = pages_s[page_ix(j) - pg0];
        vreg[u] = *reinterpret_cast<const uint4v*>(p.v_cache + page * p.vb_stride + (long long)(page_off(j) >> 2) * (4LL * G * DV) +
                                                   4LL * (g * DV + 2 * dc));
      }
    }
    if constexpr (BIAS) {
      if (tid < NB) {
        const int dist = pos0 - kt * 32 - 31 + tid;  // (row - key + 31) = tid
        breg = dist >= 0 && dist < p.window ? bias_h[dist] * kLog2e : 0.f;  // the softmax runs in the log2 domain
      }
    }
  };
  auto stash = [&](int buf) {
    bf16_t* K_s = K_s2[buf];
    bf16_t* Vt_s = Vt_s2[buf];
#pragma unroll
    for (int u = 0; u < KCH; ++u) {
      const int c = tid + 256 * u;
      if (c < 32 * (D / 8)) *reinterpret_cast<uint4v*>(&K_s[(c / (D / 8)) * KLD + (c % (D / 8)) * 8]) = kreg[u];
    }
#pragma unroll
    for (int u = 0; u < VCH; ++u) {
      const int c = tid + 256 * u;
      if (c < 8 * (DV / 2)) {
        const int kg = c / (DV / 2), dc = c % (DV / 2);
        // key group kg (keys 4 kg ..) is k-slots 8 (kg & 3) + 4 (kg >> 2) ..: a lane group's 8 slots lie together
        const int at = 8 * (kg & 3) + 4 * (kg >> 2);
        *reinterpret_cast<uint2v*>(&Vt_s[(2 * dc) * kVPad + at]) = uint2v{vreg[u][0], vreg[u][1]};
        *reinterpret_cast<uint2v*>(&Vt_s[(2 * dc + 1) * kVPad + at]) = uint2v{vreg[u][2], vreg[u][3]};
      }
    }
    if constexpr (BIAS) {
      if (tid < NB) bias_s2[buf][tid] = breg;
    }
  };

  const int kt_lo = j_lo / 32, kt_hi = j_hi / 32;
  // the pages of keys [32 kt_lo, j_hi] once, so a tile's loads do not wait for a table lookup first
  const int npg = page_ix(j_hi) - pg0 + 1;
  for (int c = tid; c < npg; c += 256) pages_s[c] = table[pg0 + c];
  __syncthreads();
  fetch(kt_lo);
  stash(0);
  __syncthreads();
  for (int kt = kt_lo; kt <= kt_hi; ++kt) {
    const int cur = (kt - kt_lo) & 1;
    const bf16_t* K_s = K_s2[cur];
    const bf16_t* Vt_s = Vt_s2[cur];
    const float* bias_s = bias_s2[cur];
    if (kt < kt_hi) fetch(kt + 1);
    // the tile's keys [32 kt, 32 kt + 31] against this wave's rows: nothing visible -> nothing to compute
    if (wave_live && kt * 32 <= w_max && kt * 32 + 31 >= w_lo_min) {
      // a K fragment read from LDS serves QS row blocks
      float4v sacc[QS][2];
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
        for (int qs = 0; qs < QS; ++qs) sacc[qs][sub] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kd = 0; kd < ND; ++kd) {
          const short8 a = *reinterpret_cast<const short8*>(&K_s[(sub * 16 + r16) * KLD + kd * 32 + 8 * g4]);
#pragma unroll
          for (int qs = 0; qs < QS; ++qs) sacc[qs][sub] = mfma16(a, qhi[qs][kd], sacc[qs][sub]);
#pragma unroll
          for (int qs = 0; qs < QS; ++qs) sacc[qs][sub] = mfma16(a, qlo[qs][kd], sacc[qs][sub]);
        }
      }
      // every key of the tile visible to every row of the wave: no masks
      const bool inner = kt * 32 + 31 <= w_min && kt * 32 >= w_lo_max && wave_full;
      short8 ph[QS], pl[QS];
#pragma unroll
      for (int qs = 0; qs < QS; ++qs) {
        const int qrow = wrow + 16 * qs + r16, i_q = pos0 + qrow;
        float s[8];
        float mx = -1e30f;
        if (p.cap > 0.f) {
#pragma unroll
          for (int e = 0; e < 8; ++e) sacc[qs][e >> 2][e & 3] = softcap_f(sacc[qs][e >> 2][e & 3], p.cap, cap_k);
        }
        const float* brow = BIAS ? bias_s + (qrow + 31 - 4 * g4) : nullptr;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = sacc[qs][e >> 2][e & 3];
          if constexpr (BIAS) s[e] = fmaf(x, kLog2e, -brow[-((e >> 2) * 16 + (e & 3))]);
          else s[e] = x * kLog2e;
        }
        if (!inner) {
          const int lo_q = lo_of(i_q);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int j = kt * 32 + (e >> 2) * 16 + 4 * g4 + (e & 3);
            if (!(qrow < nrows && j <= i_q && j >= lo_q)) s[e] = -1e30f;
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, s[e]);
        mx = row_max4(mx);
        if (__any(mx > m[qs] + kLazy)) {   // (wave-uniform; the running maxima settle after the first tiles)
          const float m_new = fmaxf(m[qs], mx);
          const float alpha = __builtin_amdgcn_exp2f(m[qs] - m_new);
          m[qs] = m_new;
          l[qs] *= alpha;
          float ar[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, 4 * g4 + r, 64);
#pragma unroll
          for (int n = 0; n < NV; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) O[qs][n][r] *= ar[r];
        }
        float pe[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pe[e] = __builtin_amdgcn_exp2f(s[e] - m[qs]);
        if (!inner) {
#pragma unroll
          for (int e = 0; e < 8; ++e) pe[e] = s[e] > -1e29f ? pe[e] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) l[qs] += pe[e];
        split8(pe, ph[qs], pl[qs]);
      }
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const short8 b = *reinterpret_cast<const short8*>(&Vt_s[(n * 16 + r16) * kVPad + 8 * g4]);
#pragma unroll
        for (int qs = 0; qs < QS; ++qs) O[qs][n] = mfma16(ph[qs], b, O[qs][n]);
#pragma unroll
        for (int qs = 0; qs < QS; ++qs) O[qs][n] = mfma16(pl[qs], b, O[qs][n]);
      }
    }  // (this wave's work on the tile)
    if (kt < kt_hi) stash(cur ^ 1);  // every wave left that image at the previous barrier
    __syncthreads();
  }
  if (!wave_live) return;
#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    float ls = row_sum4(l[qs]), a_fin = 1.0f;
    if (p.sink) {  // the sink's share: one more term of the denominator, nothing added to O
      const float sk = p.sink[h] * kLog2e, mf = fmaxf(m[qs], sk);
      a_fin = __builtin_amdgcn_exp2f(m[qs] - mf);
      ls = ls * a_fin + __builtin_amdgcn_exp2f(sk - mf);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float lr = __shfl(ls, 4 * g4 + r, 64);
      const float inv = (lr > 0.f ? 1.0f / lr : 0.f) * __shfl(a_fin, 4 * g4 + r, 64);
      const int row = wrow + 16 * qs + 4 * g4 + r;
      if (row < nrows) {
        bf16_t* orow = p.out + (size_t)(row0 + row) * p.ldo + (size_t)h * DV;
#pragma unroll
        for (int n = 0; n < NV; ++n) orow[n * 16 + r16] = f2bf(O[qs][n][r] * inv);
      }
    }
  }
}

template <int ND, int QS, bool BIAS>
int launch_mfma_nv(const WAttnMfmaParams& p, int nv, unsigned grid, size_t shm, hipStream_t s) {
  switch (nv) {
    case 2: window_attn_mfma_kernel<ND, 2, QS, BIAS><<<grid, 256, shm, s>>>(p); break;
    case 4: window_attn_mfma_kernel<ND, 4, QS, BIAS><<<grid, 256, shm, s>>>(p); break;
    case 8: window_attn_mfma_kernel<ND, 8, QS, BIAS><<<grid, 256, shm, s>>>(p); break;
    default: return -1;
  }
  return (int)hipGetLastError();
}

template <int ND, int QS>
int launch_mfma_bias(const WAttnMfmaParams& p, int nv, unsigned grid, size_t shm, hipStream_t s) {
  return p.bias ? launch_mfma_nv<ND, QS, true>(p, nv, grid, shm, s) : launch_mfma_nv<ND, QS, false>(p, nv, grid, shm, s);
}

// Whether the matrix-core kernel takes these sizes (bf16 cache only).
extern "C" int r32_window_attn_mfma_ok(int D, int Dv) {
  return (D == 32 || D == 64 || D == 128 || D == 192) && (Dv == 32 || Dv == 64 || Dv == 128);
}

extern "C" int r32_window_attn_mfma(const float* q, const void* k_cache, const void* v_cache, long long kb_stride,
                                    long long vb_stride, int block_size, const int* positions, const int* cu_q,
                                    const int* k_lens, int n_items, int T, int max_q, const int* block_tables, int bt_width,
                                    const float* bias, const float* sink, int window, int chunk, float cap, void* out, int ldo, int H, int G,
                                    int D, int Dv, hipStream_t s) {
  if (n_items <= 0 || max_q <= 0) return 0;
  if (!r32_window_attn_mfma_ok(D, Dv) || H % G != 0 || (block_size & (block_size - 1)) != 0) return -1;
  WAttnMfmaParams p;
  p.q = q; p.k_cache = (const bf16_t*)k_cache; p.v_cache = (const bf16_t*)v_cache;
  p.kb_stride = kb_stride; p.vb_stride = vb_stride; p.block_size = block_size; p.positions = positions;
  p.bs_shift = -1;
  for (int b = 0; b < 20; ++b)
    if ((1 << b) == block_size) p.bs_shift = b;
  // The XCDs' units: the heads of one key head (they share its keys) where every XCD then has as much of every item, else single
  // heads.  us, 32 heads over 8 of 128: 8 x 2048 tokens 750, with workgroups in plain order 1110; prompts of unequal length, a
  // run of items per XCD instead: 8 of 400 tokens and 56 of 10 510, so 67; one of 1000 and 63 of 20 309 / 95.
  p.unit = G % 8 == 0 ? H / G : (long long)n_items * H % 8 == 0 ? 1 : 0;
  int qs = D == 192 && T > 64LL * n_items && T / 128LL * H >= kWideFrom ? 2 : 1;
  // a workgroup's keys span at most window + its rows - 1 positions (from a 32-aligned start: + 31) and never more than the
  // table: its pages' part of the table goes to LDS
  auto table = [&](int rows) {
    const long long span = std::min((long long)window + rows - 1 + 31, (long long)bt_width * block_size);
    return (size_t)(span / block_size + 2) * sizeof(int);
  };
  if (table(64 * qs) > 48 * 1024) qs = 1;
  const size_t shm = table(64 * qs);
  if (shm > 48 * 1024) return -2;
  p.cu_q = cu_q; p.k_lens = k_lens; p.tiles_per_item = (max_q + 64 * qs - 1) / (64 * qs); p.block_tables = block_tables;
  p.bt_width = bt_width; p.bias = bias; p.sink = sink; p.window = window; p.chunk = chunk; p.cap = cap; p.out = (bf16_t*)out; p.ldo = ldo; p.H = H; p.G = G;
  const long long wgs = (long long)n_items * p.tiles_per_item * H;
  if (wgs >= (1LL << 31)) return -3;
  const unsigned grid = (unsigned)wgs;
  switch (D / 32) {
    case 1: return launch_mfma_bias<1, 1>(p, Dv / 16, grid, shm, s);
    case 2: return launch_mfma_bias<2, 1>(p, Dv / 16, grid, shm, s);
    case 4: return launch_mfma_bias<4, 1>(p, Dv / 16, grid, shm, s);
    case 6: return qs == 2 ? launch_mfma_bias<6, 2>(p, Dv / 16, grid, shm, s) : launch_mfma_bias<6, 1>(p, Dv / 16, grid, shm, s);
  }
  return -1;
}
