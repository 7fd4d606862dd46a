// Decode rows of the sliding-window attention (see wattn.hip for the scores, the cache layout and the portion kernel).
#pragma once
#include "elem.h"

using namespace lwc;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

LWC_DEVICE float4v mfma16(const short8& a, const short8& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// ---------------------------------------------------------------------------------------------------------
// window_attn_decode_kernel: one new token per sequence on the matrix cores (bf16 cache), split over the keys.
//
// One wave per (sequence b, key/value head g, head chunk, key split).  The N = 16 columns of the MFMA are the
// (up to 16) query heads that share head g, so K and V are read ONCE for all of them, straight from the paged
// cache into the operands — no LDS: a K row's 16 bytes are an A operand as they lie, the interleaved V word is a
// B operand as it lies.  Same arithmetic as the portion kernel (hi + lo halves of q and of the weights, bias
// table, fp32 online softmax).  Bound by the reads of the cache: 64 sequences of 500 to 1500 keys (1000 on average), 32
// heads over 8 of 128 entries, take 67 us for 258 MB from memory (42 us at the rate of a plain read) in tables of 4096 keys.
// (With the splits cut for the table's width and every load of a tile waited for on its own 2.5 times as long, 1.8 times at
// 2048 keys each.)  Each split leaves an unnormalised partial (o, m, l); the reduce kernel merges
// them (splits == 1: still through the reduce, which then only normalises).
struct WAttnDecodeParams {
  const float* q;          // [B, H*D]
  const bf16_t* k_cache;
  const bf16_t* v_cache;
  long long kb_stride, vb_stride;
  int block_size, bs_shift;  // block_size = 1 << bs_shift (the matrix-core kernels take power-of-two pages)
  const int* positions;    // [B]: the new token's position (its key is already in the cache)
  const int* block_tables;
  int bt_width;
  const float* bias;       // [H, window], or null: no distance bias
  int window;
  int chunk;               // > 0: the row sees only keys of its own chunk, j >= i - i % chunk (besides the window)
  float cap;               // > 0: scores become cap tanh(score / cap)
  float* part_o;           // [B, H, S, Dv]
  float* part_ml;          // [B, H, S, 2]
  int H, G, S, min_keys;  // min_keys: the fewest keys a split takes before the next one gets any (a multiple of 32)
};

struct HeadChunk {
  int g, h0, nh, last;  // kv head; first head, heads (<= 0: a wave past the last chunk only helps staging); the kv head's last one
};
// Chunk cw of the NC (below) of workgroup y.
LWC_HOST_DEVICE HeadChunk head_chunk(int y, int cw, int NC, int Hg) {
  const int cgroups = ((Hg + 15) / 16 + NC - 1) / NC;  // workgroups per kv head
  const int g = y / cgroups, h0 = g * Hg + ((y % cgroups) * NC + cw) * 16, end = g * Hg + Hg;
  return {g, h0, end - h0 < 16 ? end - h0 : 16, end - 1};
}
// The head whose q (and bias) column r16 of the MFMA loads: a column, or a whole wave, that has none loads one that there is
LWC_HOST_DEVICE int loaded_head(const HeadChunk& c, int r16) {
  return r16 < c.nh ? c.h0 + r16 : c.h0 < c.last ? c.h0 : c.last;
}

// NW waves per workgroup share one (sequence, head chunk, split).  With NW > 1 a tile's 32 key rows go through LDS
// once for all the waves (fetched into registers one tile ahead), and each wave owns NV / NW of the 16-column value
// tiles (wide value rows: the accumulators of one wave would leave no registers for loads in flight).  NW = 4: the
// waves also form the tile's scores together, each a quarter of the MFMAs (one key subtile times half of the row's
// 32-entry slices), and the partial scores meet in LDS.
// QLO = false: q enters as its bf16 rounding only (one MFMA per operand instead of two).
// VK = true (with NW > 1): the values ARE the first DV entries of the key rows (a cached latent that is key and value
// at once), so the value operands are gathered from the staged rows in LDS and the value pages are not read at all.
// NC > 1: NC head chunks (16 heads each) of one kv head share the workgroup and with it every staged key row (waves
// [c NW, (c + 1) NW) serve chunk c).
template <int ND, int NV, int NW = 1, bool QLO = true, bool VK = false, int NC = 1>
__global__ void __launch_bounds__(64 * NW * NC) window_attn_decode_kernel(const WAttnDecodeParams p) {
  constexpr int D = 32 * ND, DV = 16 * NV, NVW = NV / NW, NT = 64 * NW * NC;  // NT: threads of the workgroup
  static_assert(NV % NW == 0, "value tiles divide among the waves");
  const int b = blockIdx.x, split = blockIdx.z;
  const int H = p.H, G = p.G;
  // (one wave: the wave index is a compile-time zero, so the value tiles' offsets stay immediates)
  const int lane = NT > 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x, wv_all = NT > 64 ? (int)(threadIdx.x >> 6) : 0;
  const int wv = NC > 1 ? wv_all % NW : wv_all, cw = NC > 1 ? wv_all / NW : 0;
  const HeadChunk heads = head_chunk(blockIdx.y, cw, NC, H / G);
  const int g = heads.g, h0 = heads.h0, nh = heads.nh;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int i = p.positions[b];
  const int j_lo = max(max(0, i - p.window + 1), p.chunk > 0 ? i - i % p.chunk : 0);
  // The row's own keys divide among the splits (a multiple of 32 each): the host only knows the longest context there
  // could be, and ranges cut for that one would leave the whole row to the first split.
  const int first = (j_lo / 32) * 32, n_keys = max(i + 1 - first, 0);
  const int keys_per_split = max(((n_keys + p.S - 1) / p.S + 31) / 32 * 32, p.min_keys);
  const int base = first + split * keys_per_split;  // this split's first key (a multiple of 32)
  const int last = min(i, base + keys_per_split - 1);
  const int* table = p.block_tables + (size_t)b * p.bt_width;
  const int BS = p.block_size, bsh = p.bs_shift;
  auto page_ix = [&](int j) { return j >> bsh; };
  auto page_off = [&](int j) { return j & (BS - 1); };
  // 64 pages from the tile at hand's, one per lane: a key's page then comes from a lane exchange instead of a table load that
  // every K / V load would have to wait for.  A tile and the next one's rows need 64 pages at most.  (The exchange in `look_up` is the
  // load's wait, in the branch that loads: behind it, or behind a choice between lanes and table, the compiler waits for every load on
  // its way, three times a tile and, with wide rows, at every row that a thread stages.  us, so / here, cold: 576 / 512 entries, 32
  // heads, 64 rows of 500 to 1500 keys 98 / 61, of 4000 199 / 122, one of 4000 54 / 33; 320 / 256, 16 heads 49 / 32, 97 / 68, 36 / 25; 128 /
  // 128, 32 heads over 8, 255 rows of 400 89 / 87, 64 of 20 to 60 15.6 / 13.0, 64 of 500 to 1500 67.5 / 67.4, which memory bounds; over 32,
  // 64 of 100 to 4000 400 / 337, but of 1000 each 181 / 188 and with a bias 180 / 194: more in flight is no gain to equal rows that fill the chip.)
  int pg_base = 0, my_page = 0;
  auto look_up = [&](int t0) {
    pg_base = page_ix(t0);
    my_page = __shfl(table[min(pg_base + lane, page_ix(i))], lane, 64);
  };
  if (base <= last) look_up(base);
  auto page_of = [&](int j) { return __shfl(my_page, page_ix(j) - pg_base, 64); };
  const bool h_valid = r16 < nh;
  const int h = loaded_head(heads, r16);

  // With NW = 4 staged waves the scores of a tile are formed ONCE per chunk: wave w multiplies key subtile (w & 1) with
  // half (w >> 1) of the row's 32-entry slices, the halves meet through LDS.  Such a wave keeps only its half of q.
  constexpr bool kSplitQK = NW == 4;
  static_assert(!kSplitQK || ND % 2 == 0, "the slices divide into two halves");
  constexpr int NDW = kSplitQK ? ND / 2 : ND;
  const int kd0 = kSplitQK ? (wv >> 1) * NDW : 0;
  short8 qhi[NDW], qlo[QLO ? NDW : 1];
#pragma unroll
  for (int kd = 0; kd < NDW; ++kd) {
    typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
    const float4u* qp = reinterpret_cast<const float4u*>(p.q + ((size_t)b * H + h) * D + (kd0 + kd) * 32 + 8 * g4);
    const float4u x0 = qp[0], x1 = qp[1];
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = h_valid ? e < 4 ? x0[e] : x1[e - 4] : 0.f;
    short8 lo;
    split8(x, qhi[kd], lo);
    if (QLO) qlo[kd] = lo;
  }
  float4v O[NVW];
#pragma unroll
  for (int n = 0; n < NVW; ++n) O[n] = float4v{0.f, 0.f, 0.f, 0.f};
  float m = -1e30f, l = 0.f;
  const float cap_k = p.cap > 0.f ? 2.0f * 1.4426950408889634f / p.cap : 0.f;
  const bool biased = p.bias != nullptr;  // no table: no distance bias
  const float* bias_h = p.bias + (size_t)h * p.window;

  constexpr bool kStage = NW > 1;
  constexpr int KLD = D + 8;                                       // LDS row stride: rows start in different banks
  constexpr int KCH = (32 * (D / 8) + NT - 1) / NT;                 // 16-byte words per thread and tile
  __shared__ __attribute__((aligned(16))) bf16_t K_s[kStage ? 32 * KLD : 8];
  __shared__ __attribute__((aligned(16))) float4v S_x[NW == 4 ? NC * NW * 64 : 1];  // partial scores of the waves
  uint4v kreg[kStage ? KCH : 1];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int u = 0; u < KCH; ++u) {
      const int c = min((int)threadIdx.x + NT * u, 32 * (D / 8) - 1);
      const int key = c / (D / 8), dc = c % (D / 8);
      const int j = min(t0 + key, i);  // (rows past the token are masked below: any valid row does)
      kreg[u] = *reinterpret_cast<const uint4v*>(p.k_cache + (long long)page_of(j) * p.kb_stride +
                                                 ((long long)page_off(j) * G + g) * D + dc * 8);
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int u = 0; u < KCH; ++u) {
      const int c = (int)threadIdx.x + NT * u;
      if (c < 32 * (D / 8)) *reinterpret_cast<uint4v*>(&K_s[(c / (D / 8)) * KLD + (c % (D / 8)) * 8]) = kreg[u];
    }
  };
  if (kStage && base <= last) {
    fetch(base);
    stash();
    __syncthreads();
  }

  // One wave alone (no LDS): a tile's value words are in flight while the scores and the weights of the tile are formed, the next
  // tile's key rows while it is summed.  (Rows past the split's keys are masked below: any valid row does.)
  short8 kf[kStage ? 1 : 2 * ND];
  uint4v vf[kStage ? 1 : NVW];
  auto load_keys = [&](int t0) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int j = min(t0 + sub * 16 + r16, last);
      const bf16_t* kr = p.k_cache + (long long)page_of(j) * p.kb_stride + ((long long)page_off(j) * G + g) * D + 8 * g4;
#pragma unroll
      for (int kd = 0; kd < ND; ++kd) kf[sub * ND + kd] = *reinterpret_cast<const short8*>(kr + kd * 32);
    }
  };
  auto value_row = [&](int j) {
    return p.v_cache + (long long)page_of(j) * p.vb_stride + (long long)(page_off(j) >> 2) * (4LL * G * DV) + 4LL * (g * DV + (kStage ? 1 : 2) * r16);
  };
  if constexpr (!kStage) {
    if (base <= last) load_keys(base);
  }

  for (int t0 = base; t0 <= last; t0 += 32) {  // (base and last are the same for every wave of the workgroup)
    if (page_ix(t0 + 63) - pg_base >= 64) look_up(t0);
    if (kStage && t0 + 32 <= last) fetch(t0 + 32);
    // the lane's two 4-key groups: keys t0 + 4 g4 .. and t0 + 16 + 4 g4 .. (groups past the token: any valid one,
    // their weights are 0)
    const int ja = min(t0 + 4 * g4, (i / 4) * 4), jb = min(t0 + 16 + 4 * g4, (i / 4) * 4);
    const bf16_t *va = nullptr, *vb = nullptr;
    if constexpr (!VK) {
      va = value_row(ja);
      vb = value_row(jb);
    }
    float bias_e[8];
    if (biased) {
#pragma unroll
      for (int e = 0; e < 8; ++e) bias_e[e] = bias_h[min(max(i - (t0 + (e >> 2) * 16 + 4 * g4 + (e & 3)), 0), p.window - 1)];
    }
    if constexpr (!kStage) {
#pragma unroll
      for (int n = 0; n < NVW; n += 2) {  // two columns, 16 n + 2 r16 and the one after it, four keys of each
        vf[n] = *reinterpret_cast<const uint4v*>(va + 64 * n);
        vf[n + 1] = *reinterpret_cast<const uint4v*>(vb + 64 * n);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    float4v sacc[2];
    if constexpr (kSplitQK) {
      float4v part = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kd = 0; kd < NDW; ++kd) {
        const short8 a = *reinterpret_cast<const short8*>(&K_s[((wv & 1) * 16 + r16) * KLD + (kd0 + kd) * 32 + 8 * g4]);
        part = mfma16(a, qhi[kd], part);
        if (QLO) part = mfma16(a, qlo[kd], part);
      }
      S_x[(cw * NW + wv) * 64 + lane] = part;
      __syncthreads();  // (the barriers at the tile's end keep the next tile's partials from overtaking these reads)
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
        sacc[sub] = S_x[(cw * NW + sub) * 64 + lane] + S_x[(cw * NW + sub + 2) * 64 + lane];
    } else {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      sacc[sub] = float4v{0.f, 0.f, 0.f, 0.f};
      if (kStage) {
#pragma unroll
        for (int kd = 0; kd < ND; ++kd) {
          const short8 a = *reinterpret_cast<const short8*>(&K_s[(sub * 16 + r16) * KLD + kd * 32 + 8 * g4]);
          sacc[sub] = mfma16(a, qhi[kd], sacc[sub]);
          if (QLO) sacc[sub] = mfma16(a, qlo[kd], sacc[sub]);
        }
      } else {
#pragma unroll
        for (int kd = 0; kd < ND; ++kd) {
          sacc[sub] = mfma16(kf[sub * ND + kd], qhi[kd], sacc[sub]);
          if (QLO) sacc[sub] = mfma16(kf[sub * ND + kd], qlo[kd], sacc[sub]);
        }
      }
    }
    }  // (scores without the split)
    if (p.cap > 0.f) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sacc[e >> 2][e & 3] = softcap_f(sacc[e >> 2][e & 3], p.cap, cap_k);
    }
    float s[8];
    bool ok[8];
    float mx = -1e30f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int j = t0 + (e >> 2) * 16 + 4 * g4 + (e & 3);
      const int dist = i - j;
      ok[e] = h_valid && dist >= 0 && j >= j_lo && j <= last;
      s[e] = ok[e] ? sacc[e >> 2][e & 3] - (biased ? bias_e[e] : 0.f) : -1e30f;
      mx = fmaxf(mx, s[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m, mx);
    const float alpha = expf(m - m_new);
    float pe[8], psum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      pe[e] = ok[e] ? expf(s[e] - m_new) : 0.f;
      psum += pe[e];
    }
    psum += __shfl_xor(psum, 16, 64);
    psum += __shfl_xor(psum, 32, 64);
    l = l * alpha + psum;
    m = m_new;
    if constexpr (!kStage) {  // (ahead of the softmax, keys and values in flight at once: 64 rows of 500 to 1500 keys 68 us for 66.5)
      __builtin_amdgcn_sched_barrier(0);
      load_keys(t0 + 32);
      __builtin_amdgcn_sched_barrier(0);
    }
    short8 ph, pl;
    split8(pe, ph, pl);
    float ar[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, 4 * g4 + r, 64);
#pragma unroll
    for (int n = 0; n < NVW; ++n) {
#pragma unroll
      for (int r = 0; r < 4; ++r) O[n][r] *= ar[r];
      short8 bb;
      if (kStage && VK) {
        const bf16_t* col = &K_s[(4 * g4) * KLD + 16 * (wv * NVW + n) + r16];  // this lane's value column, key 4 g4
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          bb[e] = (short)col[e * KLD];
          bb[4 + e] = (short)col[(16 + e) * KLD];
        }
      } else if constexpr (!kStage) {
        const uint4v &b0 = vf[n & ~1], &b1 = vf[n | 1];
        bb = __builtin_bit_cast(short8, uint4v{b0[2 * (n & 1)], b0[2 * (n & 1) + 1], b1[2 * (n & 1)], b1[2 * (n & 1) + 1]});
      } else {
        const short4v b0 = *reinterpret_cast<const short4v*>(va + 64 * (wv * NVW + n));
        const short4v b1 = *reinterpret_cast<const short4v*>(vb + 64 * (wv * NVW + n));
        bb = short8{b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
      }
      O[n] = mfma16(ph, bb, O[n]);
      O[n] = mfma16(pl, bb, O[n]);
    }
    if (kStage) {
      __syncthreads();  // every wave has read this tile's rows
      if (t0 + 32 <= last) stash();
      __syncthreads();
    }
  }
  // partials: O rows are heads 4 g4 + r, columns dv 16 n + r16 (a split without keys leaves l = 0 and no row)
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int hr = 4 * g4 + r;
    if (hr < nh && base <= last) {
      float* po = p.part_o + (((size_t)b * H + h0 + hr) * p.S + split) * DV;
#pragma unroll
      for (int n = 0; n < NVW; ++n) po[kStage ? (wv * NVW + n) * 16 + r16 : 32 * (n / 2) + 2 * r16 + n % 2] = O[n][r];
    }
  }
  if (g4 == 0 && h_valid && wv == 0) {
    float* pm = p.part_ml + (((size_t)b * H + h) * p.S + split) * 2;
    pm[0] = m;
    pm[1] = l;
  }
}

