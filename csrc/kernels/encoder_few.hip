// A post-norm encoder over few packed rows (a search query, a handful of short texts), in two launches: begin_kernel sums the
// embeddings and clears the flags, chain_kernel is the whole stack (of up to 24 layers; further ones two launches more).
//
// A text of 12 tokens through bge-small is 12 layers of dependent stages over 42 MB of weights, 7 us of reading: what counts is how
// many stages there are, and what each waits for.  A stage is cut into items of a workgroup each:
//
//   qkv_attn   x = LN(pre) (first layer: LN(word[ids] + pos[positions])); q, k, v of head h = x . W^T + b; a_h = softmax(q k^T) v
//              (wider than 384: project, then attention; a head's 400 KB of weights are 20 us for one compute unit)
//   project    o = a . Wo^T
//   project    y = LN(o + bo + x); h = gelu(y . W1^T + b1)
//   project    PF parts of h . W2^T, a range of K each; pre = their sum + b2 + y, fp32, is formed by the norm that reads it
//
// and a last LN.  Every item of a stage that normalises does so for itself, under the wait for nothing: a stage of its own would be
// 2 us.  A workgroup takes the next item in order (an atomic), loads its weights, waits for the items of the stage before it and
// goes on; the weights of the next 250 items are on their way or in registers by then.  It waits only for items that were taken
// before its own, by workgroups that are running: whatever else runs on the GPU, another such launch too, the lowest item that is
// not done waits for nothing.
//
// As kernels of their own, four or five a layer, a stage was 4.3 us; here it is 2.9 (bge-small: 49 of them): 0.3 us until its stores are in memory, 0.4 to 1 until
// the flags are seen, 0.5 to 0.7 for the rows, 0.45 for a norm, 0.6 for the products and their sum (1.2 with the attention).  One
// MI355X, us a call, kernels / one launch (rows): bge-small 198 / 133 (3), 214 / 143 (14), 282 / 190 (32); bge-base 250 / 219, 274 / 232, 361 / 316;
// bge-large 632 / 558, 699 / 588, 918 / 726.  On the way there, bge-small, 14 rows: 212 as the kernels were; the stage before asked
// first and seldom, half a wave a row in the norm 184; the flags in eight copies 174, one for each XCD 153; what is
// handed on in a place of its own, read through the caches, and 32 columns an item 160 (of 174); one item a CU at a time 143 (of 154; two:
// bge-base 274 for 232).
//
// What it costs others: a workgroup waits in 81 KiB of its CU's LDS, up to 250 of them for the 130 to 720 us of a call, and kernels of another
// stream that want more than the rest wait for it.  Queries of 12 tokens one behind the other beside decode steps, us a step alone, then a
// step and a query beside each other, kernels / here: llama 1 545, 600 and 726 / 523, 667 and 220; 61 rows 790, 836 and 701 / 770, 1095 and 219;
// merudra 64 1084, 1137 and 597 / 1021, 1125 and 261; bge-large beside llama 1 545, 657 and 2400 / 523, 828 and 986.  A query takes 24 to 65 us
// from the steps beside it (28 to 67 before), bge-large's 360 (410), but there are up to three times as many.  And memory: each layer's
// rows keep a place of their own until the call's end, layers + 1 times Rows::kBytes a row: 4 MB at bge-small's 32 rows, 13 at
// bge-base's, 16 and 26 at bge-large's 16 and 32.
//
// project: 16 or 32 output columns, 8 waves over K in steps of 32 (wave w: steps w, w + 8, ..), W the A operand and the rows the B
// operand of mfma_f32_16x16x32_bf16, so that a lane holds four consecutive columns of one row.  qkv_attn: a head, 24 (16 columns,
// part of K) units over 8 waves.  Sums over waves, units and parts in a fixed order.  Two parts of a sum at 384, four at 768 and at
// 1024 up to 16 rows, two beyond.  Rows go in MT tiles of 16; rows past T are zeros and are not stored.
#include <algorithm>

#include "common.h"

namespace lwc {
namespace efew {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));

constexpr int kT = 512, kW = kT / 64;
constexpr int kLayers = 24;  // of one launch: their pointers are kernel arguments
constexpr int kCopies = 8;   // of the flags, one for the workgroups of each XCD: a line that several look at goes back and forth with each store
constexpr int kSC1 = 16;     // cache policy of buffer stores: device scope

LWC_DEVICE float4v mfma(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

LWC_DEVICE float4v widen4(const uint2v& v) {
  return float4v{__uint_as_float(v[0] << 16), __uint_as_float(v[0] & 0xffff0000u), __uint_as_float(v[1] << 16),
                 __uint_as_float(v[1] & 0xffff0000u)};
}
LWC_DEVICE uint2v narrow4(const float4v& v) { return uint2v{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}; }

// What workgroups hand to each other goes to memory at once (device scope), each layer's to a place of its own: nobody has
// read it in this launch before it was whole, so it is read through the caches
LWC_DEVICE uint4v load16(__amdgpu_buffer_rsrc_t r, int at) { return __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0)); }
LWC_DEVICE uint2v load8(__amdgpu_buffer_rsrc_t r, int at) { return __builtin_bit_cast(uint2v, __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0)); }
LWC_DEVICE void store8(const uint2v& v, __amdgpu_buffer_rsrc_t r, int at) { __builtin_amdgcn_raw_buffer_store_b64(v, r, at, 0, kSC1); }

// An item waits for the n items of the stage before it (their flags, one a thread).  Items taken long before their turn look, seldom,
// at the stage before that one first
LWC_DEVICE void wait_for(const int* flags, int n, bool first) {
  auto ready = [](const int* f) { return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; };
  if ((int)threadIdx.x < n) {
    if (!first)
      while (!ready(flags - 1)) __builtin_amdgcn_s_sleep(16);
    while (!ready(flags + threadIdx.x)) __builtin_amdgcn_s_sleep(1);
  }
  __syncthreads();
}
// ... and tells those of the next one, in each copy of the flags, that what it stored has left the compute unit
LWC_DEVICE void done(int* flag, int stride) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x < kCopies) __hip_atomic_store(flag + threadIdx.x * stride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct Norm {
  const float* part;     // [P, T, D]: the parts of what the last projection gave
  const bf16_t* res;     // [T, D] and
  const bf16_t* rbias;   // [D]: the stream and the projection's bias, added to them
  const bf16_t* g;       // [D]
  const bf16_t* b;
  float eps;
  bf16_t* out;           // [T, D]: where the rows go that do not go into LDS
};

// The rows' LayerNorm into LDS, [16 MT][D + 8] (the pad spreads 16 rows' fragments over the banks), half a wave per row.  `ready`
// comes before the loads of the rows, which go in one trip where there is room.
template <int MT, int D, int P, class F>
LWC_DEVICE void norm_rows(const Norm& n, int T, bf16_t* xs, const F& ready) {
  constexpr int RP = 8 * MT / kW, C = D / 128, PB = RP * C * P <= 32 ? P : RP * C * 2 <= 32 ? 2 : 1;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = lane >> 5, at0 = (lane & 31) * 4;
  float4v v[RP][C];
  uint2v g[C], b[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    g[c] = *reinterpret_cast<const uint2v*>(n.g + at0 + 128 * c);
    b[c] = *reinterpret_cast<const uint2v*>(n.b + at0 + 128 * c);
  }
  auto row_of = [&](int i) { return 2 * (w + i * kW) + half; };
  uint2v r[RP][C], rb[C];
#pragma unroll
  for (int c = 0; c < C; ++c) rb[c] = *reinterpret_cast<const uint2v*>(n.rbias + at0 + 128 * c);
  ready();
  // (rows past T lie past the resource's end or in the next part: finite or not, they are not stored, and zeros in LDS)
  const __amdgpu_buffer_rsrc_t rr = uniform_rsrc(n.res, T * D * 2), rp = uniform_rsrc(n.part, P * T * D * 4);
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int c = 0; c < C; ++c) r[i][c] = load8(rr, (row_of(i) * D + at0 + 128 * c) * 2);
#pragma unroll
  for (int p0 = 0; p0 < P; p0 += PB) {
    float4v t[PB][RP][C];
#pragma unroll
    for (int q = 0; q < PB; ++q)
#pragma unroll
      for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int c = 0; c < C; ++c)
          t[q][i][c] = __builtin_bit_cast(float4v, load16(rp, ((min(p0 + q, P - 1) * T + row_of(i)) * D + at0 + 128 * c) * 4));
#pragma unroll
    for (int q = 0; q < PB; ++q)
#pragma unroll
      for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int j = 0; j < 4; ++j) v[i][c][j] = p0 + q == 0 ? t[q][i][c][j] : p0 + q < P ? v[i][c][j] + t[q][i][c][j] : v[i][c][j];
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const float4v q = widen4(rb[c]);
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const float4v x = widen4(r[i][c]);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][c][j] += q[j] + x[j];
    }
  }
  auto sum32 = [](float x) {
    x = row16_sum(x);
    const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
  };
  float s[RP], s2[RP];
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    s[i] = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) s[i] += (v[i][c][0] + v[i][c][1]) + (v[i][c][2] + v[i][c][3]);
  }
#pragma unroll
  for (int i = 0; i < RP; ++i) s[i] = sum32(s[i]) * (1.f / D);
#pragma unroll
  for (int i = 0; i < RP; ++i) {
    s2[i] = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[i][c][j] -= s[i];
        s2[i] = fmaf(v[i][c][j], v[i][c][j], s2[i]);
      }
  }
#pragma unroll
  for (int i = 0; i < RP; ++i) s2[i] = rsqrtf(sum32(s2[i]) * (1.f / D) + n.eps);
  const __amdgpu_buffer_rsrc_t ro = uniform_rsrc(n.out, T * D * 2);
#pragma unroll
  for (int i = 0; i < RP; ++i)
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const float4v gf = widen4(g[c]), bf = widen4(b[c]);
      float4v y;
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = fmaf(v[i][c][j] * s2[i], gf[j], bf[j]);
      uint2v o = narrow4(y);
      if (xs) {
        if (row_of(i) >= T) o = uint2v{0u, 0u};
        *reinterpret_cast<uint2v*>(xs + row_of(i) * (D + 8) + at0 + 128 * c) = o;
      } else {
        store8(o, ro, row_of(i) < T ? (row_of(i) * D + at0 + 128 * c) * 2 : 0x7ffffff0);
      }
    }
}

// ---- attention: a head's q, k [16 MT][DH + 8], v transposed [DH][TK + 8] and probabilities [16 MT][TK + 8] in LDS ----
template <int MT, int DH>
struct Head {
  static constexpr int TK = MT == 1 ? 32 : 16 * MT;  // keys, a multiple of the MFMA's 32
  static constexpr int kK = 16 * MT * (DH + 8) * 2;
  static constexpr int kV = kK + 16 * MT * (DH + 8) * 2;
  static constexpr int kP = kV + DH * (TK + 8) * 2;
  static constexpr int kBytes = kP + 16 * MT * (TK + 8) * 2;
};

// o = softmax(q k^T scale) v of 16 queries a wave, the first MT waves.  Scores, transposed: lane (r16, g) holds query r16's keys
// 16 j + 4 g ..; bounds: lane s the first row of text s
template <int MT, int DH>
LWC_DEVICE void attend(const uint8_t* lds, int bounds, int nseq, int T, int D, int h, float scale, bf16_t* a) {
  using L = Head<MT, DH>;
  constexpr int TK = L::TK;
  const bf16_t *qs = reinterpret_cast<const bf16_t*>(lds), *ks = reinterpret_cast<const bf16_t*>(lds + L::kK);
  const bf16_t* vs = reinterpret_cast<const bf16_t*>(lds + L::kV);
  bf16_t* ps = reinterpret_cast<bf16_t*>(const_cast<uint8_t*>(lds) + L::kP);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int qi = 16 * w + r16;
  int lo = 0, hi = 0;  // the keys of the query's text
  for (int s = 0; s < nseq; ++s) {
    const int a0 = __builtin_amdgcn_readlane(bounds, s), b0 = __builtin_amdgcn_readlane(bounds, s + 1);
    if (a0 <= qi && qi < b0) lo = a0, hi = b0;
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
      sc[j][r] = key >= lo && key < hi ? sc[j][r] * scale : -INFINITY;
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
  const __amdgpu_buffer_rsrc_t ra = uniform_rsrc(a, T * D * 2);
#pragma unroll
  for (int c = 0; c < DH / 16; ++c)
    if (qi < T) store8(narrow4(o[c]), ra, (qi * D + h * DH + 16 * c + 4 * g) * 2);
}

// ---- a head's projection and attention ----
template <int MT, int D, int DH>
struct QkvAttnLds {
  static constexpr int kX = 16 * MT * (D + 8) * 2;
  static constexpr int kRed = 24 * MT * 1024;  // the units' partials, over the rows that they are done with
  static constexpr int kHead = kX > kRed ? kX : kRed;
  static constexpr int kBytes = kHead + Head<MT, DH>::kBytes;
};

template <int MT, int D, int DH, int P, class F>
LWC_DEVICE void qkv_attn(const Norm& n, const bf16_t* W, const bf16_t* bias_, const int* cu, bf16_t* a, int T, int nseq, float scale, int h,
                         uint8_t* smem, const F& ready) {
  using L = QkvAttnLds<MT, D, DH>;
  using LH = Head<MT, DH>;
  constexpr int NT = 3 * DH / 16, SPLIT = 24 / NT, KU = D / 32 / SPLIT, TK = LH::TK;
  static_assert(NT * SPLIT == 24 && KU * 32 * SPLIT == D, "24 units of whole K steps");
  bf16_t* xs = reinterpret_cast<bf16_t*>(smem);
  float4v* red = reinterpret_cast<float4v*>(smem);
  bf16_t* qs = reinterpret_cast<bf16_t*>(smem + L::kHead);
  bf16_t* ks = reinterpret_cast<bf16_t*>(smem + L::kHead + LH::kK);
  bf16_t* vs = reinterpret_cast<bf16_t*>(smem + L::kHead + LH::kV);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;

  // unit u of 24: 16 columns (q, k or v's) tt = u / SPLIT, K part u % SPLIT
  uint4v wf[3][KU];
  uint2v bias[(NT * MT * 64 + kT - 1) / kT];
#pragma unroll
  for (int i = 0; i < (NT * MT * 64 + kT - 1) / kT; ++i) {
    const int o = min(tid + i * kT, NT * MT * 64 - 1), tt = o / 64 / MT;
    bias[i] = *reinterpret_cast<const uint2v*>(bias_ + tt / (DH / 16) * D + h * DH + tt % (DH / 16) * 16 + 4 * ((o & 63) >> 4));
  }
  const int bounds = cu[min(lane, nseq)];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int u = w * 3 + i, tt = u / SPLIT, row = tt / (DH / 16) * D + h * DH + tt % (DH / 16) * 16 + r16;
#pragma unroll
    for (int s = 0; s < KU; ++s) wf[i][s] = *reinterpret_cast<const uint4v*>(W + (size_t)row * D + u % SPLIT * KU * 32 + 8 * g + s * 32);
  }
  norm_rows<MT, D, P>(n, T, xs, ready);
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
  if (w < MT) attend<MT, DH>(smem + L::kHead, bounds, nseq, T, D, h, scale, a);
}

// ---- a head's attention over projected rows qkv [T, 3 D] ----
template <int MT, int D, int DH, class F>
LWC_DEVICE void attention(const bf16_t* qkv, const int* cu, bf16_t* a, int T, int nseq, float scale, int h, uint8_t* smem, const F& ready) {
  using L = Head<MT, DH>;
  constexpr int TK = L::TK, kChunks = 3 * 16 * MT * (DH / 8);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bounds = cu[min(lane, nseq)];
  bf16_t* vs = reinterpret_cast<bf16_t*>(smem + L::kV);
  if (TK > 16 * MT)
    for (int i = tid; i < DH * 16; i += kT) vs[i / 16 * (TK + 8) + 16 + i % 16] = 0;
  ready();
  const __amdgpu_buffer_rsrc_t r = uniform_rsrc(qkv, T * 3 * D * 2);
#pragma unroll
  for (int i = 0; i < (kChunks + kT - 1) / kT; ++i) {
    const int o = tid + i * kT;
    if (o >= kChunks) break;
    const int col = o % (DH / 8) * 8, row = o / (DH / 8) % (16 * MT), which = o / (DH / 8) / (16 * MT);
    const uint4v v = load16(r, row < T ? (row * 3 * D + which * D + h * DH + col) * 2 : 0x7ffffff0);  // (past T: zeros)
    if (which < 2) {
      *reinterpret_cast<uint4v*>(smem + which * L::kK + (row * (DH + 8) + col) * 2) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) vs[(col + j) * (TK + 8) + row] = (bf16_t)(v[j >> 1] >> (16 * (j & 1)));
    }
  }
  __syncthreads();
  if (w < MT) attend<MT, DH>(smem, bounds, nseq, T, D, h, scale, a);
}

enum Out { OUT_PART = 0, OUT_BIAS = 1, OUT_GELU = 2 };

// 16 NC columns (from n0) of the product of the rows' K columns from k0 with W [N, lda].  P > 0: the rows are normalised here, from P
// parts; else they are A's [T, lda].  OUT_PART: part [T, N] fp32; else h [T, N] bf16
template <int MT, int NC, int K, int P, int OUT, class F>
LWC_DEVICE void project(const Norm& n, const bf16_t* A, const bf16_t* W, const bf16_t* bias_, float* part, bf16_t* h, int T, int N, int lda,
                        int n0, int k0, uint8_t* smem, const F& ready) {
  constexpr int S = K / 32, PER = (S + kW - 1) / kW;
  float4v* red = reinterpret_cast<float4v*>(smem);
  bf16_t* xs = reinterpret_cast<bf16_t*>(smem + kW * NC * MT * 1024);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  uint4v wf[NC][PER];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const bf16_t* wr = W + (size_t)(n0 + 16 * c + r16) * lda + k0 + 8 * g;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int s = w + i * kW;
      wf[c][i] = s < S ? *reinterpret_cast<const uint4v*>(wr + s * 32) : uint4v{0u, 0u, 0u, 0u};
    }
  }
  const int row = 16 * (w % MT) + r16, col = n0 + 16 * (w / MT) + 4 * g;  // the first NC * MT of the waves finish
  uint2v bias = {0u, 0u};
  if (OUT != OUT_PART && w < NC * MT) bias = *reinterpret_cast<const uint2v*>(bias_ + col);
  float4v acc[NC][MT];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[c][m] = float4v{0.f, 0.f, 0.f, 0.f};
  if constexpr (P > 0) {
    norm_rows<MT, K, P>(n, T, xs, ready);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int s = w + i * kW;
      if (s < S)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const uint4v x = *reinterpret_cast<const uint4v*>(xs + (16 * m + r16) * (K + 8) + s * 32 + 8 * g);
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c][m] = mfma(wf[c][i], x, acc[c][m]);
        }
    }
  } else {
    ready();
    const __amdgpu_buffer_rsrc_t ra = uniform_rsrc(A, T * lda * 2);
    uint4v af[MT][PER];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int s = w + i * kW;
        af[m][i] = load16(ra, s < S && 16 * m + r16 < T ? ((16 * m + r16) * lda + k0 + s * 32 + 8 * g) * 2 : 0x7ffffff0);  // (past it: zeros)
      }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int i = 0; i < PER; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c][m] = mfma(wf[c][i], af[m][i], acc[c][m]);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int m = 0; m < MT; ++m) red[((w * NC + c) * MT + m) * 64 + lane] = acc[c][m];
  __syncthreads();
  if (w >= NC * MT) return;
  float4v y = red[w * 64 + lane];
#pragma unroll
  for (int i = 1; i < kW; ++i) {
    const float4v z = red[(i * NC * MT + w) * 64 + lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] += z[j];
  }
  if (row >= T) return;
  if constexpr (OUT == OUT_PART) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, y), uniform_rsrc(part, T * N * 4), (row * N + col) * 4, 0, kSC1);
  } else {
    const float4v b = widen4(bias);
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = OUT == OUT_GELU ? gelu_erf(y[j] + b[j]) : y[j] + b[j];
    store8(narrow4(y), uniform_rsrc(h, T * N * 2), (row * N + col) * 2);
  }
}

LWC_HOST_DEVICE constexpr int flag_stride(int items) { return (items + 1 + 63) / 64 * 64 + 64; }

// What a layer leaves behind, bytes a row of width D: x (the layer's input) and y (behind the attention) as bf16, their heads' outputs a,
// the parts of the two sums in fp32, and h (F columns; wider than 384 also q, k and v)
template <int D, int PF>
struct Rows {
  static constexpr int kX = 0, kY = 2 * D, kA = 4 * D, kSum1 = 6 * D, kSum2 = 10 * D, kH = kSum2 + 4 * D * PF, kQkv = kH + 8 * D,
                       kBytes = kQkv + (D <= 384 ? 0 : 6 * D);
};

struct Chain {
  const bf16_t* w[12 * kLayers];
  Norm n;           // the first layer's
  const int* cu;    // [nseq + 1]
  int layers, nseq, T, last;  // last: the norm behind the layers is an item of its own
  float scale;
  uint8_t* rows;    // [layers][T * Rows::kBytes], behind that of the layer before the first
  bf16_t* out;      // [T, D]: of the last norm
  int* flags;       // [kCopies][stride]: items that are done; behind the first copy's the next item to be taken
};

template <int MT, int D, int DH>
struct Items {
  static constexpr bool kOwn = D <= 384;  // a head's projection and attention are one item
  static constexpr int F = 4 * D, H = D / DH, PF = D <= 384 || D * MT > 1536 ? 2 : 4, NC = 2;
  // items of a stage; the stages that normalise have one more, which writes the rows for the residual after them
  static constexpr int kQkv = kOwn ? 0 : 3 * D / 16 / NC + 1, kAttn = kOwn ? H + 1 : H, kO = D / 16, kUp = F / 16 / NC + 1, kDown = D / 16 * PF;
  static constexpr int kLayer = kQkv + kAttn + kO + kUp + kDown;
  static constexpr int kLn = kW * NC * MT * 1024 + 16 * MT * (D + 8) * 2;
  static constexpr int kHead = kOwn ? QkvAttnLds<MT, kOwn ? D : 384, kOwn ? DH : 32>::kBytes : Head<MT, DH>::kBytes;
  // (more than half of a compute unit's: items that share one are in each other's way)
  static constexpr int kLds = std::max(std::max(kLn, kHead), 81 * 1024);
  static_assert(kLds <= 160 * 1024 - 64, "a compute unit's LDS");
  static_assert(kQkv <= kT && kUp <= kT && kDown <= kT, "one flag a thread");
  using R = Rows<D, PF>;
};

template <int MT, int D, int DH>
__global__ void __launch_bounds__(kT) chain_kernel(Chain p) {
  using I = Items<MT, D, DH>;
  using R = typename I::R;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  __shared__ int taken;
  const int items = p.layers * I::kLayer + p.last, stride = flag_stride(items);
  if (threadIdx.x == 0) taken = __hip_atomic_fetch_add(p.flags + items, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int item = __builtin_amdgcn_readfirstlane(taken), l = item / I::kLayer, T = p.T;
  int k = item - l * I::kLayer;
  const bf16_t* const* w = p.w + 12 * l;
  const int* const layer = p.flags + (int)(__builtin_amdgcn_s_getreg(20 | 3 << 11) % kCopies) * stride + l * I::kLayer;  // (HW_REG_XCC_ID)
  uint8_t* const rows = p.rows + (size_t)l * T * R::kBytes;
  auto bf = [&](int at) { return reinterpret_cast<bf16_t*>(rows + (ptrdiff_t)T * at); };
  auto f32 = [&](int at) { return reinterpret_cast<float*>(rows + (ptrdiff_t)T * at); };
  // the norm in front of layer l, of what layer l - 1 (or begin_kernel) left; nothing to wait for where another launch did
  Norm n = p.n;
  n.part = f32(R::kSum2 - R::kBytes), n.res = bf(R::kY - R::kBytes);
  if (l > 0) n.rbias = w[9 - 12], n.g = w[10 - 12], n.b = w[11 - 12];
  auto before = [&] {
    if (l > 0) wait_for(layer - I::kDown, I::kDown, false);
  };
  constexpr int kFront = I::kQkv + I::kAttn, kWrite = (I::kOwn ? I::kAttn : I::kQkv) - 1;
  if (l == p.layers || k == kWrite) {
    n.out = l == p.layers ? p.out : bf(R::kX);
    norm_rows<MT, D, I::PF>(n, T, nullptr, before);
  } else if (k < kWrite) {
    if constexpr (I::kOwn) qkv_attn<MT, D, DH, I::PF>(n, w[0], w[1], p.cu, bf(R::kA), T, p.nseq, p.scale, k, smem, before);
    else project<MT, I::NC, D, I::PF, OUT_BIAS>(n, nullptr, w[0], w[1], nullptr, bf(R::kQkv), T, 3 * D, D, k * 16 * I::NC, 0, smem, before);
  } else if (k < kFront) {
    if constexpr (!I::kOwn)
      attention<MT, D, DH>(bf(R::kQkv), p.cu, bf(R::kA), T, p.nseq, p.scale, k - I::kQkv, smem, [&] { wait_for(layer, I::kQkv, l == 0); });
  } else if (k < kFront + I::kO) {
    project<MT, 1, D, 0, OUT_PART>(n, bf(R::kA), w[2], nullptr, f32(R::kSum1), nullptr, T, D, D, (k - kFront) * 16, 0, smem,
                                   [&] { wait_for(layer + I::kQkv, I::kAttn, I::kOwn && l == 0); });
  } else if (k < kFront + I::kO + I::kUp) {
    k -= kFront + I::kO;
    n.part = f32(R::kSum1), n.res = bf(R::kX), n.rbias = w[3], n.g = w[4], n.b = w[5];
    auto up = [&] { wait_for(layer + kFront, I::kO, false); };
    if (k == I::kUp - 1) {
      n.out = bf(R::kY);
      norm_rows<MT, D, 1>(n, T, nullptr, up);
    } else {
      project<MT, I::NC, D, 1, OUT_GELU>(n, nullptr, w[6], w[7], nullptr, bf(R::kH), T, I::F, D, k * 16 * I::NC, 0, smem, up);
    }
  } else {
    k -= kFront + I::kO + I::kUp;
    constexpr int KD = I::F / I::PF;
    const int part = k / I::kO;
    project<MT, 1, KD, 0, OUT_PART>(n, bf(R::kH), w[8], nullptr, f32(R::kSum2) + (size_t)part * T * D, nullptr, T, D, I::F, k % I::kO * 16,
                                    part * KD, smem, [&] { wait_for(layer + kFront + I::kO, I::kUp, false); });
  }
  done(p.flags + item, stride);
}

// What the first layer's norm reads, in the form that a layer leaves (part 0: the sums of the embeddings; the rest zeros), a workgroup a row; and the flags
struct Begin {
  const bf16_t* word;    // [V, D]
  const bf16_t* pos;     // [NP, D]
  const int* ids;        // [T]
  const int* positions;  // [T]
  int V, NP, T, D, parts;
  float* part;           // [parts, T, D]
  bf16_t* res;           // [T, D]
  bf16_t* rbias;         // [D]
  int* flags;
  int ints;
};

__global__ void __launch_bounds__(256) begin_kernel(Begin p) {
  const int row = blockIdx.x, at = threadIdx.x * 4;
  if (row < p.T && at < p.D) {
    const int id = min(max(p.ids[row], 0), p.V - 1), at_p = min(max(p.positions[row], 0), p.NP - 1);
    float4v x = widen4(*reinterpret_cast<const uint2v*>(p.word + (size_t)id * p.D + at));
    const float4v e = widen4(*reinterpret_cast<const uint2v*>(p.pos + (size_t)at_p * p.D + at));
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] += e[j];
    *reinterpret_cast<float4v*>(p.part + (size_t)row * p.D + at) = x;
    for (int i = 1; i < p.parts; ++i) *reinterpret_cast<float4v*>(p.part + ((size_t)i * p.T + row) * p.D + at) = float4v{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<uint2v*>(p.res + (size_t)row * p.D + at) = uint2v{0u, 0u};
    if (row == 0) *reinterpret_cast<uint2v*>(p.rbias + at) = uint2v{0u, 0u};
  }
  for (int i = blockIdx.x * 256 + threadIdx.x; i < p.ints; i += gridDim.x * 256) p.flags[i] = 0;
}

struct Call {
  const void* const* w;
  int layers;
  const int* cu;
  int nseq;
  float scale, eps;
  const bf16_t *g, *b;  // the embeddings' norm
  Begin begin;
  void *out, *scratch;
  hipStream_t s;
};

// bytes of scratch: the flags of a launch and its layers' rows
template <int MT, int D, int DH>
constexpr long long scratch_bytes(int layers, int T) {
  using I = Items<MT, D, DH>;
  const int most = std::min(layers, kLayers);
  return 4LL * kCopies * flag_stride(most * I::kLayer + 1) + (long long)(layers + 1) * T * I::R::kBytes;
}

template <int MT, int D, int DH>
int run(const Call& c) {
  using I = Items<MT, D, DH>;
  using R = typename I::R;
  static const hipError_t once = hipFuncSetAttribute((const void*)chain_kernel<MT, D, DH>, hipFuncAttributeMaxDynamicSharedMemorySize, I::kLds);
  (void)once;
  int* flags = (int*)c.scratch;
  uint8_t* rows = (uint8_t*)c.scratch + scratch_bytes<MT, D, DH>(c.layers, 0);
  auto at = [&](int place) { return rows + (size_t)c.begin.T * place; };
  Begin first = c.begin;
  first.D = D, first.parts = I::PF, first.flags = flags;
  first.part = (float*)at(R::kSum2), first.res = (bf16_t*)at(R::kY), first.rbias = (bf16_t*)at(R::kX);
  Norm n{nullptr, nullptr, first.rbias, c.g, c.b, c.eps, nullptr};
  for (int l = 0; l < c.layers; l += kLayers) {
    Chain p;
    p.layers = std::min(kLayers, c.layers - l);
    p.last = l + p.layers == c.layers;
    for (int i = 0; i < 12 * p.layers; ++i) p.w[i] = (const bf16_t*)c.w[12 * l + i];
    p.n = n;
    p.cu = c.cu;
    p.nseq = c.nseq, p.T = c.begin.T, p.scale = c.scale;
    p.rows = at(R::kBytes), p.out = (bf16_t*)c.out, p.flags = flags;
    const int items = p.layers * I::kLayer + p.last;
    first.ints = kCopies * flag_stride(items);
    first.T = l == 0 ? c.begin.T : 0;  // (later on the flags alone)
    begin_kernel<<<std::max(32, first.T), 256, 0, c.s>>>(first);
    chain_kernel<MT, D, DH><<<items, kT, I::kLds, c.s>>>(p);
    rows = at(p.layers * R::kBytes);
    auto t = [&](int i) { return (const bf16_t*)c.w[12 * (l + p.layers - 1) + i]; };
    n.rbias = t(9), n.g = t(10), n.b = t(11);
  }
  return (int)hipGetLastError();
}

}  // namespace efew
}  // namespace lwc

// Whether lwc_encoder_few takes T rows of a stack of width d, H heads and f FFN columns.
extern "C" int lwc_encoder_few_ok(int T, int d, int H, int f) {
  return T > 0 && T <= 32 && f == 4 * d && ((d == 384 && H == 12) || (d == 768 && H == 12) || (d == 1024 && H == 16));
}

// F<MT, D, DH>(args) for T rows of width d
#define LWC_FEW(F, T, d, ...)                                                                                       \
  (T <= 16 ? d == 384 ? F<1, 384, 32>(__VA_ARGS__) : d == 768 ? F<1, 768, 64>(__VA_ARGS__) : F<1, 1024, 64>(__VA_ARGS__) \
           : d == 384 ? F<2, 384, 32>(__VA_ARGS__) : d == 768 ? F<2, 768, 64>(__VA_ARGS__) : F<2, 1024, 64>(__VA_ARGS__))

// bytes of lwc_encoder_few's scratch, for sizes that it takes
extern "C" long long lwc_encoder_few_scratch(int layers, int T, int d) {
  using namespace lwc::efew;
  return LWC_FEW(scratch_bytes, T, d, layers, T);
}

// x [T, d] = the last hidden rows of `layers` layers over word[ids] + pos[positions].  w: 12 pointers a layer (qkv, its bias, o,
// its bias, norm 1 gain and bias, FFN up and bias, FFN down and bias, norm 2 gain and bias), all contiguous and 16-byte aligned,
// and so is scratch [lwc_encoder_few_scratch].
extern "C" int lwc_encoder_few(const void* word, const void* pos, const int* ids, const int* positions, int V, int P, const void* g,
                               const void* b, float eps, const void* const* w, int layers, const int* cu, int nseq, int T, int d,
                               int H, int f, float scale, void* x, void* scratch, hipStream_t s) {
  using namespace lwc::efew;
  using lwc::bf16_t;
  if (!lwc_encoder_few_ok(T, d, H, f) || nseq < 1 || nseq > 63) return -1;
  Call c{};
  c.w = w, c.layers = layers, c.cu = cu, c.nseq = nseq, c.scale = scale, c.eps = eps, c.g = (const bf16_t*)g, c.b = (const bf16_t*)b;
  c.begin.word = (const bf16_t*)word, c.begin.pos = (const bf16_t*)pos, c.begin.ids = ids, c.begin.positions = positions;
  c.begin.V = V, c.begin.NP = P, c.begin.T = T;
  c.out = x, c.scratch = scratch, c.s = s;
  return LWC_FEW(run, T, d, c);
}
