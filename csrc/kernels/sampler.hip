// K8a+K8b+K8c+K8d fused: logits processing, raw log-softmax + top-k logprobs, and top-k / top-p /
// min-p / top-a filtered multinomial sampling (or greedy argmax) in ONE pass over each logits row.
//
// Bound by the row a compute unit holds: its load takes 11 us at the CU's share of the memory rate, its passes 8 us and more
// (a round of exps 6, of masses 2).  Large batches of large vocabularies hold two rows per CU, 512 threads each with 23 of 32
// slots in registers and 9 in LDS, so that the two overlap; thresholds are searched in a list of the elements that can
// matter where those are few, and a draw that carries 1 - top_p by itself is accepted without a pass.  4096 rows, one MI355X, us,
// before -> after these: vocabulary 128256 greedy 216 -> 224, temperature 0.8 264 -> 242, with top-p 0.95 356 -> 285, with top-k 40
// and top-p 0.9 814 -> 405, with top-p 0.95 and 20 logprobs 598 -> 411; vocabulary 32000 top-p 0.95 110 -> 99, top-k 40 199 -> 157, with
// 20 logprobs 254 -> 188, with a bias and a mask 189 -> 138.  What two rows per unit cost: greedy rows a power of two of bytes apart
// (131072 tokens) 213 -> 242.
//
// One workgroup per row, of 1024 threads or of 512 that stand for two each.  The row (bf16, V <= 8*1024*SLOTS) is
// loaded ONCE from HBM as packed bf16 (16 B per load, SLOTS loads per thread) and every later phase — raw max and
// log-sum-exp, the top-K selection for `top_logprobs`, penalties/bias/grammar mask, the filter
// thresholds and the inverse-CDF draw — works on those registers plus block reductions.
// Element index of (thread t, slot j, lane-element e) = (j*1024 + t)*8 + e.
//
// Thresholds are found by exact binary search over the 16-bit order-preserving key of the bf16 value
// (over a list of the candidates, else 14 block-reduction rounds over the row), so top-p / top-k are exact (ties at the
// threshold are kept, as in the usual "keep >= threshold" convention).  Randomness: Philox4x32-10 keyed by the per-sequence seed,
// counter = per-sequence step — reproducible per (seed, step) independent of batch composition.
//
// Reference fields served: temperature/top_p/min_p/top_a/top_k/frequency_penalty/presence_penalty/
// repetition_penalty/logit_bias (src/score/llm/mod.rs:39-72, validation :376-406,:490-508),
// top_logprobs <= 20 (:455-467) feeding the vote extractor (src/score/completions/client.rs:1721-1793),
// and constrained output modes (json_schema / tool_call, src/score/llm/mod.rs:690-696).
#include "common.h"

namespace lwc {

constexpr int kSampT = 1024;
constexpr int kMaxTopK = 20;
constexpr int kCollect = 64;
constexpr int kRegSlots = 23;  // of the 32 slots of the 512-thread build

struct SampleParams {
  const bf16_t* logits;  // [B, ld]
  int ld, V;
  int nt;                    // rows of more than 131072 tokens: the logits are loaded past the caches
  const float* temperature;  // [B]  (<= 0 -> greedy)
  const float* top_p;        // [B]  (>= 1 -> off)
  const int* top_k;          // [B]  (<= 0 -> off)
  const float* min_p;        // [B]  (<= 0 -> off)
  const float* top_a;        // [B]  (<= 0 -> off)
  const float* freq_pen;     // [B] or null
  const float* pres_pen;     // [B] or null
  const float* rep_pen;      // [B] or null
  uint16_t* counts;          // [B, V] generated-token counts (or null); updated with the sample
  const int* count_rows;     // [B] row of `counts` for each batch row (or null = identity)
  const float* bias;         // [NBT, V] dense logit bias rows (or null)
  const int* bias_rows;      // [B] row of `bias` (-1 = none)
  const uint32_t* mask;      // [NMT, V/32] allowed-token bitmasks (or null)
  const int* mask_rows;      // [B] row of `mask` (-1 = none)
  const unsigned long long* seeds;    // [B]
  const unsigned long long* offsets;  // [B] (step counter)
  int num_logprobs;          // K for top logprobs (0..20)
  int mask_logprobs;         // 1: rows with a grammar mask report logprobs over the MASKED distribution
                             //    (the restricted softmax over the allowed tokens — the vote fast path)
  int need_logprob;          // 0: no caller reads out_logprob (and K == 0): the raw log-sum-exp is not
                             //    computed and out_logprob is NaN
  int* out_token;            // [B]
  float* out_logprob;        // [B]  raw logprob of the sampled token
  int* out_topk_ids;         // [B, K]
  float* out_topk_lp;        // [B, K]
};

// ---- Philox4x32-10 ----
LWC_DEVICE void philox4x32(uint32_t (&ctr)[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    const uint32_t lo0 = 0xD2511F53u * ctr[0], hi0 = __umulhi(0xD2511F53u, ctr[0]);
    const uint32_t lo1 = 0xCD9E8D57u * ctr[2], hi1 = __umulhi(0xCD9E8D57u, ctr[2]);
    const uint32_t n0 = hi1 ^ ctr[1] ^ k0, n2 = hi0 ^ ctr[3] ^ k1;
    ctr[0] = n0;
    ctr[1] = lo1;
    ctr[2] = n2;
    ctr[3] = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

LWC_DEVICE uint32_t f2key(float f) {  // order-preserving 16-bit key of the bf16-rounded value
  const uint32_t b = __float_as_uint(f) >> 16;
  return (b & 0x8000u) ? (~b & 0xffffu) : (b | 0x8000u);
}
LWC_DEVICE float key2f(uint32_t k) {
  const uint32_t b = (k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu);
  return __uint_as_float(b << 16);
}

// (Passes under a condition have it in front of the condition: inside, the two paths' rows are two values and meet in
// copies of the whole row, spilled.)
// Keep the packed row opaque at the top of every pass: otherwise LICM hoists the 8*SLOTS unpacked
// floats (or their keys) out of the binary-search loops and the kernel spills (1024 threads leave
// 128 VGPRs per lane; the packed row alone is 4*SLOTS of them).
#define OPAQUE_ROW(row)                                \
  _Pragma("unroll") for (int _j = 0; _j < RS; ++_j) { \
    asm volatile("" : "+v"(row[_j]));                  \
  }                                                    \
  if constexpr (LS > 0) asm volatile("" ::: "memory")  /* nor keep what an earlier pass read from LDS */

// The thread's slot s (compile-time s): the first RS in registers, the others in its own cells of LDS
#define SLOT(s) ((s) < RS ? row[(s) < RS ? (s) : 0] : held[((s) < RS ? 0 : (s)-RS) * T + t])
#define SET_SLOT(s, x)                                  \
  do {                                                  \
    if ((s) < RS) row[(s) < RS ? (s) : 0] = (x);        \
    else held[((s) < RS ? 0 : (s)-RS) * T + t] = (x);   \
  } while (0)
// one slot's values live at a time, LDS slots read when their turn comes
#define NEXT_SLOT()                                       \
  do {                                                    \
    __builtin_amdgcn_sched_barrier(0);                    \
    if constexpr (LS > 0) asm volatile("" ::: "memory");  \
  } while (0)
// value of element e (0..7) of a slot (compile-time e)
#define GET(x, e) (((e)&1) ? __uint_as_float((x)[(e) >> 1] & 0xffff0000u) : __uint_as_float((x)[(e) >> 1] << 16))

// fp16 helpers for the probability form of the row (u in [0,1] as packed fp16)
LWC_DEVICE uint16_t h2bits(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }
#define KEYU(x, e) ((((e)&1) ? ((x)[(e) >> 1] >> 16) : ((x)[(e) >> 1] & 0xffffu)))
#define GETU(x, e) ((float)__builtin_bit_cast(_Float16, (uint16_t)KEYU(x, e)))

// Packed selection over the probability form (two non-negative fp16 u per register: their bit patterns
// order like the values).  Per pair: a saturating 16-bit subtract against (threshold - 1) is >= 1 exactly
// where key >= threshold, min(., 1) makes that a 0/1 mask, and either a packed add counts it or a packed
// multiply by 0x3C00 turns it into fp16 0 / 1.0 for a v_dot2 that sums the kept u in fp32 — 2 VALU per
// element instead of unpack + compare + select + add (+ the SDWA hazard nops) per element.
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
LWC_DEVICE half2v as_h2(uint32_t w) { return __builtin_bit_cast(half2v, w); }
LWC_DEVICE void count2(uint32_t& c2, uint32_t w0, uint32_t w1, uint32_t thr1x2, uint32_t one2) {
  uint32_t t0, t1;
  asm("v_pk_sub_u16 %1, %3, %5 clamp\n\t"
      "v_pk_sub_u16 %2, %4, %5 clamp\n\t"
      "v_pk_min_u16 %1, %1, %6\n\t"
      "v_pk_min_u16 %2, %2, %6\n\t"
      "v_pk_add_u16 %0, %0, %1\n\t"
      "v_pk_add_u16 %0, %0, %2"
      : "+v"(c2), "=&v"(t0), "=&v"(t1)
      : "v"(w0), "v"(w1), "v"(thr1x2), "v"(one2));
}
// Two registers (four u) per block, the whole chain in one asm block: the compiler puts a hazard nop
// after every inline-asm result a compiled instruction reads, so the dot stays inside.  Ordering keeps
// each v_dot2c >= 1 instruction after the multiply that feeds it (VALU write -> DOT read) and the dots
// back to back on one accumulator (same-DOT srcC forwarding, no wait); the accumulator's final reader
// waits through dot_read().
LWC_DEVICE void mass2(float& acc, uint32_t w0, uint32_t w1, uint32_t thr1x2, uint32_t one2, uint32_t h1x2) {
  uint32_t t0, t1;
  asm("v_pk_sub_u16 %1, %3, %5 clamp\n\t"
      "v_pk_sub_u16 %2, %4, %5 clamp\n\t"
      "v_pk_min_u16 %1, %1, %6\n\t"
      "v_pk_min_u16 %2, %2, %6\n\t"
      "v_pk_mul_lo_u16 %1, %1, %7\n\t"
      "v_pk_mul_lo_u16 %2, %2, %7\n\t"
      "v_dot2c_f32_f16 %0, %3, %1\n\t"
      "v_dot2c_f32_f16 %0, %4, %2"
      : "+v"(acc), "=&v"(t0), "=&v"(t1)
      : "v"(w0), "v"(w1), "v"(thr1x2), "v"(one2), "v"(h1x2));
}
// DOT write -> VALU read needs 3 wait states
LWC_DEVICE float dot_read(float acc) {
  float r;
  asm("s_nop 2\n\tv_mov_b32 %0, %1" : "=v"(r) : "v"(acc));
  return r;
}
LWC_DEVICE uint32_t thr1x2(uint32_t key) { return ((key - 1u) & 0xffffu) * 0x10001u; }  // key >= 1

// ---- reductions by lane swaps and DPP (a shuffle is a trip through LDS, six of them per reduction) ----
#define LWC_DPP(x, ctrl) __builtin_amdgcn_mov_dpp((x), (ctrl), 0xF, 0xF, false)
LWC_DEVICE int row16_sum_i(int x) {
  x += LWC_DPP(x, 0xB1);
  x += LWC_DPP(x, 0x4E);
  x += LWC_DPP(x, 0x141);
  return x + LWC_DPP(x, 0x140);
}
LWC_DEVICE int row_sum4_i(int v) {
  auto r = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
  v = (int)(r[0] + r[1]);
  auto q = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
  return (int)(q[0] + q[1]);
}
// inclusive sum over the wave's lanes: within rows of 16, then row 0 into 1 and 2 into 3, then the lower half into the upper
LWC_DEVICE float wave_scan(float x) {
#define LWC_SCAN(ctrl, rows) \
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, rows, 0xF, false))
  LWC_SCAN(0x111, 0xF);
  LWC_SCAN(0x112, 0xF);
  LWC_SCAN(0x114, 0xF);
  LWC_SCAN(0x118, 0xF);
  LWC_SCAN(0x142, 0xA);
  LWC_SCAN(0x143, 0xC);
#undef LWC_SCAN
  return x;
}

// Block-wide reductions over two alternating sets of partials: one barrier each (a set is written again only behind the
// next reduction's barrier, which every reader of it has passed).  The partials are those of the 16 waves of 1024 threads:
// a thread that stands for two of them brings two values, so that a sum's order does not depend on the workgroup's size
template <int VT>
struct Red {
  static constexpr int kW = kSampT / 64 / VT;  // waves
  float* f;  // [2][32]
  int ph;
  LWC_DEVICE float* set() { return f + 32 * (ph++ & 1); }
  LWC_DEVICE float sum(const float (&x)[VT]) {
    float* sc = set();
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      const float w = row_sum4(row16_sum(x[v]));
      if ((threadIdx.x & 63) == 0) sc[(threadIdx.x >> 6) + v * kW] = w;
    }
    __syncthreads();
    return row16_sum(sc[threadIdx.x & 15]);
  }
  // (and the block's sum of c)
  LWC_DEVICE float sum(const float (&x)[VT], int c, int& count) {
    float* sc = set();
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      const float w = row_sum4(row16_sum(x[v]));
      if ((threadIdx.x & 63) == 0) sc[(threadIdx.x >> 6) + v * kW] = w;
    }
    c = row_sum4_i(row16_sum_i(c));
    if ((threadIdx.x & 63) == 0) reinterpret_cast<int*>(sc)[16 + (threadIdx.x >> 6)] = c;
    __syncthreads();
    count = row16_sum_i((threadIdx.x & 15) < kW ? reinterpret_cast<int*>(sc)[16 + (threadIdx.x & (kW - 1))] : 0);
    return row16_sum(sc[threadIdx.x & 15]);
  }
  LWC_DEVICE float max(float v) {
    float* sc = set();
    v = row_max4(row16_max(v));
    if ((threadIdx.x & 63) == 0) sc[threadIdx.x >> 6] = v;
    __syncthreads();
    return row16_max(sc[threadIdx.x & (kW - 1)]);
  }
  LWC_DEVICE int sum_i(int v) {
    int* sc = reinterpret_cast<int*>(set());
    v = row_sum4_i(row16_sum_i(v));
    if ((threadIdx.x & 63) == 0) sc[threadIdx.x >> 6] = v;
    __syncthreads();
    return row16_sum_i((threadIdx.x & 15) < kW ? sc[threadIdx.x & (kW - 1)] : 0);
  }
  // hi * 4096 + lo of the block, exact: |hi| < 2^21, 0 <= lo < 2^21 each
  LWC_DEVICE double sum_wide(int hi, int lo) {
    int* sc = reinterpret_cast<int*>(set());
    hi = row_sum4_i(row16_sum_i(hi));
    lo = row_sum4_i(row16_sum_i(lo));
    if ((threadIdx.x & 63) == 0) {
      sc[threadIdx.x >> 6] = hi;
      sc[16 + (threadIdx.x >> 6)] = lo;
    }
    __syncthreads();
    const bool on = (threadIdx.x & 15) < kW;
    return (double)row16_sum_i(on ? sc[threadIdx.x & (kW - 1)] : 0) * 4096.0 + (double)row16_sum_i(on ? sc[16 + (threadIdx.x & (kW - 1))] : 0);
  }
};
static_assert(kSampT == 1024, "the reductions meet over 16 waves");

// Lowest index among the thread's elements for which TEST(x, e) holds, 0x7fffffff if none.  Slot and element are kept
// apart: both are inline constants, while an index per element would be 8 * SLOTS literals, each in a register of its own
// ahead of the loop (100 spilled registers in the SLOTS = 16 build).
#define LOWEST_INDEX(TEST, OUT)                                                  \
  do {                                                                           \
    OUT = 0x7fffffff;                                                            \
    _Pragma("unroll") for (int v = 0; v < VT; ++v) {                             \
      int _bj = -1, _be = 0;                                                     \
      _Pragma("unroll") for (int j = SLOTS - 1; j >= 0; --j) {                   \
        const uint4v x = SLOT(v * SLOTS + j);                                    \
        int _e = 8;                                                              \
        _Pragma("unroll") for (int e = 7; e >= 0; --e) _e = (TEST) ? e : _e;     \
        _bj = _e < 8 ? j : _bj;                                                  \
        _be = _e < 8 ? _e : _be;                                                 \
        NEXT_SLOT();                                                             \
      }                                                                          \
      OUT = min(OUT, _bj >= 0 ? (_bj * kSampT + v * T + t) * 8 + _be : 0x7fffffff); \
    }                                                                            \
  } while (0)

// One wave: the largest key in [lo, hi] that at least K of the 1024 keys reach (lo if no larger one does)
LWC_DEVICE uint32_t kth_of_1024(const uint32_t* keys, int lane, int K, uint32_t lo, uint32_t hi) {
  uint32_t tk[kSampT / 64];
#pragma unroll
  for (int i = 0; i < kSampT / 64; ++i) tk[i] = keys[i * 64 + lane];
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    int c = 0;
#pragma unroll
    for (int i = 0; i < kSampT / 64; ++i) c += __popcll(__builtin_amdgcn_ballot_w64(tk[i] >= mid));
    if (c >= K)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// A row's scalar as what it is, the same in every lane: loaded plainly the compiler takes it for a lane's own, both sides of
// a branch on it are run one after the other, and the row stays live, in copies, through the side that does not need it
LWC_DEVICE float uniform_f(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }

// PROC: a bias, a mask or penalties may apply to the rows; TOPK: num_logprobs > 0.  Builds of their own, so that a step
// that asks for neither carries neither's registers.
// T threads: 1024, or 512 of which each stands for two of the 1024 (element order, sums and draws are those of 1024: slot
// v * SLOTS + j of thread t is slot j of thread v * T + t).  RS of the VT * SLOTS slots are in registers, the rest in LDS.
// Waves per SIMD: two workgroups of the shortest rows; with 5 for 8 slots the next row's workgroup comes in beside the last waves of
// the one before it (the wave that ranks the logprobs: 4096 rows of 65536 tokens, 5 logprobs, 256 -> 241 us).
template <int T, int SLOTS, int RS, bool PROC, bool TOPK>
__global__ void __launch_bounds__(T, SLOTS <= 4 ? (PROC && TOPK ? 7 : 8) : SLOTS == 8 ? 5 : 4) sample_kernel(SampleParams p) {
  constexpr int VT = kSampT / T, NS = SLOTS * VT, LS = NS - RS;
  static_assert(!PROC || VT == 1, "processed rows are held by 1024 threads");
  __shared__ uint4v held[LS > 0 ? LS * T : 1];
  __shared__ float sred[2 * 32];
  __shared__ int sredi[32];
  __shared__ int s_owner;
  __shared__ float s_cval[kCollect];
  __shared__ int s_cidx[kCollect];
  __shared__ int s_ccount;
  // Two workgroups per compute unit: a threshold search over a list is one wave's, the other row has the unit meanwhile.
  // One: every thread's (64 rows, top-p 0.95, 50 us by one wave, 35 by all; 4096 rows of 32000 in pairs 83 by one, 92 by all)
  constexpr bool kPairs = LS > 0 || SLOTS <= 4;
  constexpr int kList = LS > 0 ? 3456 : kPairs ? 2048 : 8192;  // 16-bit keys in LDS, which the pairs share
  // Masses are searched in lists of as many keys in every build of a vocabulary: a round over the row decides by fp32 sums, a list
  // by exact ones, and a row's draw must not depend on how many rows there are (counts are whole numbers either way)
  // (4 slots: a list is one wave's, and a round over so short a row 1 us: 64 rows of 32000 tokens, top-p 0.5, 29 us by rounds, 35 in
  // lists of up to 2048)
  constexpr int kMassList = SLOTS == 16 ? 3456 : SLOTS <= 4 ? 512 : kList;
  constexpr int kFewest = LS > 0 ? 40 * SLOTS : 24 * SLOTS + (SLOTS <= 8 ? 32 : 0);  // a top-k up to which the list of the largest pays
  static_assert(kFewest <= kSampT, "one of the threads' maxima each");
  __shared__ uint32_t s_tkey[kList / 2];
  uint16_t* const s_list = reinterpret_cast<uint16_t*>(s_tkey);
  static_assert(kList >= 2 * kSampT && kMassList <= kList, "s_tkey holds the maxima of 1024 threads too");
  __shared__ uint32_t s_lb, s_fkey;
  __shared__ uint32_t s_own[SLOTS * 4];
  __shared__ float s_oexcl;
  __shared__ int s_found;

  const int b = blockIdx.x;
  const int t = threadIdx.x;
  Red<VT> red{sred, 0};
  const bf16_t* lrow = p.logits + (size_t)b * p.ld;
  const int nvec = p.V >> 3;

  // ---- load the raw row once ----
  // (With the nt bit where the logits are many: read once, they neither stay in the last-level cache nor push out what it holds.  All
  // rows of pairs, us without / with it: 4096 rows of 128256 greedy 215 / 177, top-p 0.95 318 / 307, top-k 40 359 / 344, 1500 greedy 85 / 69,
  // 1024 47 / 48, with the logits written just before 58 / 43; longer rows from 128 MiB of logits on: 4096 of 151936 greedy 286 / 241,
  // 1000 73 / 68, written just before 79 / 59, 64 11.2 / 12.4.  Shorter rows level within 5 % either way, so not there.  Rows of pairs that the
  // last-level cache holds whole, read and written again there just before, lose: 1024 of 102400 greedy 42.4 / 44.5, top-k 40 102 / 105; written
  // by the product with the head 54.5 / 47.6 and 107 / 103.)
  uint4v row[RS];
  const uint32_t* lmask =
      (PROC && p.mask_logprobs && p.mask && p.mask_rows[b] >= 0) ? p.mask + (size_t)p.mask_rows[b] * (p.V >> 5) : nullptr;
  if constexpr (VT == 1) {
    const uint4v none = uint4v{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
    if (SLOTS > 16 && !PROC && p.nt) {
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        const int vi = j * kSampT + t;
        row[j] = vi < nvec ? __builtin_nontemporal_load(reinterpret_cast<const uint4v*>(lrow + (size_t)vi * 8)) : none;
      }
    } else {
#pragma unroll
      for (int j = 0; j < SLOTS; ++j) {
        const int vi = j * kSampT + t;
        row[j] = vi < nvec ? *reinterpret_cast<const uint4v*>(lrow + (size_t)vi * 8) : none;
      }
    }
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      const int vi = j * kSampT + t;
      if (lmask && vi < nvec) {  // constrained logprobs: disallowed tokens are -inf from the start
        const uint32_t bits = (lmask[vi >> 2] >> ((vi & 3) * 8)) & 0xffu;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t lo = (bits >> (2 * c)) & 1u ? (row[j][c] & 0xffffu) : 0xff80u;
          const uint32_t hi = (bits >> (2 * c + 1)) & 1u ? (row[j][c] >> 16) : 0xff80u;
          row[j][c] = lo | (hi << 16);
        }
      }
    }
  } else {
    // the LDS slots by LDS-DMA first, then the registers'; vectors past the row's end read nothing (and become -inf below)
    // (a resource per slot: one lane offset serves all of them)
    const int w0 = __builtin_amdgcn_readfirstlane(t >> 6) * 64;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if (i == LS) {  // (the wait below counts on it: the loads to LDS are the older ones)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      const int s = i < LS ? RS + i : i - LS, v0 = s % SLOTS * kSampT + s / SLOTS * T;
      const __amdgpu_buffer_rsrc_t r = uniform_rsrc(lrow + v0 * 8, max(0, nvec - v0) * 16);
      if (i < LS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(held + i * T + w0), 16, t * 16, 0, 0, kNT);
      else
        row[i < LS ? 0 : s] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(r, t * 16, 0, kNT));
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(RS) : "memory");
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int v0 = s % SLOTS * kSampT + s / SLOTS * T;
      if (v0 + T > nvec && v0 + t >= nvec) SET_SLOT(s, (uint4v{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u}));
    }
  }
  // ---- raw max (+ each thread's own max key: the top-K search bound) and log-sum-exp ----
  float mxv[VT];
OPAQUE_ROW(row);
#pragma unroll
  for (int v = 0; v < VT; ++v) {
    mxv[v] = -INFINITY;
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      const uint4v x = SLOT(v * SLOTS + j);
#pragma unroll
      for (int e = 0; e < 8; ++e) mxv[v] = fmaxf(mxv[v], GET(x, e));
      NEXT_SLOT();  // one slot's values live at a time
    }
  }
  const float mx = VT == 1 ? mxv[0] : fmaxf(mxv[0], mxv[VT - 1]);
  const float raw_max = red.max(mx);
  const int lane = t & 63, wid = t >> 6;
  const int K = TOPK ? p.num_logprobs : 0;
  // The raw log-sum-exp (the denominator of every reported logprob) is only computed when some output
  // needs it.  A processed row's exp sum rides along in the pass that processes it; every other row pays a
  // pass of its own, sampled ones too: formed in the sampling pass it doubles that pass's live values, and
  // the row spills.
  const bool need_lse = p.need_logprob || K > 0;
  float se[VT] = {};

  // ---- raw top-K (for top_logprobs): candidates collected here, ranked and written once the
  // log-sum-exp is known ----
  if constexpr (TOPK) {
    // Bound first: the K largest per-thread maxima are K distinct elements, so the K-th largest element
    // of the row is >= the K-th largest thread max (lb).  One wave finds lb over the 1024 thread maxima
    // (no block barriers inside the search); the elements >= lb — rarely more than a few dozen — are
    // then collected in one pass.  Only if they overflow the collection buffer does the exact 16-round
    // search over the whole row run (starting from lb).  Masked (-inf, key 0x7f) entries are never
    // candidates: a row with < K finite values returns fewer (rest: id -1).
    if (t == 0) s_ccount = 0;
#pragma unroll
    for (int v = 0; v < VT; ++v) s_tkey[v * T + t] = f2key(mxv[v]);
    __syncthreads();
    if (t < 64) {
      const uint32_t lb = kth_of_1024(s_tkey, lane, K, 0x80u, 0xffffu);
      if (t == 0) s_lb = lb;
    }
    __syncthreads();
    uint32_t lo = s_lb;
#pragma unroll 1
    for (int attempt = 0; attempt < 2; ++attempt) {
      if (attempt == 1) {  // overflow: exact search for the K-th largest key, then collect again
        uint32_t hi = 0xffffu;
        while (lo < hi) {
          const uint32_t mid = (lo + hi + 1) >> 1;
          int c = 0;
OPAQUE_ROW(row);
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const uint4v x = SLOT(s);
#pragma unroll
            for (int e = 0; e < 8; ++e) c += f2key(GET(x, e)) >= mid;
            NEXT_SLOT();  // one slot's values live at a time
          }
          if (red.sum_i(c) >= K)
            lo = mid;
          else
            hi = mid - 1;
        }
        __syncthreads();
        if (t == 0) s_ccount = 0;
        __syncthreads();
      }
      // candidates are sparse (a few dozen of 128k): one compare of a slot's largest value and a wave-uniform
      // branch on its ballot; only a slot where some lane of the wave hits looks at its elements one by one, and only
      // an element position that hits runs the exact key test and the LDS append (key2f(lo) is the smallest value with key >= lo, so the float test
      // passes a superset: -0 next to +0)
      const float thr = key2f(lo);
OPAQUE_ROW(row);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4v x = SLOT(s);
        float top = GET(x, 0);
#pragma unroll
        for (int e = 1; e < 8; ++e) top = fmaxf(top, GET(x, e));
        if (__builtin_amdgcn_ballot_w64(top >= thr)) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = GET(x, e);
            if (v >= thr && f2key(v) >= lo) {  // padding past V holds -inf (key 0x7f < lo): never collected
              const int slot = atomicAdd(&s_ccount, 1);
              if (slot < kCollect) {
                s_cval[slot] = v;
                s_cidx[slot] = (s % SLOTS * kSampT + s / SLOTS * T + t) * 8 + e;
              }
            }
          }
        }
        NEXT_SLOT();
      }
      __syncthreads();
      if (s_ccount <= kCollect) break;  // block-uniform
    }
  }

  // ---- processed values y = raw + bias - penalties (masked -> -inf), stored back as bf16 ----
  const float* brow = (PROC && p.bias && p.bias_rows[b] >= 0) ? p.bias + (size_t)p.bias_rows[b] * p.V : nullptr;
  const uint32_t* mrow = (PROC && p.mask && p.mask_rows[b] >= 0) ? p.mask + (size_t)p.mask_rows[b] * (p.V >> 5) : nullptr;
  const int crow_i = PROC && p.counts ? (p.count_rows ? p.count_rows[b] : b) : -1;
  const uint16_t* crow = crow_i >= 0 ? p.counts + (size_t)crow_i * p.V : nullptr;
  const float fpen = PROC && p.freq_pen ? p.freq_pen[b] : 0.f, ppen = PROC && p.pres_pen ? p.pres_pen[b] : 0.f;
  const float rpen = PROC && p.rep_pen ? p.rep_pen[b] : 1.f;
  const bool use_pen = crow && (fpen != 0.f || ppen != 0.f || rpen != 1.f);
  const bool processed = brow || mrow || use_pen;
  if (processed) {
OPAQUE_ROW(row);
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
      const int vi = j * kSampT + t;
      if (vi >= nvec) continue;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = GET(row[j], e);
      if (need_lse) {
#pragma unroll
        for (int e = 0; e < 8; ++e) se[0] += __expf(y[e] - raw_max);
      }
      if (brow) {
        const float4 b0 = reinterpret_cast<const float4*>(brow + (size_t)vi * 8)[0];
        const float4 b1 = reinterpret_cast<const float4*>(brow + (size_t)vi * 8)[1];
        y[0] += b0.x; y[1] += b0.y; y[2] += b0.z; y[3] += b0.w;
        y[4] += b1.x; y[5] += b1.y; y[6] += b1.z; y[7] += b1.w;
      }
      if (use_pen) {
        const uint4v c4 = *reinterpret_cast<const uint4v*>(crow + (size_t)vi * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t c = (c4[e >> 1] >> ((e & 1) * 16)) & 0xffffu;
          if (c) {
            y[e] = y[e] > 0.f ? y[e] / rpen : y[e] * rpen;
            y[e] -= fpen * (float)c + ppen;
          }
        }
      }
      if (mrow) {
        const uint32_t m = (mrow[vi >> 2] >> ((vi & 3) * 8)) & 0xffu;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (!((m >> e) & 1u)) y[e] = -INFINITY;
      }
      row[j] = pack8(y);
    }
  }

  const float temp = uniform_f(p.temperature[b]);
  int token = 0;
  float raw_lse = __builtin_nanf("");
OPAQUE_ROW(row);
  if (need_lse && !processed) {  // (in the passes below it would double their live values: spills)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint4v x = SLOT(s);
#pragma unroll
      for (int e = 0; e < 8; ++e) se[s / SLOTS] += __expf(GET(x, e) - raw_max);
      NEXT_SLOT();
    }
  }
  if (temp <= 0.f) {
    if (need_lse) raw_lse = raw_max + __logf(red.sum(se));
    // ---- greedy: argmax (lowest index on ties).  The row maximum is known (the raw max; a processed row
    // takes one max pass), so the argmax is the lowest index holding it — instead of a value-and-index
    // compare chain with a branch per element.  (Padding past V holds -inf: it can only match
    // a row that is -inf everywhere, whose answer, index 0, is found first.)
    float gm = raw_max;
    if (processed) {
      float ym = -INFINITY;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4v x = SLOT(s);
#pragma unroll
        for (int e = 0; e < 8; ++e) ym = fmaxf(ym, GET(x, e));
        NEXT_SLOT();  // one slot's values live at a time
      }
      gm = red.max(ym);
    }
    // the thread's elements visited from its highest index down, the last match wins: its lowest index,
    // one compare + one select per element, no branch
    int cand;
    if constexpr (PROC) { OPAQUE_ROW(row); }
    NEXT_SLOT();
    LOWEST_INDEX(GET(x, e) == gm, cand);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
    __syncthreads();
    if ((t & 63) == 0) sredi[t >> 6] = cand;
    __syncthreads();
    cand = (t & 63) < T / 64 ? sredi[t & 63] : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
    token = cand == 0x7fffffff ? 0 : cand;
  } else {
    const float invT = 1.f / temp;
    float ymax = raw_max;  // unprocessed row: the processed max IS the raw max (no extra pass)
OPAQUE_ROW(row);
    if (processed) {
      float ym = -INFINITY;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4v x = SLOT(s);
#pragma unroll
        for (int e = 0; e < 8; ++e) ym = fmaxf(ym, GET(x, e));
        NEXT_SLOT();  // one slot's values live at a time
      }
      ymax = red.max(ym);
      mxv[0] = ym;
    }
    if (!(ymax > -INFINITY)) ymax = 0.f;  // every token masked: all u = 0 (the argmax fallback below)
    const uint32_t kOne2 = 0x00010001u, kH1 = 0x3C003C00u;
    // ---- one exp per element: the row becomes u_i = exp((y_i - ymax)/T) in [0, 1] as packed fp16.
    // Non-negative fp16 bit patterns are order-preserving, so every later threshold search compares
    // raw 16-bit keys and sums fp16 values: no transcendental inside the searches.  The same pass
    // sums this thread's share of Z (over the ROUNDED values, as every later mass is).
    float zloc[VT] = {};
    // u = 2^(y * c1 + c0), c1 = log2(e) / T, c0 ~ -ymax * c1 rounded so that the exponent of y = ymax is
    // >= 0: with v_cvt_pkrtz (round toward zero) the max element is exactly 1.0 (0x3C00) and every other
    // element (at least one bf16 ulp below it, far above the fp32 rounding of c0) below 1; y = -inf gives
    // exactly 0.  One fma + one exp per element, two values per pack, their (rounded) sum by one v_dot2
    // against (1, 1)
    const float c1 = invT * 1.4426950408889634f;
    float c0 = -ymax * c1;
    if (__builtin_fmaf(ymax, c1, c0) < 0.f)  // one ulp toward +inf (c0 != 0 here)
      c0 = __uint_as_float(__float_as_uint(c0) + (c0 > 0.f ? 1u : 0xffffffffu));
    const half2v ones2 = {(_Float16)1.f, (_Float16)1.f};
OPAQUE_ROW(row);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      uint4v x = SLOT(s);
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = __builtin_fmaf(GET(x, e), c1, c0);
      if constexpr (LS > 0) __builtin_amdgcn_sched_barrier(0);  // (8 exps in a row: two waves per SIMD wait for each other's)
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = __builtin_amdgcn_exp2f(y[e]);
      if constexpr (LS > 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(y[2 * c], y[2 * c + 1]));
        zloc[s / SLOTS] = __builtin_amdgcn_fdot2(as_h2(w), ones2, zloc[s / SLOTS], false);
        x[c] = w;
      }
      if constexpr (LS > 0) asm volatile("" : "+v"(zloc[s / SLOTS]));  // (else the sums wait for the end, with every slot live)
      SET_SLOT(s, x);
      NEXT_SLOT();
    }
    // Z: from the scan of the first draw where that runs over every element and nothing needs it earlier (no top-k,
    // no top-a: the usual case), else a reduction of its own
    const int k = __builtin_amdgcn_readfirstlane(p.top_k[b]);
    const float mp = uniform_f(p.min_p[b]), ta = uniform_f(p.top_a[b]);
    const bool z_from_scan = k <= 0 && !(ta > 0.f) && !(mp > 0.f);
    float Z = 0.f;
    if (need_lse) raw_lse = raw_max + __logf(red.sum(se));
    if (!z_from_scan) Z = red.sum(zloc);
    // mass of the elements with key >= KEY (macro, not a lambda: a by-reference capture of `row`
    // makes it addressable and sends it to scratch)
#define MASS_LOCAL(KEY, OUT)                                                           \
  do {                                                                                 \
    OPAQUE_ROW(row);                                                                   \
    const uint32_t _t2 = thr1x2(KEY);                                                  \
    _Pragma("unroll") for (int v = 0; v < VT; ++v) {                                   \
      float _s = 0.f;                                                                  \
      _Pragma("unroll") for (int j = 0; j < SLOTS; ++j) {                              \
        const uint4v x = SLOT(v * SLOTS + j);                                          \
        mass2(_s, x[0], x[1], _t2, kOne2, kH1);                                        \
        mass2(_s, x[2], x[3], _t2, kOne2, kH1);                                        \
      }                                                                                \
      OUT[v] = dot_read(_s);                                                           \
    }                                                                                  \
  } while (0)
#define MASS_GE(KEY, OUT)        \
  do {                           \
    float _l[VT];                \
    MASS_LOCAL(KEY, _l);         \
    OUT = red.sum(_l);           \
  } while (0)
    // The keys in [LO, HI] (LO >= 1) go to s_list if they are at most MAX, thread by thread; N: how many they are.  A search
    // over the list takes 2 us, over the row 14 rounds of 1.3 (counts) or 2 us (masses).
#define COLLECT(LO, HI, N, MAX)                                                        \
  do {                                                                                 \
    OPAQUE_ROW(row);                                                                   \
    const uint32_t _a = thr1x2(LO), _b = thr1x2((HI) + 1u);                            \
    uint32_t _ca = 0u, _cb = 0u;                                                       \
    _Pragma("unroll") for (int s = 0; s < NS; ++s) {                                   \
      const uint4v x = SLOT(s);                                                        \
      count2(_ca, x[0], x[1], _a, kOne2);                                              \
      count2(_ca, x[2], x[3], _a, kOne2);                                              \
      count2(_cb, x[0], x[1], _b, kOne2);                                              \
      count2(_cb, x[2], x[3], _b, kOne2);                                              \
      NEXT_SLOT();                                                                     \
    }                                                                                  \
    const float _c = (float)((int)((_ca & 0xffffu) + (_ca >> 16)) - (int)((_cb & 0xffffu) + (_cb >> 16))); \
    const float _i = wave_scan(_c);                                                    \
    float* _sc = red.set();                                                            \
    if (lane == 63) _sc[wid] = _i;                                                     \
    __syncthreads();                                                                   \
    float _off = _i - _c, _tot = 0.f;                                                  \
    for (int w = 0; w < T / 64; ++w) {                                                 \
      const float sw = _sc[w];                                                         \
      _off += w < wid ? sw : 0.f;                                                      \
      _tot += sw;                                                                      \
    }                                                                                  \
    N = __builtin_amdgcn_readfirstlane((int)_tot);                                     \
    if (N <= (MAX) && __builtin_amdgcn_ballot_w64(_c > 0.f)) {                         \
      int _p = (int)_off;                                                              \
      _Pragma("unroll") for (int s = 0; s < NS; ++s) {                                 \
        const uint4v x = SLOT(s);                                                      \
        _Pragma("unroll") for (int e = 0; e < 8; ++e) {                                \
          const uint32_t kk = KEYU(x, e);                                              \
          if (kk - (LO) <= (HI) - (LO)) s_list[_p++] = (uint16_t)kk;                   \
        }                                                                              \
        NEXT_SLOT();                                                                   \
      }                                                                                \
    }                                                                                  \
    __syncthreads();                                                                   \
  } while (0)
    uint32_t tau_k = 0;  // top-k: keep elements with key >= tau_k
    if (k > 0) {
      uint32_t lo = 0, hi = 0x3C00u;  // keys of [0, 1.0]
      // Few: the k largest of the threads' own maxima bound the k-th largest element from below (0: fewer than k threads hold
      // any mass); the elements from there on, rarely more than a few times k, are searched in a list.  As k comes near the 1024
      // maxima the bound falls and the list grows: 64 rows of 128256 tokens 37.6 us at k = 40, 48.4 at 400, 59.2 at 600, 136 at 1000
      // (rounds over the row 48), 64 of 32000 26 at 100, 29 at 200, 60 at 1000 (26); two rows per unit 512 at 600, 621 at 800 (671)
      if (k <= kFewest) {
#pragma unroll
        for (int v = 0; v < VT; ++v) {
          const float um = __builtin_amdgcn_exp2f(__builtin_fmaf(mxv[v], c1, c0));
          s_tkey[v * T + t] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(um, um)) & 0xffffu;
        }
        __syncthreads();
        if (t < 64) {
          const uint32_t lb = kth_of_1024(s_tkey, lane, k, 0u, hi);
          if (t == 0) s_lb = lb;
        }
        __syncthreads();
        lo = __builtin_amdgcn_readfirstlane(s_lb);
        const uint32_t from = max(lo, 1u);
        int n;
        COLLECT(from, hi, n, kList);
        if (n <= kList) {
          if (t < 64) {  // (one wave: the list is short)
            while (lo < hi) {
              const uint32_t mid = (lo + hi + 1) >> 1;
              int c = 0;
              for (int i = 0; i < n; i += 64) c += __popcll(__builtin_amdgcn_ballot_w64(i + lane < n && s_list[i + lane] >= mid));
              if (c >= k)
                lo = mid;
              else
                hi = mid - 1;
            }
            if (t == 0) s_lb = lo;
          }
          __syncthreads();
          lo = hi = __builtin_amdgcn_readfirstlane(s_lb);
        }
      }
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        const uint32_t t2 = thr1x2(mid);
        uint32_t c2 = 0u;
OPAQUE_ROW(row);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const uint4v x = SLOT(s);
          count2(c2, x[0], x[1], t2, kOne2);
          count2(c2, x[2], x[3], t2, kOne2);
        }
        if (red.sum_i((int)((c2 & 0xffffu) + (c2 >> 16))) >= k)
          lo = mid;
        else
          hi = mid - 1;
      }
      tau_k = lo;
    }
    // the filters other than top-p are plain lower bounds on the key
    uint32_t L0 = tau_k;
    if (mp > 0.f) L0 = max(L0, (uint32_t)h2bits(mp));        // u_i >= min_p  (u_max = 1)
    if (ta > 0.f) L0 = max(L0, (uint32_t)h2bits(fminf(ta / Z, 1.f)));  // p_i >= top_a p_max^2 <=> u_i >= top_a / Z
    if (L0 > 0x3C00u) L0 = 0x3C00u;                            // never filter out the argmax (u = 1)
    if (L0 == 0u) L0 = 1u;                                     // zero-mass elements are never kept
    // ---- top-p by rejection first (exact): draw s from the distribution over {key >= L0}; s is in the
    // nucleus {key >= tau_p} iff the mass strictly above it is < top_p * mass(top-k set).  Accepted
    // (probability >= top_p), s is exactly a draw from the nucleus-and-filters distribution.  Rejected,
    // tau_p > key_s is known: the exact search for tau_p starts there and a fresh uniform is drawn
    // over {key >= max(tau_p, L0)} — the result is again exactly distributed (the fallback does not
    // depend on the rejected draw).  Saves the ~14 block-wide passes of a threshold search per row in
    // the common case.
    const float tp = uniform_f(p.top_p[b]);
    float target = 0.f;
    // (where the first draw runs over exactly the top-k set its total is that mass)
    const bool target_from_scan = z_from_scan || (tau_k > 0u && L0 == tau_k);
    if (tp < 1.f && !target_from_scan) {
      float mk = Z;
      if (tau_k > 0u) MASS_GE(tau_k, mk);
      target = tp * mk;
    }
    uint32_t ctr[4] = {(uint32_t)p.offsets[b], (uint32_t)(p.offsets[b] >> 32), 0u, 0u};
    philox4x32(ctr, (uint32_t)p.seeds[b], (uint32_t)(p.seeds[b] >> 32));
    uint32_t tau = L0;
    bool check = tp < 1.f;
    int found = 0;
#pragma unroll 1
    for (int attempt = 0; attempt < 2; ++attempt) {
      // ---- inverse-CDF draw over {key >= tau} (order: thread-major, then slot, then element) ----
      float local[VT], excl[VT];
      if (tau <= 1u) {
#pragma unroll
        for (int v = 0; v < VT; ++v) local[v] = zloc[v];  // every positive element is kept: the thread's share of Z
      } else {
        MASS_LOCAL(tau, local);
      }
      // exclusive scan of `local` over threads
      float* sc = red.set();
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        excl[v] = wave_scan(local[v]);
        if (lane == 63) sc[wid + v * (T / 64)] = excl[v];
      }
      if (t == 0) s_owner = 0x7fffffff;
      __syncthreads();
      float wave_off[VT] = {}, total = 0.f;
#pragma unroll
      for (int w = 0; w < kSampT / 64; ++w) {
        const float sw = sc[w];
#pragma unroll
        for (int v = 0; v < VT; ++v)
          if (w < wid + v * (T / 64)) wave_off[v] += sw;
        total += sw;
      }
#pragma unroll
      for (int v = 0; v < VT; ++v) excl[v] = wave_off[v] + excl[v] - local[v];
      if (target_from_scan && attempt == 0) target = tp * total;
      const float u01 = (((attempt == 0 ? ctr[0] : ctr[1]) >> 8) + 0.5f) * (1.0f / 16777216.0f);
      const float u = u01 * total;
      // The owner: the lowest thread whose [excl, excl + local) holds u — or, when rounding put u at or
      // past the end, the last thread with mass (its last kept element is taken).  Its packed u go to
      // LDS and its wave walks them (two elements per dword, an exclusive scan over the lanes) instead
      // of a single lane stepping through 8 * SLOTS elements with a branch each.
#pragma unroll
      for (int v = 0; v < VT; ++v)
        if (local[v] > 0.f && u >= excl[v] && u < excl[v] + local[v]) atomicMin(&s_owner, v * T + t);
      __syncthreads();
      int owner = s_owner;  // block-uniform
      const bool past_end = owner == 0x7fffffff;
      if (past_end) {
        int lastt = -1;
#pragma unroll
        for (int v = 0; v < VT; ++v) lastt = local[v] > 0.f ? v * T + t : lastt;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) lastt = max(lastt, __shfl_xor(lastt, o, 64));
        if (lane == 0) sredi[wid] = lastt;
        __syncthreads();
        lastt = lane < T / 64 ? sredi[lane] : -1;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) lastt = max(lastt, __shfl_xor(lastt, o, 64));
        owner = lastt;
      }
      found = 0x7fffffff;
      if (owner >= 0) {
        if (wid == ((owner & (T - 1)) >> 6)) {  // the owner's wave: its LDS writes are its own reads' (in order, no barrier)
#pragma unroll
          for (int v = 0; v < VT; ++v)
            if (v * T + t == owner) {
#pragma unroll
              for (int j = 0; j < SLOTS; ++j) {
                const uint4v x = SLOT(v * SLOTS + j);
#pragma unroll
                for (int c = 0; c < 4; ++c) s_own[j * 4 + c] = x[c];
              }
              s_oexcl = excl[v];
            }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
          constexpr int ND = SLOTS * 4, P = (ND + 63) / 64;  // lane: dwords [lane*P, lane*P + P)
          float v[2 * P];
          float sl = 0.f;
#pragma unroll
          for (int q = 0; q < P; ++q) {
            const int d = lane * P + q;
            const uint32_t w = d < ND ? s_own[d] : 0u;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const uint32_t kk = h ? (w >> 16) : (w & 0xffffu);
              // tau >= 1: zero-mass elements are never kept
              v[2 * q + h] = kk >= tau ? (float)__builtin_bit_cast(_Float16, (uint16_t)kk) : 0.f;
              sl += v[2 * q + h];
            }
          }
          float acc = s_oexcl + wave_scan(sl) - sl;
          int mine = -1, lastk = -1;
#pragma unroll
          for (int e = 0; e < 2 * P; ++e)
            if (v[e] > 0.f) {
              acc += v[e];
              lastk = e;
              if (mine < 0 && u < acc) mine = e;
            }
          const unsigned long long hit = __ballot(mine >= 0 && !past_end);
          int sel_lane, sel_e;
          if (hit) {
            sel_lane = __ffsll((long long)hit) - 1;
            sel_e = __shfl(mine, sel_lane, 64);
          } else {  // rounding at the owner's top edge, or u past the end: its last kept element
            const unsigned long long any = __ballot(lastk >= 0);
            sel_lane = 63 - __clzll((long long)any);
            sel_e = __shfl(lastk, sel_lane, 64);
          }
          if (lane == sel_lane) {
            const int d = lane * P + (sel_e >> 1);
            const uint32_t w = s_own[d];
            s_found = ((d >> 2) * kSampT + owner) * 8 + 2 * (d & 3) + (sel_e & 1);
            s_fkey = (sel_e & 1) ? (w >> 16) : (w & 0xffffu);
          }
        }
        __syncthreads();
        found = s_found;
      }
      if (found == 0x7fffffff) {
        // u landed past the last kept element through rounding: fall back to argmax (key 0x3C00: always
        // inside the nucleus)
        float bv = -INFINITY;
OPAQUE_ROW(row);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const uint4v x = SLOT(s);
#pragma unroll
          for (int e = 0; e < 8; ++e) bv = fmaxf(bv, GETU(x, e));  // padding past V has u = 0 < u_max = 1
        }
        const float gm = red.max(bv);
        int cand;
OPAQUE_ROW(row);
        LOWEST_INDEX(GETU(x, e) == gm, cand);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
        __syncthreads();
        if (lane == 0) sredi[wid] = cand;
        __syncthreads();
        cand = lane < T / 64 ? sredi[lane] : 0x7fffffff;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
        found = cand == 0x7fffffff ? 0 : cand;
        break;
      }
      if (!check) break;
      // ---- nucleus test of the draw (s_fkey: the drawn element's key, written by the walk) ----
      const uint32_t ks = __builtin_amdgcn_readfirstlane(s_fkey);
      // What lies above is kept too, so it is no more than the rest: an element that carries enough itself needs no sum.
      // (The margin is wider than the sums' rounding, 256 terms each: what the sum would answer is what this answers)
      const float rest = total - (float)__builtin_bit_cast(_Float16, (uint16_t)ks);
      if (__builtin_amdgcn_readfirstlane(rest * 1.0001f < target)) break;
      float mass[VT];
      MASS_LOCAL(ks + 1u, mass);
      int eighth = 0;  // of the keys above, those among an eighth of the row's
      if (T == 512 || t < 512) {
        const uint32_t t2 = thr1x2(ks + 1u);
        uint32_t c2 = 0u;
#pragma unroll
        for (int j = 0; j < SLOTS; j += 2) count2(c2, row[j][0], row[j + 1][0], t2, kOne2);
        eighth = (int)((c2 & 0xffffu) + (c2 >> 16));
      }
      const float above = red.sum(mass, eighth, eighth);
      if (above < target) break;  // accepted (block-uniform)
      // rejected: tau_p > ks.  Exact search for the largest key with mass(>= key) >= target.
      // Keys in the interval that are few go to a list; otherwise rounds over the row halve it.  (A list that does not fit costs
      // a pass: tried again every four rounds, 64 rows of 128256 tokens at top-p 0.9 took 61.5 us, by rounds alone 56.7.)
      uint32_t lo = ks + 1u, hi = 0x3C00u;
      bool listed = lo < hi && __builtin_amdgcn_readfirstlane(eighth) * 8 <= kMassList;
      if (listed) {
        int n;
        COLLECT(lo, hi, n, kMassList);
        listed = n <= kMassList;
        if (listed) {
          // masses as whole numbers of 2^-24 (every fp16 u is one): exact in any order
          const double want = (double)target * 16777216.0;
          if (!kPairs || t < 64) {
            while (lo < hi) {
              const uint32_t mid = (lo + hi + 1) >> 1;
              uint32_t c = 0;
#pragma unroll 4
              for (int i = t; i < n; i += kPairs ? 64 : T) {
                const uint16_t kk = s_list[i];
                c += kk >= mid ? (uint32_t)((float)__builtin_bit_cast(_Float16, kk) * 16777216.f) : 0u;
              }
              double m;
              if constexpr (kPairs)
                m = (double)row_sum4_i(row16_sum_i((int)(c >> 16))) * 65536.0 + (double)row_sum4_i(row16_sum_i((int)(c & 0xffffu)));
              else
                m = red.sum_wide((int)(c >> 12), (int)(c & 4095u));
              if (__builtin_amdgcn_readfirstlane(m >= want))
                lo = mid;
              else
                hi = mid - 1;
            }
            if (kPairs && t == 0) s_lb = lo;
          }
          if constexpr (kPairs) {
            __syncthreads();
            lo = __builtin_amdgcn_readfirstlane(s_lb);
          }
        }
      }
      while (!listed && lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        float mm;
        MASS_GE(mid, mm);
        if (__builtin_amdgcn_readfirstlane(mm >= target))
          lo = mid;
        else
          hi = mid - 1;
      }
      tau = max(lo, L0);
      check = false;
    }
#undef MASS_GE
#undef COLLECT
    token = found;
  }
  if (TOPK && t < 64) {  // one wave: rank-sort the collected top-K candidates (value desc, index asc)
    const int n = min(s_ccount, kCollect);
    for (int r = n + t; r < K; r += 64) {  // fewer finite values than K: empty slots
      p.out_topk_ids[(size_t)b * K + r] = -1;
      p.out_topk_lp[(size_t)b * K + r] = -INFINITY;
    }
    if (t < n) {
      const float v = s_cval[t];
      const int ix = s_cidx[t];
      int rank = 0;
      for (int u = 0; u < n; ++u) {
        const float w = s_cval[u];
        rank += (w > v) || (w == v && s_cidx[u] < ix);
      }
      if (rank < K) {
        p.out_topk_ids[(size_t)b * K + rank] = ix;
        p.out_topk_lp[(size_t)b * K + rank] = v - raw_lse;
      }
    }
  }
  if (t == 0) {
    p.out_token[b] = token;
    p.out_logprob[b] = bf2f(lrow[token]) - raw_lse;
    if (PROC && p.counts && crow_i >= 0) {
      uint16_t* c = p.counts + (size_t)crow_i * p.V + token;
      if (*c < 0xffffu) *c += 1;
    }
  }
}

}  // namespace lwc

extern "C" int lwc_sample(const void* logits, int ld, int V, int B, const float* temperature, const float* top_p,
                          const int* top_k, const float* min_p, const float* top_a, const float* freq_pen,
                          const float* pres_pen, const float* rep_pen, void* counts, const int* count_rows,
                          const float* bias, const int* bias_rows, const unsigned int* mask, const int* mask_rows,
                          const unsigned long long* seeds, const unsigned long long* offsets, int num_logprobs,
                          int mask_logprobs, int need_logprob, int* out_token, float* out_logprob, int* out_topk_ids,
                          float* out_topk_lp, hipStream_t s) {
  using namespace lwc;
  if (V % 32 != 0 || num_logprobs < 0 || num_logprobs > kMaxTopK) return -1;
  if (B == 0) return 0;
  SampleParams p{(const bf16_t*)logits, ld, V, 2LL * B * V >= 128 << 20, temperature, top_p, top_k, min_p, top_a, freq_pen, pres_pen, rep_pen,
                 (uint16_t*)counts, count_rows, bias, bias_rows, mask, mask_rows, seeds, offsets, num_logprobs,
                 mask_logprobs, need_logprob, out_token, out_logprob, out_topk_ids, out_topk_lp};
  const int nvec = V / 8;
  const int slots = (nvec + kSampT - 1) / kSampT;
  const bool proc = bias || mask || counts;
#define LWC_SAMPLE(S)                                                                                                \
  do {                                                                                                               \
    if (proc && num_logprobs > 0) sample_kernel<kSampT, S, S, true, true><<<B, kSampT, 0, s>>>(p);                   \
    else if (proc) sample_kernel<kSampT, S, S, true, false><<<B, kSampT, 0, s>>>(p);                                 \
    else if (num_logprobs > 0) sample_kernel<kSampT, S, S, false, true><<<B, kSampT, 0, s>>>(p);                     \
    else sample_kernel<kSampT, S, S, false, false><<<B, kSampT, 0, s>>>(p);                                          \
  } while (0)
  // 65537 to 131072 tokens, plain rows: two rows per compute unit from four rows per unit on, so that one's load goes on under
  // the other's passes; a thread of a pair does twice the work, and with fewer rows their latency is what counts
  // (128256 tokens, us, one row per unit against two: 64 rows top-p 0.95 35 / 61, 512 72 / 77, 1024 104 / 101, 4096 300 / 280;
  // 4096 rows greedy 216 / 224, temperature alone 258 / 229, top-k 40 537 / 403, 20 logprobs 511 / 399)
  if (slots > 8 && slots <= 16 && !proc && B >= 1024) {
    if (num_logprobs > 0) sample_kernel<512, 16, kRegSlots, false, true><<<B, 512, 0, s>>>(p);
    else sample_kernel<512, 16, kRegSlots, false, false><<<B, 512, 0, s>>>(p);
  } else if (slots <= 4)
    LWC_SAMPLE(4);
  else if (slots <= 8)
    LWC_SAMPLE(8);
  else if (slots <= 16)
    LWC_SAMPLE(16);
  else if (slots <= 20)
    LWC_SAMPLE(20);
  else
    return -1;
#undef LWC_SAMPLE
  return (int)hipGetLastError();
}
