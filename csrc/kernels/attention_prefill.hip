// K4 prefill_attn_varlen (causal, GQA) and K9c encoder_attn (bidirectional) — one flash-attention
// forward for packed variable-length sequences (cu_seqlens), head_dim 32 (bge-small), 64 or 128,
// bf16 in/out.
//
// Workgroup = 4 waves = 64 or 128 query rows of one (sequence, query head); each wave owns one or two sets of 16
// rows and walks 32-key tiles that all 4 waves share through three XOR-swizzled LDS stages filled by LDS-DMA.
// What bounds it: with one set a wave, of long sequences, the reads of K and V from LDS (twice the time of the
// MFMAs: each wave reads a whole tile for 16 rows), which two sets halve; of short ones the reads of q, k and v from
// memory.  The row tiles and query heads that share keys run next to each other on one XCD and find them in its L2.
// Measured (us, 64 rows a workgroup spread over the XCDs -> here): 8 x 2048 rows x 32 (8) heads of 128, causal, 593 -> 297 (920
// TFLOP/s), 1 x 8192 798 -> 506, 64 x 129 62 -> 45; encoders, 4096 x 128 x 12 heads of 64 693 -> 580 (5.5 TB/s), 300 x 500 558 -> 372, 64 of 45 to 180
// rows x 16 heads 24 -> 18; 400 x 256 x 12 heads of 32 211 -> 112; paged, 8 x 2048 697 -> 364, 24 x 16 rows of 900 keys 40 -> 32.
//
// Per wave and key tile (mfma_f32_16x16x32_bf16; lane l: r16 = l & 15, g = l >> 4):
//   S^T = K Q^T :  A = K rows from LDS (ds_read_b128, chunk XOR row swizzle: T2),
//                  B = Q^T held in registers for the whole kernel;
//                  C: lane reg r = S^T[key 4g + r][query r16]   (two 16-key subtiles)
//   O  += P V   :  A = the softmaxed S^T registers themselves (k permuted {4g+0..3, 16+4g+0..3}),
//                  B = V columns by ds_read_b64_tr_b16 (T10 hardware transpose), same permutation;
//                  C: lane reg r = O[query 4g + r][dim 16n + r16]
// so P never leaves registers.  Online softmax in the log2 domain; rows are finite-initialised
// (-1e30) so fully-masked tiles cannot produce NaN.
//
// PAGED mode (mixed chunked prefill, engine/engine.py): the keys / values of sequence s are read straight
// from the paged cache through its block table — K [NB, Hkv, 16, D] token-major, V [NB, Hkv, 4, D, 4]
// 4-token interleaved (the decode layout) — with key positions [0, k_lens[s]) and the sequence's queries
// the last len_q of them (a prompt chunk after its earlier chunks, or after a cached prefix).  A 32-key
// tile is exactly two blocks: each operand tile is two contiguous 4 KiB segments.  K is staged into the
// same swizzled row image; V keeps the interleaved layout in LDS (odd token groups XOR byte bit 7), where
// one ds_read_b64 returns a lane's 4 consecutive keys of one dim — the PV B operand without a transpose.
// V elements of keys past k_lens (the tail of the last block, stale bytes) are zeroed: P is 0 there, but
// 0 x a stale Inf / NaN would not be.  No per-layer gather of the cached keys into contiguous buffers.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace lwc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) short4v lds_short4;

LWC_DEVICE float4v mfma16p(const short8& a, const short8& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

LWC_DEVICE void dma16(const __amdgpu_buffer_rsrc_t& r, char* dst, uint32_t vo) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, vo, 0, 0, 0);
}

constexpr float kLazyRescale = 8.f;
constexpr int kKT = 32;  // keys per tile

struct PrefillParams {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  bf16_t* out;
  const int* cu_seqlens;
  const int* cu_seqlens_k;  // null: keys = queries; else sequence s attends keys [cu_k[s], cu_k[s+1]) and its
                            // queries are the LAST len_q of those positions (cached-prefix prefill)
  int q_stride, k_stride, v_stride, o_stride;  // elements per token row
  int Hq, Hkv, nseq, max_tiles;
  int part_bits;  // log2 of the XCDs that share a sequence's key head (prefill_part_bits)
  float scale;
  int causal;
  // PAGED: block tables [nseq, bt_stride] of the key cache; k_lens [nseq] key positions per sequence
  const int* block_tables;
  const int* k_lens;
  int bt_stride;
  // MX output (D = 128; the fp8 o projection's A operand, as the decode cascade kernel writes it): e4m3 rows
  // out8 [T, Hq * D] (row stride o_stride bytes) + e8m0 scales mx [Hq][mx_rows][4], one per 32 dims
  uint8_t* out8;
  uint8_t* mx;
  int mx_rows;
};

// The block tables come in as a const __restrict__ kernel argument (not through the params struct): the
// compiler may then read them with SCALAR loads.  As vector loads each block id needed an s_waitcnt
// vmcnt(0) — which also waits for the LDS-DMA of the tiles in flight and serialises the pipeline.
// MR: sets of 16 query rows a wave takes
template <int D, bool PAGED, int MR>
__global__ void __launch_bounds__(256) prefill_attn_kernel(PrefillParams p, const int* __restrict__ block_tables) {
  constexpr int kQT = 64 * MR;              // query rows per workgroup
  constexpr int CPR = D / 8;                // 16-byte chunks per row
  constexpr int KS = D / 32;                // k-steps for S
  constexpr int NS = D / 16;                // n-subtiles for O
  constexpr int TILE_BYTES = kKT * D * 2;   // one K or V tile
  constexpr int NST = 3;                    // LDS stages: tiles t (computing), t+1 and t+2 (in flight)
  constexpr int INSTR = TILE_BYTES / 1024;  // 1 KiB LDS-DMA wave-instructions per operand tile
  constexpr int PER_WAVE = 2 * INSTR / 4;   // K + V wave-instructions each of the 4 waves issues per tile
  constexpr int RPI = 1024 / (2 * D);       // tile rows per wave-instruction
  static_assert(PER_WAVE >= 1 && (2 * INSTR) % 4 == 0, "tile must split evenly over 4 waves");
  __shared__ __attribute__((aligned(16))) char smem[NST * 2 * TILE_BYTES];  // [stage][K|V]

  // The workgroups that read the same keys and values, a sequence's row tiles times the query heads of a key head, are
  // neighbours on one XCD (x % 8 with x fastest), or, taken in turn, on as many as parts says: they find them in its L2.
  const int share = (int)((blockIdx.z * gridDim.y + blockIdx.y) * 8 + (blockIdx.x & 7));
  const int unit = share >> p.part_bits, in = (int)(blockIdx.x >> 3 << p.part_bits) + (share & ((1 << p.part_bits) - 1));
  // (the next sequence's heads move on by one: an XCD that met the same one of each would use few channels of its L2, as a row of
  // q, k and v is often a multiple of 2 KiB: 1024 x 128 rows of 16 heads of 64 249 us instead of 194)
  const int seq = unit / p.Hkv, kvh = (unit + seq) % p.Hkv, group = p.Hq / p.Hkv;
  if (unit >= p.nseq * p.Hkv || in >= p.max_tiles * group) return;
  const int hq = kvh * group + in % group, qtile = p.causal ? p.max_tiles - 1 - in / group : in / group;  // (causal: the longest first)
  const int s0 = p.cu_seqlens[seq], len = p.cu_seqlens[seq + 1] - s0;
  const int q0 = qtile * kQT;
  if (q0 >= len) return;  // whole workgroup exits together (uniform)
  // keys: the sequence's own rows, or (cached prefix / PAGED) a longer key range whose last len rows are
  // the queries
  const int ks0 = PAGED ? 0 : p.cu_seqlens_k ? p.cu_seqlens_k[seq] : s0;
  // wave-uniform by construction; readfirstlane lets the compiler keep the DMA buffer resources in SGPRs
  const int klen = __builtin_amdgcn_readfirstlane(PAGED ? p.k_lens[seq]
                                                        : p.cu_seqlens_k ? p.cu_seqlens_k[seq + 1] - ks0 : len);
  const int* bt = PAGED ? block_tables + (size_t)seq * p.bt_stride : nullptr;
  const int qoff = klen - len;  // key position of query row 0
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  // the wave's sets are every fourth, so that the rows a short tile has divide between the waves
  const int wrow = q0 + wid * 16, qrow = wrow + r16;  // the first query of its first set, the lane's (as B-operand column)

  short8 qf[MR][KS];
#pragma unroll
  for (int i = 0; i < MR; ++i) {
    const bf16_t* qp = p.q + (size_t)(s0 + min(qrow + 64 * i, len - 1)) * p.q_stride + hq * D;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[i][s] = *reinterpret_cast<const short8*>(qp + 32 * s + 8 * g);
  }
  // (the largest score times the scale is the largest scaled one where the scale is positive: else q changes its sign.  0 as a
  // scale that leaves every score 0 and a masked one -inf)
  if (p.scale < 0.f) {
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[i][s] ^= (short)0x8000;
  }
  const float sl2 = fmaxf(fabsf(p.scale) * 1.4426950408889634f, 1e-37f);

  const int q_last = min(len, q0 + kQT) - 1;
  const int kv_end = p.causal ? q_last + 1 + qoff : klen;
  const int ntiles = (kv_end + kKT - 1) / kKT;

  // ---- LDS-DMA staging (buffer loads straight into LDS, 16 B per lane, no register round trip) ----
  // Wave-instruction j of a tile (j < INSTR: K image, else V image) writes the image's bytes
  // [1 KiB * (j % INSTR), +1 KiB) lane-linearly; the image's swizzle is applied to the SOURCE address.  Keys
  // at or past klen are out of the buffer resource's range: the hardware writes zeros, no request.
  //  K (and non-paged V) image: row r (key in tile), 16 B chunk c at ((r * CPR) + (c ^ (r % CPR))) * 16.
  //  Paged V image: the tile's two interleaved block segments [4 token groups][D][4], odd groups' bytes
  //  XOR bit 7 (the layout the ds_read_b64 PV operand reads conflict-free).
  const int lrow = lane / CPR, lpc = lane % CPR;
  // not PAGED: a tile's rows follow the last one's: an instruction's offset moves on by a tile with every issue
  uint32_t vo[PER_WAVE];
  if constexpr (!PAGED) {
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
      const int j = wid + 4 * i, r = (j >= INSTR ? j - INSTR : j) * RPI + lrow;
      vo[i] = (uint32_t)(r * (j >= INSTR ? p.v_stride : p.k_stride) * 2 + ((lpc ^ (r % CPR)) * 16));
    }
  }
  const __amdgpu_buffer_rsrc_t rK = uniform_rsrc(PAGED ? p.k : p.k + (size_t)ks0 * p.k_stride + kvh * D, PAGED ? 0 : klen * p.k_stride * 2);
  const __amdgpu_buffer_rsrc_t rV = uniform_rsrc(PAGED ? p.v : p.v + (size_t)ks0 * p.v_stride + kvh * D, PAGED ? 0 : klen * p.v_stride * 2);
  auto issue = [&](int tile, int stage) {
    char* kb = smem + stage * 2 * TILE_BYTES;
#pragma unroll
    for (int i = 0; i < PER_WAVE; ++i) {
      const int j = wid + 4 * i;  // wave-uniform
      const bool isv = j >= INSTR;
      const int jj = isv ? j - INSTR : j;
      char* dst = kb + (isv ? TILE_BYTES : 0) + jj * 1024;
      if constexpr (PAGED) {
        // the instruction's 1 KiB lies in one block segment: K rows jj*RPI.. or V bytes jj*1024..
        const int half = isv ? (jj * 1024) / 4096 : (jj * RPI) / 16;
        const int blk = bt[__builtin_amdgcn_readfirstlane(2 * tile + half)];
        const int valid = min(max(klen - (tile * kKT + half * 16), 0), 16);  // keys of this block in range
        const bf16_t* segp = (isv ? p.v : p.k) + ((size_t)blk * p.Hkv + kvh) * 16 * D;
        uint32_t vo, nrec;
        if (!isv) {
          const int r = jj * RPI + lrow;  // key in tile
          vo = (uint32_t)(((r % 16) * CPR + (lpc ^ (r % CPR))) * 16);
          nrec = (uint32_t)(valid * D * 2);
        } else {
          const int P = jj * 1024 + lane * 16;                     // byte of the V image
          const int bsrc = (P ^ (((P / (D * 8)) & 1) << 7)) % 4096;  // byte in the block segment
          vo = (uint32_t)bsrc;
          nrec = (uint32_t)(((valid + 3) / 4) * D * 8);  // whole token groups; a partial group is fixed up
        }
        // readfirstlane: uniform already, but the compiler may compute it on the VALU (then every DMA became a
        // waterfall loop over "divergent" resources)
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)segp, (short)0, __builtin_amdgcn_readfirstlane(nrec), 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16, vo, 0, 0, 0);
      } else {
        if (isv) dma16(rV, dst, vo[i]);
        else dma16(rK, dst, vo[i]);
        vo[i] += (uint32_t)(kKT * (isv ? p.v_stride : p.k_stride) * 2);
      }
    }
  };

  float4v o[MR][NS];
  float m[MR], l[MR];
#pragma unroll
  for (int i = 0; i < MR; ++i) {
#pragma unroll
    for (int n = 0; n < NS; ++n) o[i][n] = float4v{0.f, 0.f, 0.f, 0.f};
    m[i] = -1e30f, l[i] = 0.f;
  }
  // the wave's sets with rows, and the tiles they see (it loads for the others all the same)
  const int sets = wrow >= len ? 0 : MR > 1 && wrow + 64 < len ? MR : 1, last_row = min(wrow + 64 * (sets - 1) + 16, len);
  const int wtiles = sets == 0 ? 0 : p.causal ? min(ntiles, (last_row + qoff + kKT - 1) / kKT) : ntiles;
  // those that the first set sees: its rows end 64 before the second's, and the values past them may be infinite or NaN (times a
  // probability of 0)
  const int first_tiles = MR > 1 && sets > 1 && p.causal ? max(0, min(ntiles, (wrow + 16 + qoff + kKT - 1) / kKT)) : ntiles;

  issue(0, 0);
  if (ntiles > 1) issue(1, 1);
  // loop-invariant LDS read offsets of this lane (the stage base is a compile-time immediate below)
  int kofs[KS], vofs[NS];
#pragma unroll
  for (int s = 0; s < KS; ++s) kofs[s] = (r16 * CPR + ((4 * s + g) ^ (r16 & (CPR - 1)))) * 16;
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    if constexpr (PAGED) {
      vofs[n] = ((g * D + 16 * n + r16) << 3) ^ ((g & 1) << 7);
    } else {
      const int qq = r16 >> 2, pp = r16 & 3;
      const int rowA = 4 * g + qq, chunk = 2 * n + (pp >> 1);
      vofs[n] = (rowA * CPR + (chunk ^ (rowA & (CPR - 1)))) * 16 + (pp & 1) * 8;
    }
  }
  // for the sets SET0 .. SETS - 1
  auto tile_step = [&](const int t, const auto buf, auto set0, auto nsets) {
    constexpr int SET0 = decltype(set0)::value, SETS = decltype(nsets)::value;
    // own DMA of tile t landed (tile t+1's may stay in flight), then every wave's (barrier); the barrier also
    // ends every wave's reads of tile t-1, whose stage tile t+2 now refills
    if (t + 1 < ntiles)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_WAVE) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + 2 < ntiles) issue(t + 2, (t + 2) % NST);
    if constexpr (PAGED) {
      // the last tile's partially valid token group holds stale V bytes of keys >= klen (P is 0 there, but
      // 0 x a stale Inf / NaN would not be): zero them (uniform branch: the last tile only)
      const int tk = klen - t * kKT;  // keys of this tile in range
      if (tk < kKT && (tk & 3)) {
        char* vimg = smem + buf * 2 * TILE_BYTES + TILE_BYTES;
        const int half = tk / 16, grp = (tk % 16) / 4;
        if (threadIdx.x < D) {
          for (int r = tk & 3; r < 4; ++r) {
            const int bsrc = half * 4096 + grp * D * 8 + threadIdx.x * 8 + r * 2;
            *reinterpret_cast<bf16_t*>(vimg + (bsrc ^ (((bsrc / (D * 8)) & 1) << 7))) = 0;
          }
        }
        __syncthreads();
      }
    }
    const char* kb = smem + buf * 2 * TILE_BYTES;  // (a compile-time stage: LDS reads take immediate offsets)
    const char* vb = kb + TILE_BYTES;
    if (t >= wtiles) return;
    // ---- S^T for the two 16-key subtiles ----
    float4v sa[SETS], sb[SETS];
#pragma unroll
    for (int i = SET0; i < SETS; ++i) sa[i] = sb[i] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const short8 ka = *reinterpret_cast<const short8*>(kb + kofs[s]);
      const short8 kbv = *reinterpret_cast<const short8*>(kb + kofs[s] + 16 * CPR * 16);  // keys 16..31
#pragma unroll
      for (int i = SET0; i < SETS; ++i) {
        sa[i] = mfma16p(ka, qf[i][s], sa[i]);
        sb[i] = mfma16p(kbv, qf[i][s], sb[i]);
      }
    }
    // ---- mask + online softmax (per query r16 of a set) ----
    short8 pf[SETS];
    float mxs[SETS];
#pragma unroll
    for (int i = SET0; i < SETS; ++i) {
      // interior tile (every key in range and, causal, at or before the set's first query): no mask
      const int tlast = t * kKT + kKT - 1;
      if (!(tlast < klen && (!p.causal || tlast <= wrow + 64 * i + qoff))) {  // wave-uniform
        // of the lane's keys 4 g + r and 16 + 4 g + r, those below lim are seen
        const int lim = (p.causal ? min(klen, qrow + 64 * i + qoff + 1) : klen) - t * kKT - 4 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sa[i][r] = r < lim ? sa[i][r] : -INFINITY;
          sb[i][r] = 16 + r < lim ? sb[i][r] : -INFINITY;
        }
      }
      float mx = fmaxf(fmaxf(sa[i][0], sa[i][1]), sa[i][2]);
      mx = fmaxf(fmaxf(mx, sa[i][3]), sb[i][0]);
      mx = fmaxf(fmaxf(mx, sb[i][1]), sb[i][2]);
      mx = fmaxf(mx, sb[i][3]) * sl2;
      mxs[i] = mx;
    }
    // lazy rescale (log2 domain): the running max only moves, and O / l are rescaled, when some row's new
    // scores exceed it by more than kLazyRescale, so P <= 2^8 and most tiles neither reduce their maximum over the lanes of a
    // row nor shuffle alphas nor multiply O.  One branch for both sets: with one each, registers are copied around them (188 of them
    // instead of 166, and two workgroups a CU instead of three: 8 x 2048 rows x 32 heads of 128 345 us, so 297)
    if (t == 0) {
#pragma unroll
      for (int i = SET0; i < SETS; ++i) m[i] = fmaxf(m[i], row_max4(mxs[i]));
    } else {
      bool need = false;
#pragma unroll
      for (int i = SET0; i < SETS; ++i) need |= mxs[i] > m[i] + kLazyRescale;
      if (__any(need)) {  // wave-uniform
#pragma unroll
        for (int i = SET0; i < SETS; ++i) {
          const float m_new = fmaxf(m[i], row_max4(mxs[i]));
          const float alpha = __builtin_amdgcn_exp2f(m[i] - m_new);
          l[i] *= alpha;
          m[i] = m_new;
          float al[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) al[r] = __shfl(alpha, 4 * g + r, 64);
#pragma unroll
          for (int n = 0; n < NS; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[i][n][r] *= al[r];
        }
      }
    }
#pragma unroll
    for (int i = SET0; i < SETS; ++i) {
      float pa[4], pb[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pa[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[i][r], sl2, -m[i]));  // raw v_exp_f32: -inf -> 0, arguments <= 8
        pb[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sb[i][r], sl2, -m[i]));
      }
      l[i] += ((pa[0] + pa[1]) + (pa[2] + pa[3])) + ((pb[0] + pb[1]) + (pb[2] + pb[3]));  // (the lane's keys; the row's at the end)
      pf[i] = __builtin_bit_cast(short8, uint4v{pack_bf16x2(pa[0], pa[1]), pack_bf16x2(pa[2], pa[3]),
                                                pack_bf16x2(pb[0], pb[1]), pack_bf16x2(pb[2], pb[3])});
    }
    // ---- O += P V ----
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      short4v va4, vb4;
      if constexpr (PAGED) {  // lane: keys 4g..4g+3 (block A half) and 16+4g..16+4g+3 (block B half) of dim 16n + r16, 8 B each
        va4 = *reinterpret_cast<const short4v*>(vb + vofs[n]);
        vb4 = *reinterpret_cast<const short4v*>(vb + TILE_BYTES / 2 + vofs[n]);
      } else {  // V columns via the hardware transpose read; rows 4g+qq and 16+4g+qq: same swizzle
        va4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(vb + vofs[n]));
        vb4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(vb + vofs[n] + 16 * CPR * 16));
      }
      const short8 vf = __builtin_shufflevector(va4, vb4, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int i = SET0; i < SETS; ++i) o[i][n] = mfma16p(pf[i], vf, o[i][n]);
    }
  };
  constexpr std::integral_constant<int, 0> n0{};
  auto walk = [&](auto nsets) {
    for (int t = 0; t < first_tiles; t += NST) {  // unrolled by the stage count: every stage base is a constant
      tile_step(t, n0, n0, nsets);
      if (t + 1 < first_tiles) tile_step(t + 1, std::integral_constant<int, 1>{}, n0, nsets);
      if (t + 2 < first_tiles) tile_step(t + 2, std::integral_constant<int, 2>{}, n0, nsets);
    }
  };
  if (MR == 1 || sets < MR) walk(std::integral_constant<int, 1>{});
  else walk(std::integral_constant<int, MR>{});
  if constexpr (MR > 1) {
#pragma unroll 1
    for (int t = first_tiles; t < ntiles; ++t) tile_step(t, t % NST, std::integral_constant<int, MR - 1>{}, std::integral_constant<int, MR>{});
  }

  // ---- epilogue: normalise, stage the wave's rows through LDS, 16 B stores ----
  __syncthreads();
  bf16_t* ot = reinterpret_cast<bf16_t*>(smem) + wid * 16 * MR * D;
#pragma unroll
  for (int i = 0; i < MR; ++i) {
    const float li = row_sum4(l[i]);
    float linv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float lr = __shfl(li, 4 * g + r, 64);
      linv[r] = lr > 0.f ? 1.f / lr : 0.f;
    }
#pragma unroll
    for (int n = 0; n < NS; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) ot[(16 * i + 4 * g + r) * D + 16 * n + r16] = f2bf(o[i][n][r] * linv[r]);
  }
  __syncthreads();
  if constexpr (D == 128) {
    if (p.out8 != nullptr) {  // uniform
      // lane: row lane / 4 of 16, 32-dim block lane % 4 -> 32 e4m3 bytes + one e8m0 scale
#pragma unroll
      for (int i = 0; i < MR; ++i) {
        const int row = 16 * i + (lane >> 2), b = lane & 3;
        const int qr = wrow + 64 * i + (lane >> 2);
        float v[32];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float f[8];
          unpack8(*reinterpret_cast<const uint4v*>(ot + row * D + 32 * b + 8 * c), f);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[8 * c + j] = f[j];
        }
        float amax = 0.f;
#pragma unroll
        for (int j = 0; j < 32; ++j) amax = fmaxf(amax, fabsf(v[j]));
        const int e = mx_exp(amax);
        const float sc = __builtin_amdgcn_ldexpf(1.f, -e);
        uint32_t w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          uint32_t x = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * k] * sc, v[4 * k + 1] * sc, 0, false);
          w[k] = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * k + 2] * sc, v[4 * k + 3] * sc, x, true);
        }
        if (qr < len) {
          uint8_t* dst = p.out8 + (size_t)(s0 + qr) * p.o_stride + hq * D + 32 * b;
          *reinterpret_cast<uint4v*>(dst) = uint4v{w[0], w[1], w[2], w[3]};
          *reinterpret_cast<uint4v*>(dst + 16) = uint4v{w[4], w[5], w[6], w[7]};
          p.mx[((size_t)hq * p.mx_rows + s0 + qr) * 4 + b] = (uint8_t)(e + 127);
        }
      }
      return;
    }
  }
  for (int c = lane; c < 16 * MR * CPR; c += 64) {
    const int row = c / CPR, ch = c % CPR;
    const int qr = wrow + row / 16 * 64 + row % 16;
    if (qr < len)
      *reinterpret_cast<uint4v*>(p.out + (size_t)(s0 + qr) * p.o_stride + hq * D + ch * 8) =
          *reinterpret_cast<const uint4v*>(ot + row * D + ch * 8);
  }
}

}  // namespace lwc

namespace lwc {
// Two sets of rows a wave (128 rows a workgroup) where that leaves the chip enough workgroups and a sequence's last one enough
// rows.  us, one set / two: 1024 sequences x 16 heads of 64, of 40 rows 67 / 89, 70 136 / 122, 96 172 / 152, 128 194 / 192, 132 263 / 318, 160 286 /
// 325, 192 344 / 378, 200 453 / 418, 256 546 / 495; 64 x 32 (8) heads of 128, of 100 rows 39 / 38, 160 61 / 59, 260 125 / 118; few workgroups (of
// 128 rows): 1 x 1000 (256) 25 / 32, 4 x 500 (512) 24 / 26, 5 x 260 (480) 17 / 19, 20 x 120 with up to 192 rows (1280) 18 / 21, but 8 x 300 (768)
// 23 / 20, 2 x 1500 (768) 59 / 53
inline int prefill_sets(int nseq, int max_seqlen, int Hq, int D) {
  const long long wgs = (long long)nseq * ((max_seqlen + 127) / 128) * Hq;
  const bool short_second = max_seqlen > 128 && max_seqlen <= 192;
  return max_seqlen > 64 && wgs >= 768 && !(short_second && (D < 128 || wgs < 2048)) ? 2 : 1;
}
// The XCDs over which a sequence's key head goes: as few as leave none of them with an eighth more than its share because of the
// longest sequence (the others in equal parts of the rest of all rows; work by the square of the rows).
// us, a key head on one XCD / so, 32 (1) heads of 128, causal: 1 x 8192 rows 3333 / 581, 1 x 2048 293 / 57, 4096 beside 30 x 60 894 / 182; 32 (2)
// 1901 / 576, 32 (4) 987 / 555; 12 heads of 64, 1 x 8192 338 / 274; 9 heads 323 / 245.  More XCDs than that read the keys more often:
// 32 (8) heads 1 x 2048 on 1 / 2 / 4 / 8 52 / 57 / 59 / 67, 40 x 300 rows of 12 heads 30 / 37 / 40 / 63.
inline int prefill_part_bits(int nseq, int rows, int max_seqlen, int Hq, int Hkv, int sets) {
  const double longest = (double)max_seqlen * max_seqlen, other = nseq > 1 ? std::max(0.0, (double)rows - max_seqlen) / (nseq - 1) : 0;
  const double fair = Hkv / 8.0 * (longest + (nseq - 1) * other * other);
  const int workgroups = (max_seqlen + 64 * sets - 1) / (64 * sets) * (Hq / Hkv);
  int bits = 0;
  auto over = [&] { return ((((Hkv << bits) + 7) / 8) / (double)(1 << bits) - Hkv / 8.0) * longest; };
  while (bits < 3 && 2 << bits <= workgroups && over() > 0.125 * fair) ++bits;
  return bits;
}
template <int D, bool PAGED, int MR>
void launch_rows(PrefillParams p, int max_seqlen, hipStream_t s) {
  p.max_tiles = (max_seqlen + 64 * MR - 1) / (64 * MR);
  // 8 x (a part of row tiles x query heads of a key head) by the eighths of (sequences x key heads x parts)
  const int parts = 1 << p.part_bits, per = (p.max_tiles * (p.Hq / p.Hkv) + parts - 1) / parts;
  const int shares = (int)(((long long)p.nseq * p.Hkv * parts + 7) / 8), y = std::min(shares, 32768);
  prefill_attn_kernel<D, PAGED, MR><<<dim3(8 * per, y, (shares + y - 1) / y), 256, 0, s>>>(p, p.block_tables);
}
// rows: of all sequences
template <int D, bool PAGED>
int launch_prefill(PrefillParams p, int rows, int max_seqlen, hipStream_t s) {
  const int sets = prefill_sets(p.nseq, max_seqlen, p.Hq, D);
  p.part_bits = prefill_part_bits(p.nseq, rows, max_seqlen, p.Hq, p.Hkv, sets);
  if (sets == 2) launch_rows<D, PAGED, 2>(p, max_seqlen, s);
  else launch_rows<D, PAGED, 1>(p, max_seqlen, s);
  return (int)hipGetLastError();
}
}  // namespace lwc

// How a call is cut up: query rows of a workgroup, XCDs that share a sequence's key head.
extern "C" void lwc_prefill_plan(int nseq, int rows, int max_seqlen, int Hq, int Hkv, int D, int* tile, int* parts) {
  const int sets = lwc::prefill_sets(nseq, max_seqlen, Hq, D);
  *tile = 64 * sets;
  *parts = 1 << lwc::prefill_part_bits(nseq, rows, max_seqlen, Hq, Hkv, sets);
}

// rows: of q
extern "C" int lwc_prefill_attention(const void* q, const void* k, const void* v, void* out, const int* cu_seqlens,
                                     const int* cu_seqlens_k, int nseq, int rows, int max_seqlen, int q_stride, int k_stride, int v_stride,
                                     int o_stride, int Hq, int Hkv, int D, float scale, int causal, hipStream_t s) {
  using namespace lwc;
  if (Hq % Hkv != 0) return -1;
  if (nseq == 0 || max_seqlen == 0) return 0;
  PrefillParams p{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, (bf16_t*)out, cu_seqlens, cu_seqlens_k,
                  q_stride, k_stride,
                  v_stride, o_stride, Hq, Hkv, nseq, 0, 0, scale, causal, nullptr, nullptr, 0,
                  nullptr, nullptr, 0};
  return D == 128 ? launch_prefill<128, false>(p, rows, max_seqlen, s) : D == 64 ? launch_prefill<64, false>(p, rows, max_seqlen, s)
         : D == 32 ? launch_prefill<32, false>(p, rows, max_seqlen, s) : -1;
}

// The same with the output in MX form (D = 128, keys = queries): out8 [T, Hq * 128] e4m3 (row stride o8_stride
// bytes), mx [Hq][mx_rows >= T][4] e8m0 — what the fp8 o projection's block-scaled MFMAs read, so the bf16
// output and its row quantisation pass are gone.
extern "C" int lwc_prefill_attention_mx(const void* q, const void* k, const void* v, void* out8, void* mx,
                                        int mx_rows, const int* cu_seqlens, int nseq, int rows, int max_seqlen,
                                        int q_stride, int k_stride, int v_stride, int o8_stride, int Hq, int Hkv, float scale, int causal, hipStream_t s) {
  using namespace lwc;
  if (Hq % Hkv != 0 || o8_stride % 16 != 0) return -1;
  if (nseq == 0 || max_seqlen == 0) return 0;
  PrefillParams p{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, nullptr, cu_seqlens, nullptr, q_stride,
                  k_stride, v_stride, o8_stride, Hq, Hkv, nseq, 0, 0, scale, causal, nullptr, nullptr, 0,
                  (uint8_t*)out8, (uint8_t*)mx, mx_rows};
  return launch_prefill<128, false>(p, rows, max_seqlen, s);
}

// Causal prefill of query chunks against a PAGED KV cache (D = 128, block size 16): sequence s has queries
// cu_seqlens[s]..cu_seqlens[s+1] = its key positions [k_lens[s] - len_q, k_lens[s]); its keys come from
// kc / vc through block_tables[s] (bt_stride entries per row, covering ceil(k_lens[s] / 16) blocks).
extern "C" int lwc_prefill_attention_paged(const void* q, const void* kc, const void* vc, void* out,
                                           const int* cu_seqlens, const int* block_tables, const int* k_lens,
                                           int bt_stride, int nseq, int rows, int max_seqlen, int q_stride, int o_stride,
                                           int Hq, int Hkv, int D, float scale, hipStream_t s) {
  using namespace lwc;
  if (Hq % Hkv != 0 || D != 128) return -1;
  if (nseq == 0 || max_seqlen == 0) return 0;
  PrefillParams p{(const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc, (bf16_t*)out, cu_seqlens, nullptr,
                  q_stride, 0, 0, o_stride, Hq, Hkv, nseq, 0, 0, scale, 1, block_tables, k_lens, bt_stride,
                  nullptr, nullptr, 0};
  return launch_prefill<128, true>(p, rows, max_seqlen, s);
}
