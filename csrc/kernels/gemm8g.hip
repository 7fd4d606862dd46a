// K6g' grouped GEMM in the 256x256 tiles of gemm8p.hip (the MoE expert FFNs), fp8 and bf16:
//   C[r, :] = (A[a_rows[r], :] . W_g^T) * a_scale[a_rows[r]] * w_scale[g, :]   for rows r of group g
// with groups = the experts' contiguous row segments row_off[g]..row_off[g+1] (device table, no host
// sync, graph-capturable) and A gathered through a_rows (MoE dispatch without a permute copy).
//
// Why a second grouped kernel: the 128x128 register-staged kernel (gemm.hip) pays two barriers and a
// full LDS rewrite per 128-byte K step for 16 block-scaled MFMAs per wave — latency-bound at ~1.0-1.3
// PF/s fp8 (profiles/moe_r32.md: MFMA busy ~20 %).  Large decode batches give every expert >= 2 full
// 256-row tiles (T = 2048 tokens, top-2, 8 experts: 512 rows each), which is the dense tile's regime (gemm8p.hip):
//   * 8 waves = 2 (M) x 4 (N), wave tile 128 x 64; K tile = 128 BYTES (= 128 e4m3), four 16 KiB LDS
//     units A0 A1 B0 B1 per K tile, two K-tile buffers (128 KiB), LDS-DMA (buffer_load ... lds) staging
//     with the swizzle on the SOURCE address, two phases per K tile with counted vmcnt, operands in registers at the
//     raw s_barrier and the two wave rows staggered by one barrier — byte for byte the gemm8p pipeline;
//   * MFMA: the block-scaled mfma_scale_f32_16x16x128_f8f6f4 with unit e8m0 scales: a lane's two 16 B
//     fragments (k-chunks q and 4+q of the 128-byte slice) form one 32-byte operand, so a phase issues
//     16 MFMAs of twice the bf16 cycle count — the same MFMA cycles per phase as gemm8p at 2x the FLOPs;
//   * A rows: per-lane DMA source offsets from a_rows (rows past the group's end are not loaded and are
//     masked at the store); W: the group's [N, K] slab through its own descriptor;
//   * epilogue: a lane holds eight consecutive columns of eight rows: eight activation scales and 16 channel scales
//     instead of 32 and 4, no LDS, 16 B stores (rows < the group's end only).
// Measured against four phases of half the MFMAs with the wait for their reads behind the barrier and an epilogue through LDS, us:
// dense fp8 8682 rows x 28672 x 4096 SwiGLU 794 -> 751, x 4096 x 14336 468 -> 449; 8 bf16 experts of 4096 rows, [14336, 4096] 2931 ->
// 2908, [4096, 7168] 1661 -> 1617 (bound by the card's power there).  64 documents through three e5 layers 4255 -> 4045.
// Work distribution: one 256 x 256 tile per workgroup; workgroup ids are dealt round-robin to the 8
// XCDs, and XCD x walks the n-tiles n = x (mod 8) with all m-tiles of an n-tile consecutive, so the
// weight tile of an expert is read from HBM once per XCD and reused from its L2 by the expert's other
// m-tiles.  Surplus slots (routing decides the m-tile count at run time) exit immediately.
//
// bf16 (kBf16 / kBf16Swiglu): the same bytes move through the same pipeline — a K tile of 128 bytes is 64 bf16, a
// phase's 16 double-length fp8 MFMAs become 32 bf16 ones as in gemm8p — without scales.  Bound by the matrix cores (the
// 128-row kernel 4720 and 2376 us at the experts above).
#include "common.h"

namespace lwc {
namespace g8g {

typedef int v8i32 __attribute__((ext_vector_type(8)));

constexpr int kUnitB = 128 * 128;   // 128 rows x 128 B
constexpr int kBufB = 4 * kUnitB;   // one K tile: A0 A1 B0 B1
constexpr int kLdsB = 2 * kBufB;    // 128 KiB
constexpr int kUA0 = 0, kUA1 = kUnitB, kUB0 = 2 * kUnitB, kUB1 = 3 * kUnitB;

struct Params {
  const uint8_t* A;       // [rows_a, K] e4m3
  const uint8_t* W;       // [G][N, K] e4m3
  bf16_t* C;              // [rows, ldc]
  const int* row_off;     // [G + 1]
  const int* a_rows;      // [rows] or null
  const float* a_scale;   // [rows_a]
  const float* w_scale;   // [G][N]
  int G, N, K, lda, ldc;  // K and lda in BYTES of A / W rows, ldc in elements of C
  int rows_a;             // rows of A (DMA bounds)
  int slots, n_tiles;     // m-tile slots per n-tile, n-tiles
  int rows_c;             // output rows when row_off is null (dense: G = 1)
  int gn;                 // grouped: n-tiles an XCD walks per m-slot before the next slot (>= 1)
  int skip_empty;         // skip the MFMAs of empty 64-row blocks (skips_empty)
  // MX activations (kMxOut producer / kMxA consumer): e8m0 block scales [K / 128][s_rows][4] bytes, block b
  // of a 128-byte K slice = its bytes [32b, 32b + 32).  (The block-scaled MFMA takes a lane's two 16-byte
  // fragments as K [16q, 16q + 16) and [64 + 16q, ...) of its 128 and scales K block b by the byte lane
  // group b supplies — measured, scripts/mx_probe.py.)
  const uint8_t* a_mx;    // kMxA: scales of A (a_scale unused)
  uint8_t* mx_out;        // kMxOut: scales of the e4m3 output (C is then e4m3 [rows, ldc bytes])
  int s_rows;             // rows of the scale planes
};

// kernel modes: output / A operand handling
constexpr int kPlain = 0;   // bf16 out, A per-row scaled
constexpr int kSwiglu = 1;  // SwiGLU epilogue, bf16 out
constexpr int kMxOut = 2;   // SwiGLU epilogue, e4m3 out with MX block scales (feeds a kMxA GEMM)
constexpr int kMxA = 3;     // bf16 out, A carries MX block scales
constexpr int kBf16 = 4;        // bf16 A and W, bf16 out
constexpr int kBf16Swiglu = 5;  // bf16 A and W, SwiGLU epilogue, bf16 out
constexpr int kMxLds = 4096;  // kMxA: the two K buffers' scale tiles (256 rows x 4 blocks, twice: see the DMA)

// sb: the lane's e8m0 scale of the second operand (its row's, for the lane's K block)
LWC_DEVICE float4v mfma8(const uint4v& a0, const uint4v& a1, const uint4v& b0, const uint4v& b1, const float4v& c, int sb) {
  const v8i32 av = {(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w, (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
  const v8i32 bv = {(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w, (int)b1.x, (int)b1.y, (int)b1.z, (int)b1.w};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 0, 0, 0, 127, 0, sb);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
LWC_DEVICE float4v mfma16(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

// grouped default: an XCD takes all of its n-tiles for one m-slot before the next slot (gn = n-tiles per XCD).
// Config 5's routed shapes at 4096 tokens, one MI355X, medians of 5 interleaved rounds (scripts/g8g_order_ab.py):
// gate|up + SwiGLU 908.1 -> 893.4 us, down 474.3 -> 466.7 us vs gn = 1 (the n-tile-major order); with the
// empty-block MFMA skip below as well 878.0 / 443.9 us.  LWC_G8G_GN overrides.
constexpr int kDefaultGn = 1 << 20;

LWC_DEVICE float silu8(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

// SWIGLU: W's rows are gate / up interleaved in blocks of 32 (ops.swiglu_interleave per expert), so each
// wave's 64 columns are one gate block and its up block; the epilogue applies the scales, then
// silu(gate) * up, and writes [rows, N / 2] bf16 — the [rows, N] gate|up intermediate never reaches HBM.
template <int MODE>
__global__ void __launch_bounds__(512) gemm8g_kernel(Params p) {
  constexpr bool SWIGLU = MODE == kSwiglu || MODE == kMxOut || MODE == kBf16Swiglu;
  constexpr bool MXA = MODE == kMxA;
  constexpr bool BF = MODE == kBf16 || MODE == kBf16Swiglu;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // ---- work item: XCD-grouped (n-tile, m-slot), then (group, m-tile) of the slot ----
  const int id = blockIdx.x, xcd = id & 7, local = id >> 3;
  int g = 0, m_begin = 0, m_end = 0, ntile = 0;
  if (p.row_off == nullptr) {
    // dense (G = 1, rows [0, rows_c), slots = m-tiles): XCD x runs a contiguous range of the GROUPED tile
    // order (8 m-tiles x every n-tile, m fastest), so the workgroups resident on an XCD at once share a
    // few A and W panels in its L2 instead of each streaming its own A panel from HBM (at the embedder's
    // 266k-row prefill the expert-style n-major order re-read A once per n-tile)
    const int T = p.slots * p.n_tiles, per = (T + 7) / 8, t = xcd * per + local;
    if (local >= per || t >= T) return;  // uniform
    const int group = 8 * p.n_tiles, first_m = (t / group) * 8, gsz = min(p.slots - first_m, 8), in = t % group;
    m_begin = (first_m + in % gsz) * 256;
    m_end = p.rows_c;
    ntile = in / gsz;
  } else {
    // an XCD owns n-tiles xcd, xcd + 8, ...; it walks them in windows of gn: every m-slot (the experts'
    // row tiles back to back) takes the window's gn n-tiles in a row, so the workgroups resident at once
    // hold ~32/gn consecutive row tiles x gn weight panels (each expert's panel still read once, every A
    // tile once per window instead of once per n-tile)
    const int w = p.slots * p.gn, in = local % w;
    ntile = ((local / w) * p.gn + in % p.gn) * 8 + xcd;
    int slot = in / p.gn;
    if (ntile >= p.n_tiles) return;  // uniform
    for (; g < p.G; ++g) {
      const int r0 = p.row_off[g], r1 = p.row_off[g + 1];
      const int nt = (r1 - r0 + 255) / 256;
      if (slot < nt) {
        m_begin = r0 + slot * 256;
        m_end = r1;
        break;
      }
      slot -= nt;
    }
    if (g >= p.G) return;  // surplus slot (uniform)
  }
  const int n0 = ntile * 256;
  const int KT = p.K / 128;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  const int wr = wid >> 2, wc = wid & 3;

  // per-thread DMA geometry: unit u, instruction i -> unit row ru = i*64 + tid/8 at LDS chunk tid%8, holding a
  // global chunk of that row (swizzle on the source, gemm8p.hip's).  A rows are gathered: source row of tile row t.
  const int chkA = ((tid & 7) ^ ((tid >> 4) & 7)) * 16, chkW = ((tid & 7) ^ ((tid >> 6 & 3) * 2 + (tid >> 4 & 1))) * 16;
  uint32_t voA[2][2], voW[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = m_begin + i * 128 + h * 64 + (tid >> 3);
      // (past the group's end: past the resource's, zeros and no memory request)
      voA[h][i] = r < m_end ? (uint32_t)((p.a_rows ? p.a_rows[r] : r) * p.lda + chkA) : 0x7fffffffu;
      voW[h][i] = (uint32_t)(((2 * i + (tid >> 8)) * 64 + h * 32 + ((tid >> 3) & 31)) * p.K + chkW);
    }
  const int dst_lane0 = wid * 64 * 16;
  const int pos = (q ^ (r16 >> 1)) << 4;
  const int offA = (wr * 64 + r16) * 128, offW = (wc * 32 + 8 * (r16 >> 2) + (r16 & 3)) * 128;

  // kMxA: the tile's scales ([row][4 blocks], one dword per row) DMA'd with unit A0, one dword piece per thread
  // (an LDS-DMA lands every lane's piece on a 4-byte slot, so no narrower piece packs): threads 256..511 load
  // a second copy, keeping every wave's vmcnt count equal; a lane then reads its 8 fragments' bytes
  uint32_t voS = 0u;
  if constexpr (MXA) {
    int r = m_begin + (tid & 255);
    if (r >= m_end) r = m_begin;
    voS = (uint32_t)(r * 4);
  }
  const int numA = p.rows_a * p.lda, numW = min(p.N - n0, 256) * p.K, numS = MXA ? (p.K / 128) * p.s_rows * 4 : 0;
  const uint8_t* srcW = p.W + ((size_t)g * p.N + n0) * p.K;
  // unit u of K tile kt; past the last one the same instructions without a memory request
  auto stage = [&](int u, int kt) {
    uint8_t* buf = smem + (kt & 1) * kBufB;
    const bool live = kt < KT;
    const __amdgpu_buffer_rsrc_t r = u < 2 ? uniform_rsrc(p.A, live ? numA : 0) : uniform_rsrc(srcW, live ? numW : 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      auto* dst = (__attribute__((address_space(3))) void*)(buf + u * kUnitB + i * 512 * 16 + dst_lane0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, u < 2 ? voA[u][i] : voW[u - 2][i], kt * 128, 0, 0);
    }
    if constexpr (MXA) {
      if (u == 0) {
        auto* dst = (__attribute__((address_space(3))) void*)(smem + kLdsB + (kt & 1) * 2048 + (wid >> 2) * 1024 +
                                                              (wid & 3) * 256);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(uniform_rsrc(p.a_mx, live ? numS : 0), dst, 4, voS, kt * p.s_rows * 4, 0, 0);
      }
    }
  };

  // acc[i][jj]: 16 rows (tile i) x columns 32 (jj / 2) + 8 q + 4 (jj % 2) .. of the wave's 128 x 64, row r16 of the tile
  float4v acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) acc[i][jj] = float4v{0.f, 0.f, 0.f, 0.f};

  uint4v a[4][2], b[4][2];
  int sc[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // kMxA: this K tile's scale (block q) of the lane's 8 row fragments
  auto mma = [&](int i0) {
    if constexpr (BF) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[i0 + i][jj] = mfma16(b[jj][s], a[i][s], acc[i0 + i][jj]);
    } else {
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[i0 + i][jj] = mfma8(b[jj][0], b[jj][1], a[i][0], a[i][1], acc[i0 + i][jj], MXA ? sc[i0 + i] : 127);
    }
  };
  auto rdA = [&](const uint8_t* unit) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i][0] = *reinterpret_cast<const uint4v*>(unit + offA + pos + i * 2048);
      a[i][1] = *reinterpret_cast<const uint4v*>(unit + offA + (pos ^ 64) + i * 2048);
    }
  };
  auto rdB = [&](const uint8_t* unit, int j0) {
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      b[j0 + jj][0] = *reinterpret_cast<const uint4v*>(unit + offW + pos + jj * 512);
      b[j0 + jj][1] = *reinterpret_cast<const uint4v*>(unit + offW + (pos ^ 64) + jj * 512);
    }
  };

#define G8_BAR() __builtin_amdgcn_s_barrier()
#define G8_VM(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")
  // rows of this wave row that hold data (wave-uniform): a ragged last tile of an expert (on average half of
  // it) may skip the MFMAs of its empty 64-row blocks — the barriers, LDS reads and DMA stay, so the two wave
  // rows keep their schedule
  const int live = p.skip_empty ? __builtin_amdgcn_readfirstlane(m_end - m_begin - wr * 128) : 256;
#define G8_MFMA(i0)                                  \
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
  G8_BAR();                                          \
  __builtin_amdgcn_s_setprio(1);                     \
  if ((i0) * 16 < live) mma(i0);                     \
  __builtin_amdgcn_s_setprio(0);                     \
  G8_BAR()
  // gemm8p.hip's two phases per K tile: P1 reads B0, B1 and A0 of tile t and stages A1 of t + 1, P2 reads A1 and stages A0
  // (kMxA: and the scales), B0 and B1 of t + 2; a whole K tile is in flight at each wait
  constexpr int kAhead = MXA ? 9 : 8;
  stage(0, 0), stage(2, 0), stage(3, 0), stage(1, 0);
  stage(0, 1), stage(2, 1), stage(3, 1);
  G8_VM(kAhead);
  G8_BAR();
  if (wr == 1) G8_BAR();  // stagger the two wave rows by one barrier
  for (int r = 0; r < KT; ++r) {
    const uint8_t* cb = smem + (r & 1) * kBufB;
    rdB(cb + kUB0, 0);
    rdB(cb + kUB1, 2);
    rdA(cb + kUA0);
    if constexpr (MXA) {
      const uint8_t* st = smem + kLdsB + (r & 1) * 2048 + (wr * 128 + r16) * 4 + q;
#pragma unroll
      for (int i = 0; i < 8; ++i) sc[i] = st[i * 64];
    }
    stage(1, r + 1);
    G8_VM(kAhead);
    G8_MFMA(0);
    rdA(cb + kUA1);
    stage(0, r + 2), stage(2, r + 2), stage(3, r + 2);
    G8_VM(kAhead);
    G8_MFMA(4);
  }
  if (wr == 0) G8_BAR();  // re-align the wave rows
  G8_VM(0);               // the requests past the end have landed before the LDS is given back
#undef G8_MFMA
#undef G8_VM
#undef G8_BAR

  // ---- epilogue: a lane holds eight consecutive columns of a row: scales, SwiGLU and 16 B stores from the registers ----
  const int col0 = n0 + wc * 64 + 8 * q;
  float ws[2][8];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) ws[c][e] = !BF && col0 + 32 * c < p.N ? p.w_scale[(size_t)g * p.N + col0 + 32 * c + e] : 1.f;
  float as[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int m = m_begin + wr * 128 + 16 * i + r16, row = m < m_end ? m : m_begin;
    as[i] = MXA || BF ? 1.f : p.a_scale[p.a_rows ? p.a_rows[row] : row];
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int m = m_begin + wr * 128 + 16 * i + r16;
    float x[2][8];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[c][e] = BF ? acc[i][2 * c + e / 4][e % 4] : acc[i][2 * c + e / 4][e % 4] * (as[i] * ws[c][e]);
    if constexpr (!SWIGLU) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
        if (m < m_end && col0 + 32 * c < p.N) *reinterpret_cast<uint4v*>(p.C + (size_t)m * p.ldc + col0 + 32 * c) = pack8(x[c]);
    } else {  // the wave's first 32 columns are gate, the other 32 the matching up columns
      const int col = n0 / 2 + wc * 32 + 8 * q;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = silu8(x[0][e]) * x[1][e];
      const uint4v packed = pack8(y);
      if constexpr (MODE != kMxOut) {
        if (m < m_end && col < p.N / 2) *reinterpret_cast<uint4v*>(p.C + (size_t)m * p.ldc + col) = packed;
      } else {
        // e4m3 rows with one e8m0 scale per (row, MX block): the wave's 32 outputs of a row are exactly block wc of
        // the workgroup's 128 (= one K slice of the down GEMM), held by four lanes (8 each)
        float v[8];
        unpack8(packed, v);
        float mx = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
        const int e = mx_exp(row_max4(mx));
        const float inv = __builtin_amdgcn_ldexpf(1.f, -e);
        uint32_t lo = 0, hi = 0;
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0] * inv, v[1] * inv, lo, false);
        lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2] * inv, v[3] * inv, lo, true);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4] * inv, v[5] * inv, hi, false);
        hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6] * inv, v[7] * inv, hi, true);
        if (m < m_end && col < p.N / 2) {
          *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(p.C) + (size_t)m * p.ldc + col) = uint2{lo, hi};
          if (q == 0) p.mx_out[((size_t)(n0 / 256) * p.s_rows + m) * 4 + wc] = (uint8_t)(e + 127);
        }
      }
    }
  }
}

}  // namespace g8g
}  // namespace lwc

extern "C" int lwc_gemm2g(const void*, const void*, void*, const int*, const int*, const float*, const float*, int, int, int, int,
                              int, int, int, int, const void*, void*, int, hipStream_t);

// Whether a group's last tile skips the MFMAs of its empty rows.  Where it does it walks K ahead of the tile that shares its weights, and
// where nearly every group has a nearly empty tile beside a full one, its part of the weights comes from memory twice: groups of 300 rows,
// MB fetched skipping / not (and as four phases per K tile, whose barriers held the lead back): bf16 [1536, 2048] x 64 1070 / 864 (905), [4096, 14336]
// x 8 2320 / 2275 (2010).  us, skipping / not (and in four phases), 258 to 340 rows a group, bf16 [4096, 14336] x 8 362 to 369 / 328 to 334 (345 to
// 352), [4096, 7168] x 8 177 to 181 / 167 to 171 (167 to 176), [2048, 2048] x 32 118 to 126 / 110 to 115 (107 to 116), [1536, 2048] x 64 227 to 242 / 216
// to 227 (205 to 220), fp8 [4096, 14336] x 8 180 to 182 / 171 to 174 (170 to 175); the SwiGLU's of short K: [3072, 2048] x 32 198 / 192 (191), [1536,
// 2048] x 64 220 / 207 (200).  But SwiGLU [14336, 4096] x 8 330 / 350, fp8 [28672, 4096] x 8 345 / 361; from 400 rows on level, and for uneven groups of 400 on
// average [4096, 14336] x 8 516 / 542; K 768 112 / 114.
static int skips_empty(long long rows, int G, int K, bool swiglu, bool bf16) {
  return rows <= 256LL * G || rows > 384LL * G || K <= 2048 || (swiglu && !(bf16 && K <= 4096));
}

// Whether the weights bound a grouped fp8 call, and gemm2g.hip takes it: rows per group on average, and cols, its columns of
// 128 in all groups (one workgroup each, two of them a CU: 512 in a round).  The lines were laid when this kernel had four phases per K
// tile; it has become 1 to 16 % faster since, which the figures say (us, here / gemm2g, equal groups), but the lines stand:
// Up to 256 columns every CU has one workgroup or none there, and half as many here: from MX [4096, 14336] x 8 at 128 rows 142
// / 117, 144 rows 143 / 114; [2048, 7168] x 8 at 144 rows 67 / 52.  Above 144 rows an uneven routing needs a second tile.
// More of them without the SwiGLU (short K, or several rounds): [4096, 6400] x 16 (512) at 80 rows 86 / 87 (then 92 / 88), at 112 rows from MX
// 90 / 103; [2048, 1408] x 64 (1024) at 80 rows 57 / 63 (63 / 63), at 144 rows from MX 71 / 98; [4096, 1536] x 128 (4096) at 32 rows
// 229 / 230 (265 / 230), at 64 rows 261 / 283, at 100 rows 300 / 351.  Rows of a multiple of 16 KiB: 128 of them at
// a time meet on fewer memory channels than 256 do: [6144, 16384] x 8 (384) at 32 rows 166 / 166 (177 / 166), with K 14336 or 18432 1.06 (0.89).
// With the SwiGLU (K 2048 to 6144): [28672, 4096] x 8 (1792) at 128 rows 251 / 185, at 176 rows 257 / 225; one round not quite full,
// x 2 (448): at 104 rows 63 / 49, at 176 rows 64 / 64; x 4 (896): at 144 rows 120 / 108, at 176 rows 122 / 130.
static bool weight_bound(long long rows, int G, int N, int K, bool swiglu) {
  const long long cols = (long long)((N + 127) / 128) * G;
  long long most = swiglu ? 176 : 144;
  if (cols > 256) {
    if (swiglu) most = cols <= 512 ? 104 : cols <= 1024 ? 144 : 176;
    else most = K % 16384 == 0 ? 0 : cols < 2048 ? 80 : 40;
  }
  return rows <= most * G;
}
// and the dense calls: up to this many 256 x 256 tiles.  us, here / gemm2g, K 4096: 512 rows x 4096 (32 tiles) 44 / 20, 2048 x
// 4096 (128) 49 / 36, 256 x 28672 SwiGLU to MX (112) 52 / 44, 2048 x 6144 (192) 48 / 58, 512 x 28672 (224) 52 / 76
constexpr long long kSmallTiles = 128;

// Grouped fp8 GEMM in 256 x 256 tiles.  Requires K % 128 == 0, N % 8 == 0, lda / ldc % 16 == 0 (bytes
// / elements: 16-byte rows), rows_a * lda < 2^31 and 256 * K < 2^31 (32-bit buffer offsets); max_slots >=
// sum_g ceil(M_g / 256) (ceil(rows / 256) + G always is).  row_off == null: dense, G = 1, rows [0, rows_c).
// mode: 0 plain, 1 SwiGLU epilogue (bf16 out), 2 SwiGLU epilogue with e4m3 + MX block-scale output (C is
// e4m3 [rows_c, ldc bytes], mx_out [N / 256][s_rows][4]); a_mx != null: A carries MX block scales
// [K / 128][s_rows][4] (mode 0 only; a_scale unused).  core: 0 the kernel that the sizes call for, 2 gemm2g.hip's, 8 this file's.
extern "C" int lwc_gemm8g_fp8(const void* A, const void* W, void* C, const int* row_off, const int* a_rows,
                              const float* a_scale, const float* w_scale, int G, int max_slots, int N, int K, int lda,
                              int ldc, int rows_a, int rows_c, int mode, const void* a_mx, void* mx_out, int s_rows,
                              int core, hipStream_t s) {
  using namespace lwc::g8g;
  if (K % 128 != 0 || K < 128 || N % 8 != 0 || lda % 16 != 0 || ldc % 8 != 0 || G < 1) return -1;
  if ((long long)rows_a * lda >= (1LL << 31) || 256LL * K >= (1LL << 31)) return -1;
  const int swiglu = mode == 1 || mode == 2;
  if (mode < 0 || mode > 2 || !w_scale || (!a_scale && !a_mx)) return -2;
  if (swiglu && N % 64 != 0) return -1;  // whole gate / up block pairs per wave
  if (mode == 2 && (N % 256 != 0 || !mx_out || s_rows < rows_c || ldc % 16 != 0)) return -1;
  if (a_mx && (mode != 0 || a_rows || s_rows < rows_a || (long long)(K / 128) * s_rows * 4 >= (1LL << 31))) return -1;
  if (max_slots <= 0) return 0;
  const bool small = core != 0 ? core == 2 : row_off ? weight_bound(rows_c, G, N, K, swiglu)
                                             : (long long)((rows_c + 255) / 256) * ((N + 255) / 256) <= kSmallTiles;
  if (small && rows_c > 0)
    return lwc_gemm2g(A, W, C, row_off, a_rows, a_scale, w_scale, G, N, K, lda, ldc, rows_a, rows_c, a_mx ? 3 : mode, a_mx, mx_out,
                          s_rows, s);
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)gemm8g_kernel<kPlain>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsB);
    (void)hipFuncSetAttribute((const void*)gemm8g_kernel<kSwiglu>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsB);
    (void)hipFuncSetAttribute((const void*)gemm8g_kernel<kMxOut>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsB);
    (void)hipFuncSetAttribute((const void*)gemm8g_kernel<kMxA>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              kLdsB + kMxLds);
    attr = true;
  }
  const int n_tiles = (N + 255) / 256;
  const char* gv = getenv("LWC_G8G_GN");
  const int nj = (n_tiles + 7) / 8, gn = std::max(1, std::min(gv ? atoi(gv) : kDefaultGn, nj));
  Params p{(const uint8_t*)A, (const uint8_t*)W, (lwc::bf16_t*)C, row_off, a_rows, a_scale, w_scale,
           G, N, K, lda, ldc, rows_a, max_slots, n_tiles, rows_c, gn, row_off ? skips_empty(rows_c, G, K, swiglu, false) : 1,
           (const uint8_t*)a_mx, (uint8_t*)mx_out, s_rows};
  if (const char* sv = getenv("LWC_G8G_SKIP")) p.skip_empty = atoi(sv);
  // dense: 8 XCD ranges of ceil(tiles / 8) grouped tiles; grouped: per XCD, windows of gn n-tiles x
  // max_slots m-slots
  const unsigned grid = row_off ? (unsigned)(((nj + gn - 1) / gn) * gn * max_slots * 8)
                                : (unsigned)(8 * ((n_tiles * max_slots + 7) / 8));
  if (a_mx)
    gemm8g_kernel<kMxA><<<grid, 512, kLdsB + kMxLds, s>>>(p);
  else if (mode == 2)
    gemm8g_kernel<kMxOut><<<grid, 512, kLdsB, s>>>(p);
  else if (mode == 1)
    gemm8g_kernel<kSwiglu><<<grid, 512, kLdsB, s>>>(p);
  else
    gemm8g_kernel<kPlain><<<grid, 512, kLdsB, s>>>(p);
  return (int)hipGetLastError();
}

// Grouped bf16 GEMM on the same schedule: C[r, :] = A[a_rows[r], :] . W_g^T for rows r of group g (a_rows null: A's row
// r), or with swiglu = 1 silu(gate) * up over rows interleaved in blocks of 32, C [rows, N / 2].  Requires K % 64 == 0,
// N % 8 == 0 (SwiGLU: N % 64 == 0), lda % 8 == 0, ldc % 8 == 0, rows_a * lda * 2 < 2^31 and 512 * K < 2^31; max_slots >=
// sum_g ceil(M_g / 256).  core: 2 gemm2g.hip's kernel, 8 this file's.
extern "C" int lwc_gemm8g_bf16(const void* A, const void* W, void* C, const int* row_off, const int* a_rows, int G,
                               int max_slots, int N, int K, int lda, int ldc, int rows_a, int rows_c, int swiglu, int core,
                               hipStream_t s) {
  using namespace lwc::g8g;
  if (!row_off || K % 64 != 0 || K < 64 || N % (swiglu ? 64 : 8) != 0 || lda % 8 != 0 || ldc % 8 != 0 || G < 1) return -1;
  if ((long long)rows_a * lda * 2 >= (1LL << 31) || 512LL * K >= (1LL << 31)) return -1;
  if (max_slots <= 0) return 0;
  if (rows_c > 0 && core == 2)
    return lwc_gemm2g(A, W, C, row_off, a_rows, nullptr, nullptr, G, N, K * 2, lda * 2, ldc, rows_a, rows_c, swiglu ? 5 : 4, nullptr,
                      nullptr, 0, s);
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)gemm8g_kernel<kBf16>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsB);
    (void)hipFuncSetAttribute((const void*)gemm8g_kernel<kBf16Swiglu>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsB);
    attr = true;
  }
  const int n_tiles = (N + 255) / 256, nj = (n_tiles + 7) / 8;
  Params p{(const uint8_t*)A, (const uint8_t*)W, (lwc::bf16_t*)C, row_off, a_rows, nullptr, nullptr,
           G, N, K * 2, lda * 2, ldc, rows_a, max_slots, n_tiles, rows_c, nj, skips_empty(rows_c, G, K * 2, swiglu, true), nullptr, nullptr, 0};
  const unsigned grid = (unsigned)(nj * max_slots * 8);
  if (swiglu)
    gemm8g_kernel<kBf16Swiglu><<<grid, 512, kLdsB, s>>>(p);
  else
    gemm8g_kernel<kBf16><<<grid, 512, kLdsB, s>>>(p);
  return (int)hipGetLastError();
}
