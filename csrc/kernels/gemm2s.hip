// Grouped bf16 GEMM of tens of rows per group (gfx950): the calls of gemm2g.hip with many columns while the weights' read bounds
// them, as one weight stream per CU.
//
// gemm2g's two workgroups a CU start each tile with nothing in flight and read as many bytes of rows (from L2) as of weights; all
// walk K in step, from its start (the next layer's router reads the sums, gemm2g.hip), where weight rows of a stride whose low bits
// are zero lie on few memory channels: 8 experts of 16 rows read [14336, 4096] at 4.7 TB/s.  Here one persistent workgroup of
// eight waves per CU takes tiles of 192 or 64 rows of a group by 256 columns, one after the other of a contiguous share of all
// tiles, and its loads run ahead over the ends of tiles, with up to four steps (64 entries of every row) of weights and two of rows
// in flight.  Rows past the group's end are neither loaded nor multiplied.  LDS layout, operand order and the order of sums are
// gemm2g's: the same bits.
// Measured, gemm2g -> here, us: 8 experts of 16 / 64 rows [14336, 4096] 199 / 206 -> 162 / 175, of 106 to 143 227 -> 192, [28672, 4096] of
// 16 365 -> 355; with as many columns as give a workgroup half a tile, [4096, 7168] 82 -> 104.  Those are calls in a row; in a routed
// decode step of 64 requests, behind other kernels, [14336, 4096] x 8 takes 191 to 203, gemm2g 207 to 214.  fp8 rows, whose walk
// over K may start anywhere, gain nothing: [28672, 4096] of 16 / 128 rows 158 / 201 in gemm2g, 187 / 212 so.
#include <algorithm>

#include "common.h"

namespace lwc {
namespace g2s {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct Params {
  const uint8_t* A;  // [rows_a, lda] (lda, K in bytes)
  const uint8_t* W;  // [G][N, K]
  bf16_t* C;
  const int* row_off;  // [G + 1]
  const int* a_rows;
  int G, N, K, lda, ldc, rows_a;
  int nt;  // weights_pass (common.h), for the groups of one tile
};

LWC_DEVICE float4v mfma16(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
LWC_DEVICE float silu8(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
LWC_DEVICE int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <int CP = 0>
LWC_DEVICE void dma16(const __amdgpu_buffer_rsrc_t& r, uint8_t* dst, uint32_t vo, int so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, vo, so, 0, CP);
}
template <int N>
LWC_DEVICE void wait_rows() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 64 groups beginning with g0, one a lane: its rows and the number of row tiles up to and with it
struct Groups {
  int r0, r1, upto;
};
LWC_DEVICE Groups groups_at(const Params& p, int g0, int tm) {
  const int lane = threadIdx.x & 63, g = g0 + lane;
  Groups t{g < p.G ? p.row_off[g] : 0, g < p.G ? p.row_off[g + 1] : 0, 0};
  t.upto = (t.r1 - t.r0 + tm - 1) / tm;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(t.upto, o, 64);
    t.upto += lane >= o ? up : 0;
  }
  return t;
}

// Tile t: columns n0 .. n1 of group g's weights times its rows begin .. end (slot: which row tile of all groups; once: the group's only one)
struct Tile {
  int slot, g, begin, end, n0, n1;
  bool once;
};
LWC_DEVICE Tile tile_of(const Params& p, const Groups& first, int t, int n_tiles, int tm, int tn) {
  Tile c;
  c.slot = uni(t / n_tiles);
  c.n0 = (t - c.slot * n_tiles) * tn;
  c.n1 = min(p.N, c.n0 + tn);
  Groups gr = first;  // (the first 64 groups stay in registers: a search through memory takes 3 us)
  int slot = c.slot, g0 = 0;
  while (slot >= __builtin_amdgcn_readlane(gr.upto, 63)) {
    slot -= __builtin_amdgcn_readlane(gr.upto, 63);
    g0 += 64;
    gr = groups_at(p, g0, tm);
  }
  const int l = (int)__builtin_ctzll(__ballot(gr.upto > slot)), r0 = __builtin_amdgcn_readlane(gr.r0, l), r1 = __builtin_amdgcn_readlane(gr.r1, l);
  c.g = g0 + l;
  c.begin = uni(r0 + (slot - __builtin_amdgcn_readlane(gr.upto, l) + (r1 - r0 + tm - 1) / tm) * tm);
  c.end = uni(min(r1, c.begin + tm));
  c.once = r1 - r0 <= tm;
  return c;
}

template <bool SWIGLU, int TM, int NW, int NA>
__global__ void __launch_bounds__(512) gemm2s_kernel(const Params p) {
  constexpr int TN = 256, WC = 4, WR = 2, MI = TM / 16 / WR;  // waves across columns (64 each) and rows; 16-row tiles of a wave
  static_assert(MI * WR * 16 == TM && NW >= NA, "whole row tiles a wave");
  constexpr int kW = TN * 128, kA = TM * 128, kAt = NW * kW;  // bytes of a step; LDS: weights, then rows
  constexpr int IW = TN / 64, IA = TM / 64, kStep = IA + IW;  // DMA instructions of a wave and step
  constexpr int kStores = SWIGLU ? MI : 2 * MI;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = uni(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4, wr = wid / WC, wc = wid % WC;
  const int nk = p.K / 128, n_tiles = (p.N + TN - 1) / TN;

  // this workgroup's share of the tiles: row tiles of all groups one after the other, all columns of one before the next.  An
  // XCD's workgroups are neighbours: they share a group's rows in its L2
  const Groups groups = groups_at(p, 0, TM);
  int slots = __builtin_amdgcn_readlane(groups.upto, 63);
  for (int g0 = 64; g0 < p.G; g0 += 64) slots += __builtin_amdgcn_readlane(groups_at(p, g0, TM).upto, 63);
  const int per = gridDim.x >> 3, w = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const long long total = (long long)slots * n_tiles;
  const int first = uni((int)(total * w / (8 * per))), last = uni((int)(total * (w + 1) / (8 * per)));
  if (first >= last) return;

  // DMA: a wave's instruction fills 8 rows; lane l carries row l / 8 and the chunk of it that belongs at position l % 8 (gemm2g)
  uint32_t voA[IA], voW[IW];
#pragma unroll
  for (int i = 0; i < IW; ++i) {
    const int row = (i * 8 + wid) * 8 + (lane >> 3);
    voW[i] = (uint32_t)(row * p.K + (((lane & 7) ^ ((row >> 3 & 3) * 2 + (row >> 1 & 1))) << 4));
  }
  // the weights' and the rows' cursors; behind the last tile the same instructions without a memory request
  int tw = first, kw = nk, atw = 0, num_w = 0;
  bool past = false;  // the weights at hand pass the caches by
  const uint8_t* src_w = p.W;
  auto stage_w = [&] {
    if (kw == nk) {
      kw = 0;
      num_w = 0;
      if (tw < last) {
        const Tile c = tile_of(p, groups, tw++, n_tiles, TM, TN);
        src_w = p.W + ((size_t)c.g * p.N + c.n0) * p.K;
        num_w = (c.n1 - c.n0) * p.K;
        past = p.nt && c.once;
      }
    }
    const __amdgpu_buffer_rsrc_t r = uniform_rsrc(src_w, num_w);
    auto weights = [&](auto cp) {
#pragma unroll
      for (int i = 0; i < IW; ++i) dma16<decltype(cp)::value>(r, smem + atw + (i * 8 + wid) * 1024, voW[i], uni(kw * 128));
    };
    if (past) weights(std::integral_constant<int, kNT>{});
    else weights(std::integral_constant<int, 0>{});
    ++kw;
    atw = atw == (NW - 1) * kW ? 0 : atw + kW;
  };
  int ta = first, ka = nk, ata = 0, slot_a = -1, num_a = 0;
  auto stage_a = [&] {
    if (ka == nk) {
      ka = 0;
      num_a = 0;
      if (ta < last) {
        const Tile c = tile_of(p, groups, ta++, n_tiles, TM, TN);
        num_a = p.rows_a * p.lda;
        if (c.slot != slot_a) {
          slot_a = c.slot;
#pragma unroll
          for (int i = 0; i < IA; ++i) {
            const int row = (i * 8 + wid) * 8 + (lane >> 3), r = c.begin + row;
            voA[i] = r < c.end ? (uint32_t)((p.a_rows ? p.a_rows[r] : r) * p.lda + (((lane & 7) ^ ((row >> 1) & 7)) << 4)) : 0x7fffffffu;
          }
        }
      }
    }
    const __amdgpu_buffer_rsrc_t r = uniform_rsrc(p.A, num_a);
#pragma unroll
    for (int i = 0; i < IA; ++i) dma16(r, smem + kAt + ata * kA + (i * 8 + wid) * 1024, voA[i], uni(ka * 128));
    ++ka;
    ata = ata == NA - 1 ? 0 : ata + 1;
  };

  // operand reads: as in gemm2g; the wave's row tiles are every other one, so that a short group's rows divide between the waves
  const int pos0 = (q ^ (r16 >> 1)) << 4;
  const int offA = kAt + (wr * 16 + r16) * 128, offW = (wc * 64 + 8 * (r16 >> 2) + (r16 & 3)) * 128;

#pragma unroll
  for (int i = 0; i < NW - NA; ++i) stage_w();
#pragma unroll
  for (int i = 0; i < NA; ++i) stage_a(), stage_w();

  int rw = 0, ra = 0, behind = 0;  // LDS places of the step at hand; steps for which a tile's stores are younger than what they need
  for (int t = first; t < last; ++t) {
    const Tile c = tile_of(p, groups, t, n_tiles, TM, TN);
    const int live = wc * 64 < c.n1 - c.n0 ? c.end - c.begin : 0;  // rows that the wave has work for
    float4v acc[MI][2][2];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[i][cc][h] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      // this step's rows and weights have landed: younger than its rows are that step's weights and the later steps
      if (behind > 0) wait_rows<IW + (NA - 1) * kStep + kStores>();
      else wait_rows<IW + (NA - 1) * kStep>();
      --behind;
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      uint4v a[2][MI], wv[2][2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int pos = s ? pos0 ^ 64 : pos0;
#pragma unroll
        for (int i = 0; i < MI; ++i) a[s][i] = *reinterpret_cast<const uint4v*>(smem + ra * kA + offA + pos + i * WR * 2048);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
          for (int h = 0; h < 2; ++h) wv[s][cc][h] = *reinterpret_cast<const uint4v*>(smem + rw + offW + pos + cc * 4096 + h * 512);
      }
      rw = rw == (NW - 1) * kW ? 0 : rw + kW;
      ra = ra == NA - 1 ? 0 : ra + 1;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();  // every wave holds the step's operands: their places take later steps
      asm volatile("" ::: "memory");
      stage_a();
      stage_w();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < MI; ++i)
        if ((WR * i + wr) * 16 < live) {
#pragma unroll
          for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[i][cc][h] = mfma16(wv[1][cc][h], a[1][i], mfma16(wv[0][cc][h], a[0][i], acc[i][cc][h]));
        }
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
    }

    // ---- epilogue from the registers; stores past the group's rows or N fall outside the resource, so that their number, which
    // the waits count, is always the same ----
    const int ncols = SWIGLU ? c.n1 / 2 : c.n1, col0 = SWIGLU ? c.n0 / 2 + wc * 32 : c.n0 + wc * 64;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m0 = c.begin + (WR * i + wr) * 16, rows = c.end - m0;
      const __amdgpu_buffer_rsrc_t rc = uniform_rsrc(p.C + (size_t)m0 * p.ldc + col0, 16 * p.ldc * 2);
      const uint32_t off = (r16 * p.ldc + 8 * q) * 2;
      float x[2][8];
#pragma unroll
      for (int cc = 0; cc < 2; ++cc)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[cc][e] = acc[i][cc][e >> 2][e & 3];
      if constexpr (SWIGLU) {  // the wave's first 32 columns are gate, the other 32 the matching up columns
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = silu8(x[0][e]) * x[1][e];
        __builtin_amdgcn_raw_buffer_store_b128(pack8(y), rc, r16 < rows && col0 + 8 * q < ncols ? off : 0x7ffffff0u, 0, 0);
      } else {
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
          __builtin_amdgcn_raw_buffer_store_b128(pack8(x[cc]), rc, r16 < rows && col0 + 32 * cc + 8 * q < ncols ? off + 64 * cc : 0x7ffffff0u, 0, 0);
      }
    }
    behind = NA;
  }
  wait_rows<0>();  // what was asked for past the last tile has ended before the LDS is given back
}

template <bool SWIGLU, int TM, int NW, int NA>
int launch(const Params& p, hipStream_t s) {
  constexpr int kLds = NW * 256 * 128 + NA * TM * 128;
  static_assert(kLds <= 160 * 1024, "a compute unit's LDS");
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)gemm2s_kernel<SWIGLU, TM, NW, NA>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  (void)attr;
  gemm2s_kernel<SWIGLU, TM, NW, NA><<<256, 512, kLds, s>>>(p);
  return (int)hipGetLastError();
}

}  // namespace g2s
}  // namespace lwc

// The grouped bf16 calls of lwc_gemm2g (K and lda in bytes, checked there), in tiles of 64 or 192 rows.  -1, and nothing
// launched, for sizes that it does not take.
extern "C" int lwc_gemm2s(const void* A, const void* W, void* C, const int* row_off, const int* a_rows, int G, int N, int K, int lda,
                          int ldc, int rows_a, int swiglu, int tm, hipStream_t s) {
  using namespace lwc::g2s;
  // (a cursor is at most four steps ahead; 32-bit offsets in a tile)
  if (!row_off || K % 128 != 0 || K < 4 * 128 || N % (swiglu ? 64 : 8) != 0 || 256LL * K >= (1LL << 31) || 32LL * ldc >= (1LL << 30)) return -1;
  const Params p{(const uint8_t*)A, (const uint8_t*)W, (lwc::bf16_t*)C, row_off, a_rows, G, N, K, lda, ldc, rows_a,
                 lwc::weights_pass((long long)G * N * K)};
  if (swiglu) return tm == 64 ? launch<true, 64, 4, 2>(p, s) : launch<true, 192, 3, 2>(p, s);
  return tm == 64 ? launch<false, 64, 4, 2>(p, s) : launch<false, 192, 3, 2>(p, s);
}
