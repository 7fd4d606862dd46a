// bf16 GEMM of up to 64 rows (gfx950), the weights' read being the bound: gemm2w.hip's 64 x 64 tiles as one weight stream per CU.
//
// gemm2w's tiles cover the columns in whole numbers of 64, two workgroups a CU: 448 tiles leave 64 CUs with half the work of the
// others, a quarter of all loads is the rows' (each tile reads all 64), and what a workgroup does in a step (wait, read
// operands, multiply) hides only behind the other's.  Here a workgroup of eight waves has a CU to itself and an even share of
// the columns, in units of 16, in tiles of at most 8 units; its loads run on over the ends of tiles.  Every wave multiplies a unit
// by all rows, or, in tiles of up to 4 units, by half of them.  A step is 128 entries of K, 256 bytes of every row (with 64: the
// operands' latency per step counts twice, and memory gives 3 % less).  Three steps in LDS are enough (as fast as more, two are not).
// Rows 8 KiB apart lie on few memory channels: each run of columns starts its walk over K at a step of its own (28672 x 4096: 53 us
// without, 43 with; steps of one run and the next 1, 5, 7 or 13 apart instead of 3 lose 5 to 15 % at some sizes).
// Measured, gemm2w -> here (us, 61 rows, weights from memory): 28672 x 4096 SwiGLU 53 -> 43 (5.4 TB/s), 128256 x 4096 207 -> 197, 22016 x
// 4096 47 -> 35, 6144 x 4096 19 -> 15, 10240 x 8192 45 -> 35, 2048 x 2048 11.7 -> 8.4, 3072 x 1024 7.7 -> 6.3; 1465 settings of 1, 24
// and 64 rows 0.90 on average.  What is left: some 4 us of a launch and its first loads, and where K is split 2 to 5 us in which the
// ranges' sums meet.
#include <algorithm>

#include "common.h"
#include "step_fuse.h"

namespace lwc {
namespace g1s {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

enum Epi { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_BIAS = 3, EPI_BIAS_GELU = 4, EPI_ROPE_KV = 5 };

struct Params {
  const bf16_t* A;
  const bf16_t* W;
  bf16_t* C;
  const bf16_t* R;  // EPI_RESIDUAL: residual [M, ldc] (may be C); EPI_BIAS / EPI_BIAS_GELU: bias [N]
  int M, N, K, lda, ldc;
  int runs, splits;  // workgroups across the columns, and K ranges of each
  int share, more;   // blocks (of kGrain units) of a run, and how many runs have one more
  int tiles, wide;   // a run's tiles, and the blocks of each
  float* part;       // splits > 1: [N / 16][splits][1024] partial sums
  int* count;        // splits > 1: [runs * tiles] finished ranges (zero between launches)
  int turned;        // a run's walk over its K range starts at a step of its own, 0 .. turned
  RowSumsq ss;       // NORM: read by EPI_PLAIN, EPI_SWIGLU and EPI_ROPE_KV, written by EPI_RESIDUAL
  RopeKV kv;         // EPI_ROPE_KV
};

LWC_DEVICE float4v mfma(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
LWC_DEVICE float silu(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
LWC_DEVICE int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <int CP = 0>
LWC_DEVICE void dma16(const __amdgpu_buffer_rsrc_t& r, uint8_t* dst, uint32_t vo, int so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, vo, so, 0, CP);
}
LWC_DEVICE void unpack4(const uint2& v, float (&x)[4]) {
  x[0] = __uint_as_float(v.x << 16), x[1] = __uint_as_float(v.x & 0xffff0000u);
  x[2] = __uint_as_float(v.y << 16), x[3] = __uint_as_float(v.y & 0xffff0000u);
}

constexpr int kRows = 64, kA = kRows * 128, kUnit = 16 * 128;  // bytes of 64 entries of all rows, and of a unit's
constexpr int kSide = 8 * kRows * 4 + 16;                      // sums that waves exchange, and a flag

// UW: the most units of a tile, 8, or 4: two waves share one, each with half of the rows.  NST steps of 128 entries in LDS.
// NT: the weights pass the caches by (weights_pass, common.h).
template <int EPI, bool NORM, int UW, int NST, bool NT>
__global__ void __launch_bounds__(512, 2) gemm1s_kernel(const Params p) {
  constexpr bool kPairs = EPI == EPI_SWIGLU || EPI == EPI_ROPE_KV;  // a unit is 8 columns and the 8 that meet them
  constexpr bool kScale = NORM && EPI != EPI_RESIDUAL, kSums = NORM && EPI == EPI_RESIDUAL;
  constexpr int kGrain = kSums ? 2 : 1;  // units that stay together: 32 columns of a row make one partial sum of squares
  constexpr int WPU = 8 / UW, MI = 4 / WPU, IW = 2 / WPU;  // waves of a unit, their 16-row tiles and their DMA instructions of it
  constexpr int kLoads = 2 * (1 + IW), kStage = 2 * (kA + UW * kUnit);
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float* side = reinterpret_cast<float*>(smem + NST * kStage);
  int* flag = reinterpret_cast<int*>(side + 8 * kRows);
  const int tid = threadIdx.x, lane = tid & 63, wid = uni(tid >> 6), mu = wid / WPU, mr = wid % WPU, r16 = lane & 15, q = lane >> 4;
  const int row0 = 16 * mr * MI + r16;  // the lane's first row

  // (the ranges of a tile are neighbours: they run on one XCD)
  const int i0 = xcd_remap(blockIdx.x, p.runs * p.splits), run = uni(i0 / p.splits), split = i0 - run * p.splits;
  const int b0 = run * p.share + min(run, p.more), b1 = b0 + p.share + (run < p.more ? 1 : 0), tiles = p.tiles;
  const int KT = p.K / 128, k0 = uni(KT * split / p.splits), nk = uni(KT * (split + 1) / p.splits) - k0;
  const int first_k = k0 * 256, past_k = first_k + nk * 256, turn = (run * 3 & p.turned) * 256;

  // DMA: a wave's instruction fills 8 rows of 128 bytes; chunk c of row r lies at c ^ (r / 2 % 8), so that the 16-lane groups in
  // which an operand read is served meet every bank once
  uint32_t voA, voW[IW];
  {
    const int row = wid * 8 + (lane >> 3);
    voA = row < p.M ? (uint32_t)(row * p.lda * 2 + (((lane & 7) ^ ((row >> 1) & 7)) << 4)) : 0x7fffffffu;
  }
  const int far = EPI == EPI_SWIGLU ? 32 : EPI == EPI_ROPE_KV ? p.kv.D / 2 : 0;
#pragma unroll
  for (int j = 0; j < IW; ++j) {
    const int row = (j + mr) * 8 + (lane >> 3);  // of pairs, a lane group's four: two columns and the two that meet them
    const int at = kPairs ? (row >> 2) * 2 + (row & 1) + (row & 2 ? far : 0) : row;
    voW[j] = (uint32_t)(at * p.K * 2 + (((lane & 7) ^ ((row >> 1) & 7)) << 4));
  }
  const __amdgpu_buffer_rsrc_t rA = uniform_rsrc(p.A, ((p.M - 1) * p.lda + p.K) * 2);
  auto tile_unit = [&](int c) { return (b0 + c * p.wide) * kGrain + mu; };
  auto tile_end = [&](int c) { return min(b0 + (c + 1) * p.wide, b1) * kGrain; };
  auto unit_row = [&](int u) {  // the first W row of a unit
    if (EPI == EPI_SWIGLU) return (u >> 2) * 64 + (u & 3) * 8;
    if (EPI == EPI_ROPE_KV) return u / (p.kv.D / 16) * p.kv.D + u % (p.kv.D / 16) * 8;
    return u * 16;
  };
  // the loads' cursor: tile, steps left in it, byte of K.  Past the last tile nothing is read, and the count of loads stays.
  int load_tile = 0, load_left = nk, load_k = first_k + turn;
  __amdgpu_buffer_rsrc_t rX = rA, rW;
  auto load_unit = [&]() {
    const int u = tile_unit(load_tile);
    const bool there = load_tile < tiles && u < tile_end(load_tile);
    rW = uniform_rsrc(p.W + (size_t)(there ? unit_row(u) : 0) * p.K, there ? (kPairs ? far + 8 : 16) * p.K * 2 : 0);
  };
  load_unit();
  auto stage = [&](int buf) {
    uint8_t* b = smem + buf * kStage;
#pragma unroll
    for (int s = 0; s < 2; ++s) dma16(rX, b + s * kA + wid * 1024, voA, load_k + s * 128);
#pragma unroll
    for (int j = 0; j < IW; ++j)
#pragma unroll
      for (int s = 0; s < 2; ++s) dma16<NT ? kNT : 0>(rW, b + 2 * kA + s * UW * kUnit + mu * kUnit + (j + mr) * 1024, voW[j], load_k + s * 128);
    load_k += 256;
    load_k = load_k == past_k ? first_k : load_k;
    if (--load_left == 0) {
      ++load_tile;
      load_left = nk;
      load_k = first_k + turn;
      if (load_tile >= tiles) rX = uniform_rsrc(p.A, 0);
      load_unit();
    }
  };
  const int pos0 = (q ^ (r16 >> 1)) << 4, pos1 = pos0 ^ 64;
  const int offA = row0 * 128, offW = 2 * kA + mu * kUnit + r16 * 128;

  // What the epilogue reads goes out ahead of the first K steps: the rows' partial sums of squares, each wave eight rows, 16
  // lanes per row; the rows' slots and positions (the angles follow the first steps)
  float4v ssv[2][4];
  float sumsq[2];
  if constexpr (kScale) {
    const __amdgpu_buffer_rsrc_t rS = uniform_rsrc(p.ss.ss, p.M * p.ss.P * 4);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        ssv[i][c] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
            rS, 64 * c + 4 * r16 < p.ss.P ? ((wid * 8 + 4 * i + q) * p.ss.P + 64 * c + 4 * r16) * 4 : 0x7fffffff, 0, 0));
  }
  RopeAhead<2> ahead[EPI == EPI_ROPE_KV ? MI : 1];
  int head = 0, head_col = 0;
  if constexpr (EPI == EPI_ROPE_KV) {  // (one tile)
    head = uni(tile_unit(0) / (p.kv.D / 16));
    head_col = uni(tile_unit(0) % (p.kv.D / 16)) * 8 + 2 * q;
#pragma unroll
    for (int i = 0; i < MI; ++i) rope_kv_row(p.kv, ahead[i], min(row0 + 16 * i, p.M - 1), head);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < NST - 1; ++k) stage(k);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (EPI == EPI_ROPE_KV) {
#pragma unroll
    for (int i = 0; i < MI; ++i) rope_kv_angles(p.kv, ahead[i], head, head_col);
  }
  if constexpr (kScale) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float t = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) t += (ssv[i][c][0] + ssv[i][c][1]) + (ssv[i][c][2] + ssv[i][c][3]);
      sumsq[i] = row16_sum(t);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  float scale[MI];

  int buf = 0, put = NST - 1;
  for (int c = 0; c < tiles; ++c) {
    float4v acc[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[i] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int kt = 0; kt < nk; ++kt) {
      // this step's rows have landed, the following steps' may be in flight; every wave is past its reads of the step before
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NST - 2) * kLoads) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      stage(put);
      put = put == NST - 1 ? 0 : put + 1;
      const uint8_t* b = smem + buf * kStage;
      buf = buf == NST - 1 ? 0 : buf + 1;
      uint4v a[4][MI], w[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int pos = s & 1 ? pos1 : pos0;
        w[s] = *reinterpret_cast<const uint4v*>(b + offW + (s >> 1) * UW * kUnit + pos);
#pragma unroll
        for (int i = 0; i < MI; ++i) a[s][i] = *reinterpret_cast<const uint4v*>(b + offA + (s >> 1) * kA + pos + i * 2048);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[i] = mfma(w[s], a[s][i], acc[i]);
    }
    const int u = tile_unit(c);
    const bool mine = u < tile_end(c);
    if constexpr (kScale) {
      if (c == 0 && r16 == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) side[wid * 8 + 4 * i + q] = sumsq[i];
      }
    }
    if (p.splits > 1) {  // the last range to arrive adds all of them up, in their order, and writes the output
      // (device scope, past the caches: the ranges of a tile may run on several XCDs)
      const __amdgpu_buffer_rsrc_t rP = uniform_rsrc(p.part + (size_t)(mine ? u : 0) * p.splits * 1024, mine ? p.splits * 4096 : 0);
      const int at = mr * MI * 1024 + lane * 16;
#pragma unroll
      for (int i = 0; i < MI; ++i) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, acc[i]), rP, at + i * 1024, split * 4096, 16);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // they have arrived
      __syncthreads();
      if (tid == 0) {
        int* count = p.count + run * tiles + c;
        const int n = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (n == p.splits - 1) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = n;
      }
      __syncthreads();
      if (uni(*flag) != p.splits - 1) break;  // (of split ranges, a run has one tile)
      float4v x[8][MI];
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)  // (past the last range: zeros, and no load)
          x[j][i] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(rP, at + i * 1024, j * 4096, 16));
#pragma unroll
      for (int i = 0; i < MI; ++i) acc[i] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[i] += x[j][i];
    } else if (kScale && c == 0) {
      __syncthreads();
    }
    if constexpr (kScale) {
      if (c == 0) {
#pragma unroll
        for (int i = 0; i < MI; ++i) scale[i] = rsqrtf(side[row0 + 16 * i] / p.K + p.ss.eps);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) acc[i] *= scale[i];
    }
    if constexpr (EPI == EPI_ROPE_KV) {
      if (mine) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const float x[2] = {acc[i][0], acc[i][1]}, y[2] = {acc[i][2], acc[i][3]};
          if (row0 + 16 * i < p.M) rope_kv_store<2>(p.kv, ahead[i], p.C, p.ldc, row0 + 16 * i, head, head_col, x, y);
        }
      }
    } else if constexpr (EPI == EPI_SWIGLU) {
      if (mine) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
          if (row0 + 16 * i < p.M)
            *reinterpret_cast<uint32_t*>(p.C + (size_t)(row0 + 16 * i) * p.ldc + u * 8 + 2 * q) =
                pack_bf16x2(silu(acc[i][0]) * acc[i][2], silu(acc[i][1]) * acc[i][3]);
      }
    } else {
      float t2[MI];
      if (mine) {
        const int col = u * 16 + 4 * q;
        float b[4];
        if (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) unpack4(*reinterpret_cast<const uint2*>(p.R + col), b);
        uint2 rv[MI];
        if (EPI == EPI_RESIDUAL) {
#pragma unroll
          for (int i = 0; i < MI; ++i) rv[i] = *reinterpret_cast<const uint2*>(p.R + (size_t)min(row0 + 16 * i, p.M - 1) * p.ldc + col);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          if (EPI == EPI_RESIDUAL) unpack4(rv[i], b);
          float x[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = acc[i][e];
            if (EPI != EPI_PLAIN) x[e] += b[e];
            if (EPI == EPI_BIAS_GELU) x[e] = gelu_erf(x[e]);
          }
          const uint2 o = {pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
          if (row0 + 16 * i < p.M) *reinterpret_cast<uint2*>(p.C + (size_t)(row0 + 16 * i) * p.ldc + col) = o;
          if constexpr (kSums) {  // of the row as stored
            unpack4(o, x);
            t2[i] = row_sum4((x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]));
          }
        }
      }
      if constexpr (kSums) {  // one partial per 32 columns: a unit and the next
        if (mine && (mu & 1) && q == 0) {
#pragma unroll
          for (int i = 0; i < MI; ++i) side[mu * kRows + row0 + 16 * i] = t2[i];
        }
        __syncthreads();
        if (mine && !(mu & 1) && q == 0) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
            if (row0 + 16 * i < p.M) p.ss.ss[(size_t)(row0 + 16 * i) * p.ss.P + u / 2] = t2[i] + side[(mu + 1) * kRows + row0 + 16 * i];
        }
        __syncthreads();
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the loads past the end write zeros to LDS)
}

template <int EPI, bool NORM, int UW, int NST, bool NT>
int go(const Params& p, hipStream_t s) {
  constexpr int kLds = NST * 2 * (kA + UW * kUnit) + kSide;
  static_assert(kLds <= 160 * 1024, "LDS of a CU");
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)gemm1s_kernel<EPI, NORM, UW, NST, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  (void)attr;
  gemm1s_kernel<EPI, NORM, UW, NST, NT><<<p.runs * p.splits, 512, kLds, s>>>(p);
  return (int)hipGetLastError();
}

// (Kernels of their own for NT: where a branch in the K loop chose, the compiler took each step for fewer loads than it has and waited for
// later ones too early.  us, chosen so / now: residual 64 x 3072 x 4096 16.7 / 15.4, 33 x 8192 x 1024 12.8 / 10.9, 64 x 3072 x 768 10.4 / 9.3.)
template <int EPI, bool NORM>
int launch(const Params& p, hipStream_t s) {
  const bool narrow = p.wide * (NORM && EPI == EPI_RESIDUAL ? 2 : 1) <= 4;
  if (weights_pass(2LL * p.N * p.K)) return narrow ? go<EPI, NORM, 4, 4, true>(p, s) : go<EPI, NORM, 8, 3, true>(p, s);
  return narrow ? go<EPI, NORM, 4, 4, false>(p, s) : go<EPI, NORM, 8, 3, false>(p, s);
}

// How the columns go over the CUs with K in so many ranges: as evenly as units allow (runs of a whole 64 columns each would start at rows
// that meet on the memory channels: 14336 x 4096 in 224 runs 27 us, in 256 24; 32000 x 4096 in 250 51, in 256 48)
struct Cut {
  int runs, tiles, wide, units;  // units: of the widest tile
};
inline Cut cut(int N, int splits, int grain) {
  const int blocks = N / (16 * grain);
  Cut c;
  c.runs = std::min(256 / splits, splits > 1 ? (N + 63) / 64 : blocks);  // (of split ranges as many as 64 columns each make: the workspace)
  const int widest = (blocks + c.runs - 1) / c.runs;
  c.tiles = (widest * grain + 7) / 8;
  c.wide = (widest + c.tiles - 1) / c.tiles;
  c.units = c.wide * grain;
  return c;
}

}  // namespace g1s
}  // namespace lwc

// Whether a call of lwc_gemm2w runs here, and in how many K ranges (max_splits: its workspace in 64 x 64 partial tiles; a unit of a
// range takes a quarter of one).  A plain product without the folded norm does not: its walk over K starts at its beginning (a router
// may stand behind it, gemm2g.hip), where the streams gain nothing (32000 x 4096 57 us either way).
// The ranges: fitted to 420 settings (us, 61 and 32 rows, K 1024 to 14336, N 1024 to 128256).  A step of 128 entries takes a CU 0.4 us
// and 0.035 more per unit, memory gives 5.9 TB/s, a ninth less where a quarter of the CUs has no workgroup, and the ranges'
// sums meet in 2.6 to 5.2: 4096 x 4096 in 1 / 2 / 4 / 8 16.5 / 14.9 / 12.0 / 14.1, 1024 x 8192 26.8 / 17.8 / 12.5 / 10.5, 10240 x
// 11008 54.7 / 48.0.  Against gemm2w the best of them is 0.72 to 1.04, 0.87 on average.
extern "C" int lwc_gemm1s_plan(int M, int N, int K, int epi, bool norm, long long max_splits) {
  using namespace lwc::g1s;
  if (M < 1 || M > kRows || N % 16 != 0 || K % 128 != 0 || (epi == EPI_PLAIN && !norm) || (epi == EPI_SWIGLU && N % 64 != 0)) return 0;
  const int grain = norm && epi == EPI_RESIDUAL ? 2 : 1, KT = K / 128;
  if (N % (16 * grain) != 0) return 0;
  // gemm2w's tiles in its K ranges where they give nearly every CU one workgroup: level or ahead from K 8192 on, up to 1024 and in three
  // ranges (24 or 32 rows, us, there / here: 4096 x 8192 17.3 / 18.6, 4096 x 14336 26.0 / 26.0, 8192 x 8192 27.3 / 29.1, 14336 x 8192 42.6 /
  // 46.7, 14336 x 1024 8.8 / 9.4, 5120 x 5120 15.6 / 17.3), else behind (4096 x 4096 12.3 / 11.9, 8192 x 4096 18.3 / 17.1, 14336 x 4096 25.4 / 24.4)
  const long long tiles = (N + 63) / 64, ranges = std::max(1LL, std::min(std::min(256 / tiles, (long long)K / 1024), max_splits / tiles));
  if ((K >= 8192 || K <= 1024 || ranges == 3) && tiles * ranges >= 224 && tiles * ranges <= 256) return 0;
  int best = 0;
  double least = 0;
  for (int s : {1, 2, 4, 8}) {
    const Cut c = cut(N, s, grain);
    if (s > 1 && (KT < 4 * s || c.tiles > 1 || (long long)(N + 63) / 64 * s > max_splits)) break;
    if (epi == EPI_ROPE_KV && c.tiles > 1) continue;
    const double step = c.tiles * ((KT + s - 1) / s) * (0.4 + 0.035 * c.units);
    const double mem = 2.0 * N * K / 5.9e6 * (1 + std::max(0, 256 - c.runs * s) / 512.0);
    const double us = std::max(step, mem) + (s == 1 ? 0 : s == 2 ? 2.6 : s == 4 ? 3.4 : 5.2);
    if (best == 0 || us < least) best = s, least = us;
  }
  return best;
}

// The operands of lwc_gemm2w (checked there) where lwc_gemm1s_plan takes them.
extern "C" int lwc_gemm1s(const void* A, const void* W, void* C, const void* R, int M, int N, int K, int lda, int ldc, int epi,
                          int splits, float* part, int* count, const lwc::RowSumsq* ss, const lwc::RopeKV* kv, hipStream_t s) {
  using namespace lwc::g1s;
  const int grain = ss != nullptr && epi == EPI_RESIDUAL ? 2 : 1;
  if (M < 1 || M > kRows || N % (16 * grain) != 0 || K % 128 != 0 || splits < 1 || splits > 8 || K / 128 < splits) return -1;
  if (splits > 1 && (part == nullptr || count == nullptr)) return -1;
  const Cut c = cut(N, splits, grain);
  if (c.tiles > 1 && (splits > 1 || epi == EPI_ROPE_KV)) return -1;
  int turned = 0;  // (a power of two less one)
  while (2 * turned + 2 <= K / 128 / splits) turned = 2 * turned + 1;
  const int blocks = N / (16 * grain);
  const Params p{(const lwc::bf16_t*)A, (const lwc::bf16_t*)W, (lwc::bf16_t*)C, (const lwc::bf16_t*)R, M, N, K, lda, ldc, c.runs, splits,
                 blocks / c.runs, blocks % c.runs, c.tiles, c.wide, part, count, turned, ss != nullptr ? *ss : lwc::RowSumsq{},
                 kv != nullptr ? *kv : lwc::RopeKV{}};
  if (ss != nullptr) {
    switch (epi) {
      case EPI_PLAIN: return launch<EPI_PLAIN, true>(p, s);
      case EPI_RESIDUAL: return launch<EPI_RESIDUAL, true>(p, s);
      case EPI_SWIGLU: return launch<EPI_SWIGLU, true>(p, s);
      case EPI_ROPE_KV: return launch<EPI_ROPE_KV, true>(p, s);
    }
    return -1;
  }
  switch (epi) {
    case EPI_RESIDUAL: return launch<EPI_RESIDUAL, false>(p, s);
    case EPI_SWIGLU: return launch<EPI_SWIGLU, false>(p, s);
    case EPI_BIAS: return launch<EPI_BIAS, false>(p, s);
    case EPI_BIAS_GELU: return launch<EPI_BIAS_GELU, false>(p, s);
  }
  return -1;
}
