// bf16 GEMM in tiles for two independent workgroups per CU (gfx950): C = A W^T with the epilogues of gemm8p.
//
// gemm8p's persistent 256 x 256 tiles leave CUs idle below some 8000 rows, hand partial tiles over through memory, and no
// other work covers a tile's prologue and epilogue.  Here a workgroup is four waves with a tile of 64 to 192 rows or columns,
// at most 80 KiB of LDS and 256 registers, so that two share a CU: one's MFMAs run while the other waits for its first rows,
// reads operands or stores.  Rows arrive by LDS-DMA, 64 entries (a whole 128-byte line: with 32 the rate halves) at a time;
// accumulators hold eight consecutive columns of a row, so the epilogue needs no LDS.
// What bounds it: the rate at which rows reach LDS (12 to 15 TB/s over the chip), so the larger tiles at many rows, where it
// stays behind the library's 256 x 256; below, the time of a K step on a CU that has one workgroup (0.33 us), which the K
// ranges of few tiles shorten.
// Measured against gemm8p and the library (us): 1000 rows x 4096 x K 1024, bias + GELU: 43 and 22 -> 16; 3600 x 1024 x 1024: 46 and
// 20 -> 8 to 16; 7155 x 1024 x 1024: 40 and 24 -> 21; 61 x 4096 x 4096 (weights from memory): skinny 20, library 18 -> 13;
// 61 x 28672 x 4096 SwiGLU 61 (library) -> 51; 61 x 4096 x 14336 39 (library) -> 28; 65536 x 4096 x 1024: 641 and 515, here 634.
#include <algorithm>

#include "common.h"
#include "step_fuse.h"

namespace lwc {
namespace g2w {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

enum Epi { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_BIAS = 3, EPI_BIAS_GELU = 4, EPI_ROPE_KV = 5 };

struct Params {
  const bf16_t* A;
  const bf16_t* W;
  bf16_t* C;
  const bf16_t* R;  // EPI_RESIDUAL: residual [M, ldc] (may be C); EPI_BIAS / EPI_BIAS_GELU: bias [N]
  int M, N, K, lda, ldc;
  int tiles_m, tiles_n;
  int splits;   // K ranges per tile
  float* part;  // splits > 1: [tiles][splits][TM * TN] partial tiles
  int* count;   // [tiles] finished ranges (zero between launches)
  int turned;   // > 0: a tile's walk over its K range starts at a step of its own, 0 .. turned
};

// Arguments of the builds with the folded norm alone: the others neither take nor load them
struct NormParams : Params {
  RowSumsq ss;  // read by EPI_PLAIN, EPI_SWIGLU and EPI_ROPE_KV, written by EPI_RESIDUAL
  RopeKV kv;    // EPI_ROPE_KV
};
template <bool NORM>
struct ArgsOf { using type = Params; };
template <>
struct ArgsOf<true> { using type = NormParams; };

LWC_DEVICE float4v mfma(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
LWC_DEVICE float silu(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

template <int CP = 0>
LWC_DEVICE void dma16(const __amdgpu_buffer_rsrc_t& r, uint8_t* dst, uint32_t vo, int so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, vo, so, 0, CP);
}

// every outstanding load but the last N, and all LDS reads
template <int N>
LWC_DEVICE void wait_rows() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

constexpr int kGroupM = 8;

// EPI_ROPE_KV (64 x 64 tiles, step_fuse.h): a tile takes 32 columns of a head and the 32 that rotate with them, D / 2 further.
// NORM (64 x 64 tiles): the folded RMSNorm of step_fuse.h.  NT: the weights pass the caches by (past_caches).
template <int EPI, int TM, int TN, int NST, bool NORM, bool NT>
__global__ void __launch_bounds__(256, 2) gemm2w_kernel(const typename ArgsOf<NORM>::type p) {
  static_assert((!NORM && EPI != EPI_ROPE_KV) || (TM == 64 && TN == 64), "one row of partial sums per lane group");
  constexpr bool kPairs = EPI == EPI_SWIGLU || EPI == EPI_ROPE_KV;  // columns that meet in a lane: groups of 32, two by two
  constexpr int WC = kPairs && TN == 64 ? 1 : 2, WR = 4 / WC;  // waves across the tile's columns and rows
  constexpr int kA = TM * 128, kStage = kA + TN * 128;  // bytes of a 64-deep K step: A rows, then W rows, 128 bytes each
  constexpr int IA = TM / 32, IW = TN / 32;             // DMA instructions per wave and step
  constexpr int MI = TM / WR / 16, NP = TN / WC / 32;   // the wave's 16-row tiles and its groups of 32 columns
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4, wr = wid / WC, wc = wid % WC;

  // (the ranges of a tile are neighbours: they run on one XCD, and their partial sums meet in its L2)
  const int u = xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n * p.splits), t = u / p.splits, split = u % p.splits;
  const int first_m = t / (kGroupM * p.tiles_n) * kGroupM, gsz = min(p.tiles_m - first_m, kGroupM);
  const int in = t % (kGroupM * p.tiles_n);
  const int m0 = (first_m + in % gsz) * TM;
  int n0 = in / gsz * TN, far = 0;  // far: W rows between the tile's two halves beyond those of a contiguous tile
  if constexpr (EPI == EPI_ROPE_KV) {
    const int strips = p.kv.D / 64, h = in / gsz / strips;
    n0 = h * p.kv.D + in / gsz % strips * 32;
    far = p.kv.D / 2 - 32;
  }

  // DMA: a wave's instruction fills 8 rows; lane l carries row l / 8 and the chunk of it that belongs at position l % 8:
  // chunk c of A row r lies at c ^ (r / 2 % 8), of W row r at c ^ (r / 8 % 4 * 2 + r / 2 % 2), so that the 16-lane groups
  // in which an operand read is served meet every bank once
  const int rows_m = min(p.M - m0, TM), rows_n = EPI == EPI_ROPE_KV ? TN : min(p.N - n0, TN);
  const __amdgpu_buffer_rsrc_t rA = uniform_rsrc(p.A + (size_t)m0 * p.lda, ((rows_m - 1) * p.lda + p.K) * 2);
  const __amdgpu_buffer_rsrc_t rW = uniform_rsrc(p.W + (size_t)n0 * p.K, (rows_n + far) * p.K * 2);
  uint32_t voA[IA], voW[IW];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int row = (i * 4 + wid) * 8 + (lane >> 3);
    voA[i] = row < rows_m ? (uint32_t)(row * p.lda * 2 + (((lane & 7) ^ ((row >> 1) & 7)) << 4)) : 0x7fffffffu;
  }
#pragma unroll
  for (int i = 0; i < IW; ++i) {
    const int row = (i * 4 + wid) * 8 + (lane >> 3);
    voW[i] = row < rows_n ? (uint32_t)((row + (EPI == EPI_ROPE_KV && row >= 32 ? far : 0)) * p.K * 2 + (((lane & 7) ^ ((row >> 3 & 3) * 2 + (row >> 1 & 1))) << 4)) : 0x7fffffffu;
  }
  const int KT = p.K / 64, k0 = KT * split / p.splits, nk = KT * (split + 1) / p.splits - k0;
  // (the steps are asked for in order: the byte of K that the next one begins at)
  const int first_k = k0 * 128, past_k = first_k + nk * 128;
  int next_k = first_k + (in / gsz * 3 & p.turned) * 128;
  auto stage = [&](uint8_t* buf) {
#pragma unroll
    for (int i = 0; i < IA; ++i) dma16(rA, buf + (i * 4 + wid) * 1024, voA[i], next_k);
#pragma unroll
    for (int i = 0; i < IW; ++i) dma16<NT ? kNT : 0>(rW, buf + kA + (i * 4 + wid) * 1024, voW[i], next_k);
    next_k += 128;
    next_k = next_k == past_k ? first_k : next_k;
  };
  // operand reads: A tile i holds rows 16 i + r16; W tile (g, h) holds rows 32 g + 8 (r16 / 4) + 4 h + r16 % 4, so that a
  // lane's accumulators of the pair h = 0, 1 are the eight consecutive columns 32 g + 8 q .. of output row r16
  const int pos0 = (q ^ (r16 >> 1)) << 4, pos1 = pos0 ^ 64;
  const int offA = (wr * (TM / WR) + r16) * 128;
  const int offW = kA + (wc * (TN / WC) + 8 * (r16 >> 2) + (r16 & 3)) * 128;

  float4v acc[MI][NP][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int g = 0; g < NP; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[i][g][h] = float4v{0.f, 0.f, 0.f, 0.f};

  // The rows' partial sums of squares go out ahead of the first K steps and are added up while those are on their way, each
  // wave its own rows: 16 lanes per row, four rows at a time.  (In registers: a store to LDS waits for every row on its way
  // there, 1.6 us.)  So do a row's slot and position; the angles follow the first K steps.
  constexpr bool kScale = NORM && EPI != EPI_RESIDUAL;
  float4v ssv[kScale ? 4 * MI : 1][4];
  float sumsq[kScale ? 4 * MI : 1];
  if constexpr (kScale) {
    const __amdgpu_buffer_rsrc_t rS = uniform_rsrc(p.ss.ss + (size_t)m0 * p.ss.P, rows_m * p.ss.P * 4);
#pragma unroll
    for (int i = 0; i < 4 * MI; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        ssv[i][c] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
            rS, 64 * c + 4 * r16 < p.ss.P ? ((wr * (TM / WR) + 4 * i + q) * p.ss.P + 64 * c + 4 * r16) * 4 : 0x7fffffff, 0, 0));
  }
  RopeAhead<8> ahead;
  if constexpr (EPI == EPI_ROPE_KV) rope_kv_row(p.kv, ahead, min(m0 + wr * 16 + r16, p.M - 1), n0 / p.kv.D);
  if constexpr (NORM) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < NST; ++k)  // (NORM: steps past the range too, rows that nothing reads: behind a branch the sums would wait for all)
    if (NORM || k < nk) stage(smem + k * kStage);
  if constexpr (NORM) __builtin_amdgcn_sched_barrier(0);
  if constexpr (EPI == EPI_ROPE_KV) rope_kv_angles(p.kv, ahead, n0 / p.kv.D, n0 % p.kv.D + 8 * q);
  if constexpr (kScale) {
#pragma unroll
    for (int i = 0; i < 4 * MI; ++i) {
      float t = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) t += (ssv[i][c][0] + ssv[i][c][1]) + (ssv[i][c][2] + ssv[i][c][3]);
      sumsq[i] = row16_sum(t);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  int at = 0;
  for (int kt = 0; kt < nk; ++kt) {
    uint8_t* buf = smem + at;
    at = at == (NST - 1) * kStage ? 0 : at + kStage;
    // this step's rows have landed, the following steps' may be in flight
    if (kt + NST <= nk) wait_rows<(NST - 1) * (IA + IW)>();
    else if (NST > 2 && kt + 3 <= nk) wait_rows<2 * (IA + IW)>();
    else if (kt + 2 <= nk) wait_rows<IA + IW>();
    else wait_rows<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    uint4v a[2][MI], w[2][NP][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int pos = s ? pos1 : pos0;
#pragma unroll
      for (int i = 0; i < MI; ++i) a[s][i] = *reinterpret_cast<const uint4v*>(buf + offA + pos + i * 2048);
#pragma unroll
      for (int g = 0; g < NP; ++g)
#pragma unroll
        for (int h = 0; h < 2; ++h) w[s][g][h] = *reinterpret_cast<const uint4v*>(buf + offW + pos + g * 4096 + h * 512);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave holds the step's operands: its buffer takes the step after next
    asm volatile("" ::: "memory");
    if (kt + NST < nk) stage(buf);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int g = 0; g < NP; ++g)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < MI; ++i) acc[i][g][h] = mfma(w[s][g][h], a[s][i], acc[i][g][h]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
  }

  if constexpr (TM == 64)
  if (p.splits > 1) {  // the last range to arrive adds all of them up, in their order, and writes the output
    // (partial sums pass the caches by stores and loads of device scope: a fence per workgroup writes the whole L2 back and
    // took 10 us and more)
    constexpr int kAcc = MI * NP * 8;  // accumulators per lane
    float* mine = p.part + ((size_t)t * p.splits + split) * (TM * TN) + tid;
#pragma unroll
    for (int e = 0; e < kAcc; ++e)
      __hip_atomic_store(mine + e * 256, acc[e / (NP * 8)][e / 8 % NP][e / 4 % 2][e % 4], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // they have arrived
    __syncthreads();
    int* flag = reinterpret_cast<int*>(smem);
    if (tid == 0) {
      const int n = __hip_atomic_fetch_add(p.count + t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (n == p.splits - 1) __hip_atomic_store(p.count + t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = n;
    }
    __syncthreads();
    if (*flag != p.splits - 1) return;
    float sum[kAcc];
#pragma unroll
    for (int e = 0; e < kAcc; ++e) sum[e] = 0.f;
    // (four ranges on their way at once: 61 x 4096 x 4096 in four 12.8 -> 12.1 us)
    for (int s = 0; s < p.splits; s += 4) {
      float x[4][kAcc];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float* part = p.part + ((size_t)t * p.splits + min(s + j, p.splits - 1)) * (TM * TN) + tid;
#pragma unroll
        for (int e = 0; e < kAcc; ++e) x[j][e] = __hip_atomic_load(part + e * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < kAcc; ++e) sum[e] += s + j < p.splits ? x[j][e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < kAcc; ++e) acc[e / (NP * 8)][e / 8 % NP][e / 4 % 2][e % 4] = sum[e];
  }

  const int mrow = m0 + wr * (TM / WR) + r16;
  if constexpr (kScale) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      float t = 0.f;  // row r16 = 4 j + q' was added up by lane group q' of the j-th four
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float u = __shfl(sumsq[4 * i + j], 16 * (r16 & 3), 64);
        t = r16 >> 2 == j ? u : t;
      }
      const float f = rsqrtf(t / p.K + p.ss.eps);
#pragma unroll
      for (int g = 0; g < NP; ++g)
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[i][g][h] *= f;
    }
  }
  if constexpr (EPI == EPI_ROPE_KV) {
    const int head = n0 / p.kv.D, c0 = n0 % p.kv.D;
    if (head >= p.kv.Hq + p.kv.Hkv) {
      // v: its entries lie four tokens apart, so a row's 64 are turned through LDS to go out side by side, a sector of four
      // per 32 bytes (as the lanes hold them every one was a sector of its own: 61 rows x 6144 x 4096 22 -> 18 us)
      bf16_t* turn = reinterpret_cast<bf16_t*>(smem) + 64 + wid * 16 * 72;  // (behind the splits' flag; the wave's own)
      float x[8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = acc[0][h][e >> 2][e & 3];
        *reinterpret_cast<uint4v*>(turn + r16 * 72 + h * 32 + 8 * q) = pack8(x);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      const int c = c0 + (lane & 31) + (lane >= 32 ? p.kv.D / 2 : 0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int slot = __builtin_amdgcn_readlane(ahead.slot, r), row = m0 + wr * 16 + r;
        if (row < p.M && slot >= 0) rope_v_row(p.kv, slot, head)[4 * c] = turn[r * 72 + lane];
      }
      return;
    }
    float x[8], y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = acc[0][0][e >> 2][e & 3], y[e] = acc[0][1][e >> 2][e & 3];
    if (mrow < p.M) rope_kv_store<8>(p.kv, ahead, p.C, p.ldc, mrow, head, c0 + 8 * q, x, y);
  } else if constexpr (EPI == EPI_SWIGLU) {  // groups 2 g: gate columns, 2 g + 1: the matching up columns
#pragma unroll
    for (int g = 0; g < NP / 2; ++g) {
      const int col = (n0 + wc * (TN / WC)) / 2 + g * 32 + 8 * q;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = silu(acc[i][2 * g][e >> 2][e & 3]) * acc[i][2 * g + 1][e >> 2][e & 3];
        if (mrow + 16 * i < p.M && col < p.N / 2) *reinterpret_cast<uint4v*>(p.C + (size_t)(mrow + 16 * i) * p.ldc + col) = pack8(x);
      }
    }
  } else {
#pragma unroll
    for (int g = 0; g < NP; ++g) {
      const int col = n0 + wc * (TN / WC) + g * 32 + 8 * q;
      if (col >= p.N) continue;
      float b[8];
      if (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) unpack8(*reinterpret_cast<const uint4v*>(p.R + col), b);
      uint4v rv[MI];
      if (EPI == EPI_RESIDUAL) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
          rv[i] = *reinterpret_cast<const uint4v*>(p.R + (size_t)min(mrow + 16 * i, p.M - 1) * p.ldc + col);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        float x[8];
        if (EPI == EPI_RESIDUAL) unpack8(rv[i], b);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[e] = acc[i][g][e >> 2][e & 3];
          if (EPI != EPI_PLAIN) x[e] += b[e];
          if (EPI == EPI_BIAS_GELU) x[e] = gelu_erf(x[e]);
        }
        const uint4v o = pack8(x);
        if (mrow + 16 * i < p.M) *reinterpret_cast<uint4v*>(p.C + (size_t)(mrow + 16 * i) * p.ldc + col) = o;
        if constexpr (EPI == EPI_RESIDUAL && NORM) {  // of the row as stored: one partial per 32 columns
          unpack8(o, x);
          float t2 = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) t2 += x[e] * x[e];
          t2 = row_sum4(t2);
          if (q == 0 && mrow + 16 * i < p.M) p.ss.ss[(size_t)(mrow + 16 * i) * p.ss.P + (n0 + wc * (TN / WC)) / 32 + g] = t2;
        }
      }
    }
  }
}

// Whether the weights of a call in tiles of tm x tn pass the caches by (weights_pass, common.h): where one tile of rows reads them, but not from
// 49 rows on where they are wide, nor in tiles of 192 rows.  Time with it over without, weights from memory: 64 x 64 tiles up to 48 rows 0.85 to
// 0.99 (13 weights, 28672 x 4096 to 256000 x 3584), 56 and 64 rows of 65536 columns at most 0.92 to 1.00, of 128256 and 151936 x 2048 0.96 to
// 0.98, but 81920 to 151936 x 4096 up to 1.03; 128 x 128, 65 to 128 rows of 65536 columns at most 0.93 to 0.99, more columns up to 1.05; 128 x 192
// 0.93 to 1.01 throughout; 192 x 128, 160 and 192 rows 0.97 to 1.04.
bool past_caches(int M, int N, int K, int tm, int tn) {
  if (M > tm || tm > 128 || !weights_pass(2LL * N * K)) return false;
  return M <= 48 || N <= 65536 || tn == 192 || (tm == 64 && (long long)N * K < 5 << 26);
}

template <int EPI, int TM, int TN, int NST, bool NORM, bool NT>
int go(const typename ArgsOf<NORM>::type& p, hipStream_t s) {
  constexpr int kLds = NST * (TM + TN) * 128;
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)gemm2w_kernel<EPI, TM, TN, NST, NORM, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  (void)attr;
  gemm2w_kernel<EPI, TM, TN, NST, NORM, NT><<<p.tiles_m * p.tiles_n * p.splits, 256, kLds, s>>>(p);
  return (int)hipGetLastError();
}

// (Kernels of their own for NT, as gemm1s.hip's.  us, by a branch / now: bias 256 x 4096 x 4096 27.5 / 26.2, 96 x 8192 x 8192 47.4 /
// 44.8.)
template <int EPI, int TM, int TN, int NST, bool NORM = false>
int launch(typename ArgsOf<NORM>::type p, hipStream_t s) {
  p.tiles_m = (p.M + TM - 1) / TM;
  p.tiles_n = (p.N + TN - 1) / TN;
  // W rows of a stride whose low bits are zero lie on few memory channels, and all tiles walk K in step (gemm2g.hip): another
  // first step for each column tile spreads them.  N x K at 24 / 64 / 128 rows, us, before -> after: 16384 x 2048 17 / 17 / 26 -> 15 /
  // 15 / 23, 28672 x 4096 50 / 54 / 59 -> 48 / 52 / 51, 32000 x 4096 55 / 57 / 64 -> 55 / 57 / 52, 8192 x 8192 33 / 33 / 44 -> 27 /
  // 29 / 42, 4096 x 11008 23 / 25 / 35 -> 21 / 24 / 33; 4096 x 14336 and 6144 x 4096 level.  Many rounds of tiles spread by
  // themselves (128256 x 4096 185 / 202 / 212 -> 199 / 213 / 217), and from 300 rows on the matrix cores are the bound.  Plain
  // products without the folded norm, the projections of the models with routed experts, walk K from its start: behind them a
  // router picks experts, and another order of the sums moves rows that nearly tie (gemm2g.hip).
  const bool turned = (NORM || EPI != EPI_PLAIN) && p.M <= 256 && (long long)p.tiles_m * p.tiles_n <= 1024 && (p.K % 2048 == 0 || p.K % 1024 != 0);
  p.turned = 0;  // (a power of two less one: a division would hold the first loads back)
  while (turned && 2 * p.turned + 2 <= p.K / 64 / p.splits) p.turned = 2 * p.turned + 1;
  if constexpr (TM <= 128)
    if (past_caches(p.M, p.N, p.K, TM, TN)) return go<EPI, TM, TN, NST, NORM, true>(p, s);
  return go<EPI, TM, TN, NST, NORM, false>(p, s);
}

}  // namespace g2w
}  // namespace lwc

extern "C" int lwc_gemm1s_plan(int M, int N, int K, int epi, bool norm, long long max_splits);
extern "C" int lwc_gemm1s(const void*, const void*, void*, const void*, int, int, int, int, int, int, int, float*, int*, const lwc::RowSumsq*,
                          const lwc::RopeKV*, hipStream_t);

// (for tests)
extern "C" int lwc_gemm2w_past_caches(int M, int N, int K, int tm, int tn) { return lwc::g2w::past_caches(M, N, K, tm, tn); }

// epi 0: C = A W^T; 1: C = A W^T + R (R may be C); 2: C[:, :N/2] = silu(gate) * up over 32-row interleaved W (N % 64 == 0);
// 3: C = A W^T + bias (R = bias [N]); 4: C = gelu(A W^T + bias) (exact erf GELU).
// tile 0: 128 x 128, 1: 192 x 128, 2: 128 x 192 (not epi 2), 3: 64 x 64, there with splits K ranges per tile (part: tiles x
// splits x 4096 floats, count: tiles ints, zero on the first call; the kernel leaves them zero), 4: gemm1s.hip's weight streams (as
// lwc_gemm2w_plan says, with its K ranges over the same workspace).
// epi 5: the qkv projection with k and v written into the paged cache (kv; tile 3).  ss (tile 3): the folded RMSNorm: epi 0, 2
// and 5 scale their rows by it (epi 5 always), epi 1 writes N / 32 partials per row (N % 32 == 0).
// Requires K % 64 == 0, K / 64 >= splits, N % 8 == 0 and 16-byte rows and pointers.
// The tile and the K ranges of a call (max_splits: what the caller's workspace holds, in 64 x 64 partial tiles; norm: with the
// folded norm).  Up to 64 rows the weight streams where they take the call (lwc_gemm1s_plan); else:
// 64 x 64 up to 512 tiles (two workgroups per CU) and for any call of up to 64 rows.  Measured (us, 64 x 64 against 128 x 128):
// 512 rows x 4096 x K 1024 9.9 / 14.8, 512 x 4096 x 4096 35.5 / 42.8, 1000 x 3072 x 1024 (768 tiles) 14.9 / 13.8, 1000 x 4096 x
// 4096 (1024 tiles) 62 / 44.  Its K ranges: as many as fit one workgroup per CU, none below 16 steps.
// Measured, one / two / four / eight ranges: 61 x 4096 x 4096 22.3 / 15.7 / 12.1 / 14.8, 61 x 6144 x 4096 23.1 / 18.9 / 17.6 / 21.0,
// 61 x 4096 x 14336 70 / 44 / 28 / 31, 128 x 4096 x 4096 22.2 / 17.3 / 16.8 / 23.6, 256 x 1024 x 4096 21.5 / 15.1 / 11.3 / 12.4, 61 x
// 3072 x 1024 7.7 / 8.0 / 7.6 / 9.8.  (Ranges of 8 steps up to 32 tiles, 64 x 64 x 4096 9.4 -> 8.1, would be
// another order of sums in front of a router, as a walk from another step is.)
// Larger ones: the tile that takes the least time in whole rounds of two workgroups per CU, the larger of two that tie.
// Measured (128 x 128 against 128 x 192): 3600 x 2304 x 768 (522 and 348 tiles) 25.3 / 20.3, 3600 x 4096 x 1024 (928 and
// 638) 40.8 / 46.7, 7155 x 3072 x 768 (1344 and 896) 51.5 / 48.1.
extern "C" void lwc_gemm2w_plan(int M, int N, int K, int epi, bool norm, long long max_splits, int* tile, int* splits) {
  if (const int s = lwc_gemm1s_plan(M, N, K, epi, norm, max_splits)) {
    *tile = 4;
    *splits = s;
    return;
  }
  auto tiles = [&](int tm, int tn) { return ((long long)M + tm - 1) / tm * ((N + tn - 1) / tn); };
  *splits = 1;
  const long long small = tiles(64, 64);
  if (M <= 64 || small <= 512) {
    *tile = 3;
    const long long s = std::min(std::min(256 / std::max(small, 1LL), (long long)K / 1024), max_splits / std::max(small, 1LL));
    *splits = (int)std::max(1LL, s);
    return;
  }
  const long long square = (tiles(128, 128) + 511) / 512 * (128 * 128);
  const int wide = epi != lwc::g2w::EPI_SWIGLU ? 2 : 1;
  const long long rect = ((wide == 2 ? tiles(128, 192) : tiles(192, 128)) + 511) / 512 * (128 * 192);
  *tile = rect <= square ? wide : 0;
}

extern "C" int lwc_gemm2w(const void* A, const void* W, void* C, const void* R, int M, int N, int K, int lda, int ldc, int epi,
                          int tile, int splits, float* part, int* count, const lwc::RowSumsq* ss, const lwc::RopeKV* kv,
                          hipStream_t s) {
  using namespace lwc::g2w;
  if (K % 64 != 0 || K < 64 || N % 8 != 0 || lda % 8 != 0 || ldc % 8 != 0 || tile < 0 || tile > 4) return -1;
  if (192LL * (lda + K) * 2 >= (1LL << 31)) return -1;  // 32-bit buffer offsets in a tile
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C | (uintptr_t)R) & 15) return -1;
  if (splits < 1 || splits > K / 64 || (splits > 1 && (tile < 3 || part == nullptr || count == nullptr))) return -1;
  if (epi == EPI_SWIGLU && (N % 64 != 0 || tile == 2)) return -1;
  if ((epi == EPI_RESIDUAL || epi == EPI_BIAS || epi == EPI_BIAS_GELU) && R == nullptr) return -1;
  if (ss != nullptr && (tile < 3 || epi == EPI_BIAS || epi == EPI_BIAS_GELU || ss->P < 4 || ss->P % 4 != 0 || ss->P > 256 ||
                        (epi == EPI_RESIDUAL && (N % 32 != 0 || ss->P != N / 32)))) return -1;
  if (epi == EPI_ROPE_KV && (ss == nullptr || kv == nullptr || !lwc::rope_kv_ok(*kv, N) || (64LL + kv->D) * K * 2 >= (1LL << 31))) return -1;
  if (M == 0 || N == 0) return 0;
  if (((long long)M + 63) / 64 * ((N + 63) / 64) * splits >= (1LL << 31)) return -1;
  if (tile == 4) return lwc_gemm1s(A, W, C, R, M, N, K, lda, ldc, epi, splits, part, count, ss, kv, s);
  const Params p{(const lwc::bf16_t*)A, (const lwc::bf16_t*)W, (lwc::bf16_t*)C, (const lwc::bf16_t*)R, M, N, K, lda, ldc, 0, 0,
                 splits, part, count, 0};
  if (ss != nullptr) {
    const NormParams np{p, *ss, kv != nullptr ? *kv : lwc::RopeKV{}};
    switch (epi) {
      case EPI_PLAIN: return launch<EPI_PLAIN, 64, 64, 4, true>(np, s);
      case EPI_RESIDUAL: return launch<EPI_RESIDUAL, 64, 64, 4, true>(np, s);
      case EPI_SWIGLU: return launch<EPI_SWIGLU, 64, 64, 4, true>(np, s);
      default: return launch<EPI_ROPE_KV, 64, 64, 4, true>(np, s);
    }
  }
#define LWC_G2W(E)                                                                     \
  case E:                                                                              \
    if constexpr (E != EPI_SWIGLU)                                                     \
      if (tile == 2) return launch<E, 128, 192, 2>(p, s);                              \
    return tile == 3 ? launch<E, 64, 64, 4>(p, s) : tile == 1 ? launch<E, 192, 128, 2>(p, s) : launch<E, 128, 128, 2>(p, s);
  switch (epi) {
    LWC_G2W(EPI_PLAIN)
    LWC_G2W(EPI_RESIDUAL)
    LWC_G2W(EPI_SWIGLU)
    LWC_G2W(EPI_BIAS)
    LWC_G2W(EPI_BIAS_GELU)
  }
#undef LWC_G2W
  return -1;
}
