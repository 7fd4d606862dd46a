// K6 dense projection GEMM in two-phase K tiles + stream-K tail: C = A . W^T for the decode-batch projections
// (M = decode batch 512..4096; N, K >= 4096), with fused epilogues.
//
//   C[M, N]  = A[M, K] . W[N, K]^T  (+ R)            EPI_PLAIN / EPI_RESIDUAL
//   H[M, N/2] = silu(A . Wg^T) * (A . Wu^T)          EPI_SWIGLU, W rows gate/up interleaved in blocks of 32
//                                                     (ops.swiglu_interleave), so one tile holds both halves
//
// Tile pipeline:
//   workgroup : 8 waves (512 threads) = 2 (M) x 4 (N); wave tile 128 x 64 = 8 x 4 MFMA 16x16 tiles,
//               mfma_f32_16x16x32_bf16, 128 fp32 accumulators per lane.  Row tiles of 224 and 192 (R1 = 3, 2, row_tile): the
//               second quadrant has R1 instead of 4 tiles of 16 rows, the rest of unit A1 is not loaded.
//   K tile    : BK = 64 (128 B per row), staged global -> LDS by LDS-DMA (global_load_lds_dwordx4) in four
//               16 KiB UNITS, each of which is exactly what one compute phase reads:
//                 A0 = rows {0..63, 128..191}   (quadrant mi=0 of both wave rows)
//                 A1 = rows {64..127, 192..255} (mi=1)
//                 B0 = W rows {0..31, 64..95, 128..159, 192..223} (ni=0 of the 4 wave columns)
//                 B1 = the other 128 W rows (ni=1)
//               Two K-tile buffers (128 KiB LDS).
//   phases    : 2 per K tile, half of the wave's rows times all of its columns (32 MFMAs) each:
//                 P1 reads B0 B1 A0 -> acc[0..3]   stages A1 of tile t+1           vmcnt(8) (retires A1(t))
//                 P2 reads A1       -> acc[4..7]   stages A0, B0, B1 of tile t+2   vmcnt(8) (retires A0, B0, B1 (t+1))
//               Each phase: ds_reads, LDS-DMA, counted vmcnt, lgkmcnt(0), s_barrier, MFMA cluster at raised priority,
//               s_barrier.  vmcnt never reaches 0 inside the loop: a whole K tile stays in flight across the
//               barriers.  The two wave rows run one barrier apart (wr == 1 passes an extra barrier first),
//               so on every SIMD one wave issues MFMAs while its partner reads LDS and issues loads.  What bounds the loop is
//               the MFMAs and the hand-over of the matrix cores at the barriers.  Measured, us: four phases of 16 MFMAs with
//               the wait for their reads behind the barrier 719 at 8192^3, 657 at 4096 x 28672 x 4096; two phases 686 and
//               618; two with the DMA between the MFMAs instead 791 and 716; four with reads a phase ahead 736 and 662.
//   hazards   : RAW - a unit is read in the phase after the wait that retired it (every wave waits for its
//               own DMAs, then the barrier).  WAR - a wave comes to a phase's first barrier with its operands in registers;
//               a partner that stages in the next phase has passed that barrier.
//   tiles     : the loads run ahead over the end of a tile: its last K tile stages the first of the next one, and the epilogue
//               goes from the registers to memory while they are on their way (its stores are counted in the waits that
//               follow).  Through LDS, with nothing in flight, a tile of K 768 took 27 us, so 21.
//   LDS image : lane-linear DMA image, 16 B chunk c of A's unit row r stored at chunk c ^ ((r >> 1) & 7), of W's at c ^ ((r >> 3 &
//               3) * 2 + (r >> 1 & 1)): the 16 lanes of a ds_read_b128 group (A: 16 consecutive rows, W: rows 8 (l / 4) + l % 4,
//               same chunk) hit 16 distinct bank quads.  The swizzle is applied to the DMA SOURCE address and to the read.
//
// Work distribution (persistent, one workgroup per CU, grid = 8 XCDs x wpx):
//   The decode shapes do not divide into whole rounds of 256 tiles (qkv at M=3072: 288 tiles = 1.1 rounds;
//   o / down: 192 = 0.75; gate_up: 1344 = 5.25), so a plain one-tile-per-workgroup grid idles 12-44 % of the
//   chip in its last round.  Here the first `sk_tiles` tiles (the remainder plus one full round) are split
//   by K iterations (stream-K; where that costs less than it saves, call_cost): each XCD owns a contiguous, tile-aligned share of them and its wpx workgroups
//   split that share's K iterations evenly.  The remaining tiles run data-parallel, one per workgroup per
//   round, XCD x taking wpx consecutive tiles (m fastest: the XCD's tiles share W panels in its L2).
//   A tile cut between workgroups is finished by the one holding its last K iteration (the finaliser),
//   which adds the fp32 partials the others wrote to the workspace.  Each workgroup walks its stream-K
//   range backwards, so it publishes its partial (range end) first and finalises (range start) last, and
//   a finaliser only waits on LOWER block ids of its own XCD — workgroups dispatched earlier, hence
//   resident: no co-residency assumption, no deadlock.  Partial hand-off: stores of device scope, vmcnt(0), barrier, flag
//   store; the reader polls the flag, resets it for the next launch (flags start zeroed), barrier, loads of device
//   scope.  (With fences instead, each of which writes an XCD's L2 back or drops it: 1095 rows x 6144 x 4096 72 us, so 67; 4096 x
//   14336 143 and 135.)
// fp8 (EPI_FP8, EPI_FP8_SWIGLU): e4m3 rows are the same bytes; a phase's 32 bf16 MFMAs are 16 scaled ones of four times the K at twice the
// cycles, and the scales of a tile's rows and columns come into LDS with its last K tile.  Against one tile per workgroup (gemm8g.hip's dense
// mode), whose last round of 32 to 48 tiles idles most of the chip, us, 8682 rows: x 28672 x 4096 SwiGLU 731 -> 690 (2.95 PFLOP/s), x 4096
// x 14336 410 -> 336, x 6144 x 4096 194 -> 171, x 4096 x 4096 143 -> 116; with block scales, which come with each K tile, from MX x 4096 x 4096 151 -> 121,
// x 4096 x 14336 449 -> 356, SwiGLU to MX of 16641 rows x 28672 x 4096 1407 -> 1334; 64 documents through three e5 layers 3897 -> 3605.  (The
// residual added here spilled, and cost 32 to 38 us for the 17 that the norm behind it gains.)
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "common.h"

namespace lwc {
namespace g8p {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kUnitB = 128 * 128;   // 128 rows x 128 B
constexpr int kBufB = 4 * kUnitB;   // one K tile: A0 A1 B0 B1
constexpr int kLdsB = 2 * kBufB;    // 128 KiB
constexpr int kUA0 = 0, kUA1 = kUnitB, kUB0 = 2 * kUnitB, kUB1 = 3 * kUnitB;
// cache policy of buffer loads and stores: device scope (past the caches of one XCD), streaming
constexpr int kSC1 = 16;
constexpr int kPartialF = 256 * 256;  // fp32 partial tile per workgroup

// (fp8: e4m3 A and W, their element counts halved as of bf16, scales of A's rows and W's rows applied to the accumulators)
enum Epi { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_BIAS = 3, EPI_BIAS_GELU = 4, EPI_FP8 = 5, EPI_FP8_SWIGLU = 6,
  EPI_FP8_MX_OUT = 7,    // SwiGLU, its result as e4m3 with a scale per row and 32 columns
  EPI_FP8_MX = 8 };      // A with such scales, a scale per row and 32 of K, instead of one a row
// fp8: the scales of two tiles, behind the K tiles, and of A's blocks in two K tiles, [256 rows][4] (twice: the waves' loads are as many)
constexpr int kScalesB = 2 * 2048, kMxB = 2 * 2048;

struct Params {
  const bf16_t* A;
  const bf16_t* W;
  bf16_t* C;
  const bf16_t* R;     // EPI_RESIDUAL: residual [M, ldc]; EPI_BIAS / EPI_BIAS_GELU: bias [N]
  float* ws;    // [8 * wpx, kPartialF] partial tiles
  int* flags;   // [8 * wpx] partial-ready flags (zero between launches)
  int M, N, K, lda, ldc;  // N = rows of W
  int tiles_m, tiles_n, KT;
  int gm;  // tile order: groups of gm m-tiles, n fastest across a group (32 consecutive tiles ~ 4 x 8)
  int wpx, sk_tiles, dp_rounds;
  const float *a_scale, *w_scale;  // fp8: [M], [N]
  // e8m0 block scales [K / 128][s_rows][4] of A, [N / 256][s_rows][4] of the result (as in gemm8g.hip)
  const uint8_t* a_mx;
  uint8_t* mx_out;
  int s_rows;
  int nt;  // the output is larger than the last-level cache: its stores pass the caches by
};

LWC_DEVICE float4v mfma(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef int v8i32 __attribute__((ext_vector_type(8)));
// (sb: the scale of b's row, its block of the lane's K; 127: one)
LWC_DEVICE float4v mfma8(const uint4v (&a)[2], const uint4v (&b)[2], const float4v& c, int sb) {
  const v8i32 av = {(int)a[0].x, (int)a[0].y, (int)a[0].z, (int)a[0].w, (int)a[1].x, (int)a[1].y, (int)a[1].z, (int)a[1].w};
  const v8i32 bv = {(int)b[0].x, (int)b[0].y, (int)b[0].z, (int)b[0].w, (int)b[1].x, (int)b[1].y, (int)b[1].z, (int)b[1].w};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 0, 0, 0, 127, 0, sb);
}

// Bytes from row m0 of A's first plane of block scales to the end of its last one: M rows of s_rows there, which other calls' may follow,
// or the tensor's end
LWC_HOST_DEVICE int mx_bytes(int planes, int s_rows, int M, int m0) { return ((planes - 1) * s_rows + M - m0) * 4; }

// x * sigmoid(x) with v_rcp_f32 (1 ulp) instead of the IEEE division sequence (v_div_scale x2, v_div_fmas,
// v_div_fixup around an rcp: ~9 VALU per element in an epilogue of 256 per lane); the result is rounded
// to bf16 (or e4m3) anyway.  x -> -inf: rcp(inf) = 0, x * 0 = -0 as the division gives
LWC_DEVICE float silu(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
// K-iteration range [a, e) of stream-K workgroup j (of wpx) on XCD x.
LWC_DEVICE void sk_range(const Params& p, int x, int j, int& a, int& e) {
  const int t0 = p.sk_tiles * x / 8, t1 = p.sk_tiles * (x + 1) / 8;
  const int ix = (t1 - t0) * p.KT;
  a = t0 * p.KT + (int)((long long)ix * j / p.wpx);
  e = t0 * p.KT + (int)((long long)ix * (j + 1) / p.wpx);
}

// Tile t -> (m, n): grouped order, gm m-tiles per group, m fastest inside the group, so the wpx
// consecutive tiles an XCD runs in one round form a ~gm x (wpx / gm) block whose A and W panels its
// L2 shares (a plain m-fastest order spans every m-tile of the matrix: 1.5x the L2 misses at 4096^3).
LWC_DEVICE void tile_mn(const Params& p, int t, int& m, int& n) {
  const int group = p.gm * p.tiles_n;
  const int first_m = (t / group) * p.gm;
  const int gsz = min(p.tiles_m - first_m, p.gm);
  const int in = t % group;
  m = first_m + in % gsz;
  n = in / gsz;
}

// A piece of a workgroup's work: the K iterations [klo, khi) of a tile.
struct Item {
  int it, round;  // the items before it: what is left of the stream-K range, data-parallel rounds
  int tile, klo, khi;
};

template <int EPI, int R1>
__global__ void __launch_bounds__(512) gemm8p_kernel(Params p) {
  constexpr int BMH = 64 + 16 * R1;  // rows of a wave row
  constexpr bool kF8 = EPI >= EPI_FP8, kMx = EPI == EPI_FP8_MX, kMxOut = EPI == EPI_FP8_MX_OUT;
  constexpr bool kSwiglu = EPI == EPI_SWIGLU || EPI == EPI_FP8_SWIGLU || kMxOut;
  constexpr int kAhead = kMx ? 9 : 8;  // loads of a K tile
  constexpr int CW = kSwiglu ? 32 : 64, NH = CW / 32;  // output columns of a wave, in groups of 32
  constexpr int kStores = (4 + R1) * (kMxOut ? 2 : NH);  // store instructions of an epilogue
  constexpr bool kBias = EPI == EPI_BIAS || EPI == EPI_BIAS_GELU;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int KT = p.KT;
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4;
  const int wr = wid >> 2, wc = wid & 3;

  int sk_a = 0, sk_e = 0;
  if (p.sk_tiles > 0) sk_range(p, xcd, j, sk_a, sk_e);
  // (divisions run on the vector units; what follows from their results is to stay scalar)
  auto uni = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  sk_a = uni(sk_a), sk_e = uni(sk_e);
  // ---- the work items, one after the other: stream-K segments (backwards), then data-parallel tiles ----
  auto next = [&](Item& w) -> bool {
    if (w.it > sk_a) {
      w.tile = uni((w.it - 1) / KT);
      const int seg = max(sk_a, w.tile * KT);
      w.klo = seg - w.tile * KT;
      w.khi = w.it - w.tile * KT;
      w.it = seg;
      return true;
    }
    if (w.round >= p.dp_rounds) return false;
    // (a last round that is not full is spread over the XCDs)
    const int begin = p.sk_tiles + w.round * 8 * p.wpx, each = min(p.wpx, (p.tiles_m * p.tiles_n - begin + 7) / 8);
    w.tile = begin + xcd * each + j;
    if (j >= each || w.tile >= p.tiles_m * p.tiles_n) return false;
    w.klo = 0;
    w.khi = KT;
    ++w.round;
    return true;
  };

  // per-thread DMA geometry (byte offsets from the tile's buffer base): unit u, instruction i -> unit row
  // ru = i*64 + tid/8 at LDS chunk tid%8, which holds a global chunk of that row (swizzle on the source): chunk c of A row r
  // lies at c ^ (r / 2 % 8), of W row r at c ^ (r / 8 % 4 * 2 + r / 2 % 2)
  const int chkA = ((tid & 7) ^ ((tid >> 4) & 7)) * 8, chkW = ((tid & 7) ^ ((tid >> 6 & 3) * 2 + (tid >> 4 & 1))) * 8;
  uint32_t voA[2][2], voW[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // (R1 < 4: the rest of unit A1 lies past the resource's end, no memory request)
      voA[h][i] = h == 0 || (tid >> 3) < 16 * R1 ? (uint32_t)(((i * BMH + h * 64 + (tid >> 3)) * p.lda + chkA) * 2) : 0x60000000u;
      voW[h][i] = (uint32_t)((((2 * i + (tid >> 8)) * 64 + h * 32 + ((tid >> 3) & 31)) * p.K + chkW) * 2);
    }
  const int dst_lane0 = wid * 64 * 16;  // wave-uniform LDS destination of instruction 0 inside a unit
  // operand reads: A tile i holds rows 16 i + r16; W tile h holds rows 8 (r16 / 4) + 4 h + r16 % 4, so that a lane's
  // accumulators of the pair h = 0, 1 are the eight consecutive columns 8 q .. of output row r16
  const int pos = (q ^ (r16 >> 1)) << 4;  // of K entries 0 .. 31; 32 .. 63 lie at pos ^ 64
  const int offA = (wr * 64 + r16) * 128, offW = (wc * 32 + 8 * (r16 >> 2) + (r16 & 3)) * 128;

  // the K tile that is being staged, of an item that may be ahead of the one being multiplied: rows past M / N fall outside
  // num_records and load as zeros (their outputs are not stored); behind the last K tile nothing is asked for
  Item ahead{sk_e, 0, 0, 0, 0};
  const bf16_t *srcA = nullptr, *srcW = nullptr;
  int numA = 0, numW = 0, kt = -1, mS = 0;
  auto advance = [&] {
    kt = uni(kt + 1);
    if (kt < ahead.khi) return;
    numA = numW = 0;
    if (!next(ahead)) return;
    int tm, tn;
    tile_mn(p, ahead.tile, tm, tn);
    const int m0 = uni(tm) * 2 * BMH, n0 = uni(tn) * 256;
    srcA = p.A + (size_t)m0 * p.lda;
    srcW = p.W + (size_t)n0 * p.K;
    numA = min(p.M - m0, 2 * BMH) * p.lda * 2;
    numW = min(p.N - n0, 256) * p.K * 2;
    mS = m0;
    kt = uni(ahead.klo);
  };
  auto stage = [&](int u, uint8_t* buf) {
    const __amdgpu_buffer_rsrc_t r = u < 2 ? uniform_rsrc(srcA, numA) : uniform_rsrc(srcW, numW);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      auto* dst = (__attribute__((address_space(3))) void*)(buf + u * kUnitB + i * 512 * 16 + dst_lane0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, u < 2 ? voA[u][i] : voW[u - 2][i], kt * 128, 0, 0);
    }
    if constexpr (kMx) {
      if (u == 0) {  // the scales of the K tile's rows, four bytes a row
        auto* dst = (__attribute__((address_space(3))) void*)(smem + kLdsB + kScalesB + (buf == smem ? 0 : 2048) + wid * 256);
        const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(p.a_mx + (size_t)mS * 4, numA ? mx_bytes(KT, p.s_rows, p.M, mS) : 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 4, (tid & 255) * 4, kt * p.s_rows * 4, 0, 0);
      }
    }
  };

  // acc[i][jj]: 16 rows (tile i) x columns 32 (jj / 2) + 8 q + 4 (jj % 2) .. of the wave's 128 x 64, row r16 of the tile.
  // (The 32x32x16 MFMA with the same units and phases measured ~10 % slower on every shape.)
  float4v acc[4 + R1][4];
  uint4v a[4][2], b[4][2];
  int sc[kMx ? 4 + R1 : 1];
  auto mma = [&](auto n, int i0) {
    if constexpr (kF8) {
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int i = 0; i < decltype(n)::value; ++i) acc[i0 + i][jj] = mfma8(b[jj], a[i], acc[i0 + i][jj], kMx ? sc[kMx ? i0 + i : 0] : 127);
      // (else the compiler sinks the scaled MFMAs past the barriers into the next phase: 8682 x 28672 x 4096 SwiGLU 814 us for 690)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int i = 0; i < decltype(n)::value; ++i) asm volatile("" : "+v"(acc[i0 + i][jj]));
      return;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int i = 0; i < decltype(n)::value; ++i) acc[i0 + i][jj] = mfma(b[jj][s], a[i][s], acc[i0 + i][jj]);
  };
  auto rdA = [&](const uint8_t* unit, auto n) {
#pragma unroll
    for (int i = 0; i < decltype(n)::value; ++i) {
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
  constexpr std::integral_constant<int, 4> n4{};
  constexpr std::integral_constant<int, R1> n1{};

#define G8_BAR() __builtin_amdgcn_s_barrier()
#define G8_VM(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")
// (a wave comes to the barrier with its operands in registers: behind it their units may be filled anew)
#define G8_MFMA(n, i0)                               \
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
  G8_BAR();                                          \
  __builtin_amdgcn_s_setprio(1);                     \
  mma(n, i0);                                        \
  __builtin_amdgcn_s_setprio(0);                     \
  G8_BAR()

  advance();
  stage(0, smem), stage(2, smem), stage(3, smem), stage(1, smem);
  advance();
  stage(0, smem + kBufB), stage(2, smem + kBufB), stage(3, smem + kBufB);
  G8_VM(kAhead);
  G8_BAR();
  if (wr == 1) G8_BAR();  // stagger the two wave rows by one barrier
  int at = 0;           // LDS buffer of the K tile at hand
  bool stored = false;  // an epilogue's stores have gone out after unit B1 of the next K tile
  uint4v bias[2];
  int scales = kLdsB;  // fp8: where the scales of the tile at hand lie

  for (Item cur{sk_e, 0, 0, 0, 0}; next(cur);) {
#pragma unroll
    for (int i = 0; i < 4 + R1; ++i)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) acc[i][jj] = float4v{0.f, 0.f, 0.f, 0.f};
    int tm, tn;
    tile_mn(p, cur.tile, tm, tn);
    const int m0 = uni(tm) * 2 * BMH, n0 = uni(tn) * 256;

    int left = cur.khi - cur.klo;  // (at least one)
    do {
      uint8_t* cb = smem + at;
      at ^= kBufB;
      uint8_t* nb = smem + at;
      if constexpr (kBias) {
        if (left == 1) {
          const int col = n0 + wc * 64 + 8 * q;
          const __amdgpu_buffer_rsrc_t rb = uniform_rsrc(p.R, p.N * 2);
#pragma unroll
          for (int h = 0; h < 2; ++h) bias[h] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(rb, (col + 32 * h) * 2, 0, 0));
        }
      }
      if constexpr (kF8) {
        if (left == 1) {  // the scales of the tile's rows (waves 0 .. 3) and columns, one a thread
          auto* dst = (__attribute__((address_space(3))) void*)(smem + scales + wid * 256);
          const __amdgpu_buffer_rsrc_t rs = wr == 0 ? uniform_rsrc(p.a_scale + m0, kMx ? 0 : min(p.M - m0, 256) * 4) : uniform_rsrc(p.w_scale + n0, min(p.N - n0, 256) * 4);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 4, (tid & 255) * 4, 0, 0, 0);
        }
      }
      rdB(cb + kUB0, 0);
      rdB(cb + kUB1, 2);
      rdA(cb + kUA0, n4);
      if constexpr (kMx) {
        const uint8_t* st = smem + kLdsB + kScalesB + (cb == smem ? 0 : 2048) + (wr * BMH + r16) * 4 + q;
#pragma unroll
        for (int i = 0; i < 4 + R1; ++i) sc[i] = st[i * 64];
      }
      stage(1, nb);
      if (stored) G8_VM(kAhead + kStores);
      else G8_VM(kAhead);
      G8_MFMA(n4, 0);
      advance();
      rdA(cb + kUA1, n1);
      stage(0, cb), stage(2, cb), stage(3, cb);
      if (stored && !(kF8 && left == 1)) G8_VM(kAhead + kStores);  // (the scales have landed with the tile's last K tile)
      else G8_VM(kAhead);
      G8_MFMA(n1, 4);
      stored = false;
    } while (--left > 0);

    // (an opaque copy of the lane: what follows is computed here, not ahead of the loop, where it would cost it registers)
    int el = lane, ew = wid;
    asm volatile("" : "+v"(el), "+s"(ew));
    // ---- stream-K hand-off (the wave rows meet for it and part again) ----
    const bool whole = cur.khi == KT;
    if (!whole || cur.klo > 0) {
      if (wr == 0) G8_BAR();
      if (!whole) {  // contributor: publish the fp32 partial, no store of C
        const __amdgpu_buffer_rsrc_t rp = uniform_rsrc(p.ws + (size_t)blockIdx.x * kPartialF, kPartialF * 4);
#pragma unroll
        for (int i = 0; i < 4 + R1; ++i)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, acc[i][jj]), rp, (ew * 2048 + el) * 16, (i * 4 + jj) * 1024, kSC1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) __hip_atomic_store(p.flags + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {  // finaliser: add the partials of the lower workgroups of this XCD covering [0, klo)
        const int tile_begin = cur.tile * KT;
        for (int jp = j - 1; jp >= 0; --jp) {
          int pa, pe;
          sk_range(p, xcd, jp, pa, pe);
          if (pe <= tile_begin) break;
          if (pa == pe) continue;  // empty range: no partial
          const int blk = jp * 8 + xcd;
          if (tid == 0) {
            while (__hip_atomic_load(p.flags + blk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
              __builtin_amdgcn_s_sleep(1);
            __hip_atomic_store(p.flags + blk, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          __syncthreads();
          const __amdgpu_buffer_rsrc_t rp = uniform_rsrc(p.ws + (size_t)blk * kPartialF, kPartialF * 4);
#pragma unroll
          for (int i = 0; i < 4 + R1; i += 2) {
            float4v part[2][4];
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (i + k / 4 < 4 + R1)
                part[k / 4][k % 4] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(rp, (ew * 2048 + el) * 16, (i * 4 + k) * 1024, kSC1));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (i + k / 4 < 4 + R1) acc[i + k / 4][k % 4] += part[k / 4][k % 4];
            __builtin_amdgcn_sched_barrier(0);
          }
          if (pa <= tile_begin) break;
        }
      }
      if (wr == 1) G8_BAR();
    }

    // ---- epilogue: a lane holds eight consecutive columns of a row, so its 16 bytes go out from the registers.  Stores past M or
    // N fall outside the resource: the number of store instructions, which the waits above count, is always the same ----
    if (whole) {
      const int ncols = kSwiglu ? p.N / 2 : p.N;
      const int ncol0 = kSwiglu ? n0 / 2 + wc * 32 : n0 + wc * 64, row0 = m0 + wr * BMH;
      const int cols_here = max(0, min(ncols - ncol0, CW));
      uint32_t vo[NH];
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int col = 32 * h + 8 * (el >> 4);
        vo[h] = col < cols_here ? (uint32_t)(((el & 15) * p.ldc + col) * 2) : 0xfffffff0u;
      }
      auto rows_of = [&](const bf16_t* base, int i) {
        const int rows = cols_here == 0 ? 0 : min(p.M - row0 - 16 * i, 16);
        return uniform_rsrc(base + (size_t)(row0 + 16 * i) * p.ldc + ncol0, rows > 0 ? ((rows - 1) * p.ldc + cols_here) * 2 : 0);
      };
      // the residual of all rows is asked for before the first store, behind which it would have to wait for it
      uint4v rv[EPI == EPI_RESIDUAL ? 4 + R1 : 1][NH];
      if constexpr (EPI == EPI_RESIDUAL) {
#pragma unroll
        for (int i = 0; i < 4 + R1; ++i) {
          const __amdgpu_buffer_rsrc_t rr = rows_of(p.R, i);
#pragma unroll
          for (int h = 0; h < NH; ++h) rv[i][h] = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(rr, vo[h], 0, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      float ws[kF8 ? 2 : 1][8];
      if constexpr (kF8) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 8; e += 4)
            *reinterpret_cast<float4v*>(&ws[c][e]) = *reinterpret_cast<const float4v*>(smem + scales + 1024 + (wc * 64 + 32 * c + 8 * (el >> 4) + e) * 4);
      }
      auto store = [&](auto policy) {
#pragma unroll
      for (int i = 0; i < 4 + R1; ++i) {
        const __amdgpu_buffer_rsrc_t rc = rows_of(p.C, i);
        float as = 1.f;
        if constexpr (kF8 && !kMx) as = *reinterpret_cast<const float*>(smem + scales + (wr * BMH + 16 * i + (el & 15)) * 4);
#pragma unroll
        for (int h = 0; h < NH; ++h) {
          float x[8], y[8];
          if constexpr (kBias) unpack8(bias[h], y);
          if constexpr (EPI == EPI_RESIDUAL) unpack8(rv[i][h], y);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[e] = acc[i][2 * h + e / 4][e % 4];
            if constexpr (kF8) x[e] *= as * ws[h][e];
            if constexpr (EPI == EPI_SWIGLU) x[e] = silu(x[e]) * acc[i][2 + e / 4][e % 4];
            if constexpr (kF8 && kSwiglu) x[e] = silu(x[e]) * (acc[i][2 + e / 4][e % 4] * (as * ws[1][e]));
            if constexpr (kBias || EPI == EPI_RESIDUAL) x[e] += y[e];
            if constexpr (EPI == EPI_BIAS_GELU) x[e] = gelu_erf(x[e]);
          }
          if constexpr (!kMxOut) {
            __builtin_amdgcn_raw_buffer_store_b128(pack8(x), rc, vo[h], 0, decltype(policy)::value);
          } else {  // the wave's 32 columns of a row are a block, held by four lanes
            float v[8];
            unpack8(pack8(x), v);
            float mx = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
            const int exp = mx_exp(row_max4(mx)), m = row0 + 16 * i, rows = min(max(p.M - m, 0), 16);
            const float inv = __builtin_amdgcn_ldexpf(1.f, -exp);
            uint32_t lo = 0, hi = 0;
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[0] * inv, v[1] * inv, lo, false);
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(v[2] * inv, v[3] * inv, lo, true);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[4] * inv, v[5] * inv, hi, false);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(v[6] * inv, v[7] * inv, hi, true);
            const __amdgpu_buffer_rsrc_t r8 = uniform_rsrc((uint8_t*)p.C + (size_t)m * p.ldc + ncol0, rows > 0 ? (rows - 1) * p.ldc + 32 : 0);
            __builtin_amdgcn_raw_buffer_store_b64(uint2v{lo, hi}, r8, (el & 15) * p.ldc + 8 * (el >> 4), 0, decltype(policy)::value);
            const __amdgpu_buffer_rsrc_t rm = uniform_rsrc(p.mx_out + ((size_t)(n0 / 256) * p.s_rows + m) * 4, rows * 4);
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)(exp + 127), rm, el < 16 ? el * 4 + wc : 0x7ffffff0, 0, 0);
          }
        }
      }
      };
      if (p.nt) store(std::integral_constant<int, kNT>{});
      else store(std::integral_constant<int, 0>{});
      stored = true;
    }
    if constexpr (kF8) scales ^= kLdsB ^ (kLdsB + 2048);
  }
  if (wr == 0) G8_BAR();  // re-align the wave rows
  G8_VM(0);               // the last K tile's requests have ended before the LDS is given back
#undef G8_MFMA
#undef G8_VM
#undef G8_BAR
}

template <int EPI, int R1>
int launch(const Params& p, hipStream_t s) {
  constexpr int kLds = kLdsB + (EPI >= EPI_FP8 ? kScalesB : 0) + (EPI == EPI_FP8_MX ? kMxB : 0);
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)gemm8p_kernel<EPI, R1>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    attr = true;
  }
  gemm8p_kernel<EPI, R1><<<8 * p.wpx, 512, kLds, s>>>(p);
  return (int)hipGetLastError();
}

template <int EPI>
int launch(const Params& p, int r1, hipStream_t s) {
  return r1 == 4 ? launch<EPI, 4>(p, s) : r1 == 3 ? launch<EPI, 3>(p, s) : launch<EPI, 2>(p, s);
}

// Experiment knob (A/B in one process, scripts/microbench.py g8ab): LWC_G8_GM, the tile group height
// (default 8; 1 = plain m-fastest order).
int env_int(const char* name, int dflt) {
  const char* v = getenv(name);
  return v ? atoi(v) : dflt;
}

int device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 8) cus = 256;
  }
  return cus;
}

// Workgroups per XCD: at least ~8 K iterations per stream-K workgroup, so small problems get a smaller grid.
int grid_wpx(int tiles, int KT) {
  const int wpx = device_cus() / 8;
  const long long iters = (long long)tiles * KT;
  return iters < 8LL * 8 * wpx ? (int)std::max(1LL, iters / 64) : wpx;
}

// The time of `tiles` tiles on 8 x wpx workgroups, us, and whether those of a last round that is not full are cut between all
// workgroups (or run as they are while the others idle), whichever is less.  R1: tiles of 256, 224 or 192 rows.
//   With whole rounds, 256 rows are 1.45 us per K iteration and round, 224 0.93 and 192 0.85 of that (28672 x 4096 and 4096 x 14336).  A
// round that is not full: the others run at a higher clock, three quarters of the idle time are lost.  A cut costs its hand-off, 256
// KiB through one compute unit each way, and workgroups that walk K apart no longer share their rows' way through an XCD's L2.  Cut less
// uncut, us, by how full the last round is: K 768 0.05 / 0.38 / 0.75 / 0.89 -3 / +3 / +9 / +10; K 2048 0.06 / 0.5 / 0.88 -18 / -7 / +29; K 4096
// -46 / -16 / +50; K 8192 -99 / -34 / +81; K 14336 0.25 / 0.88 -129 / +123; K 384 0.05 / 0.89 +2 / +8.
//   With fewer tiles than workgroups the times were fitted to 253 calls of 200 to 7156 rows, 384 to 8192 columns and K 256 to 14336, each with
// every row tile, cut and uncut (rms 0.10 and 0.04): uncut a start, an end and the iterations, slower as more CUs run; cut the
// iterations of the XCD that has the most tiles, a hand-off per workgroup of a tile, more where these do not divide a tile's K evenly
// and for each tile of an XCD.  The choice is 1.008 of the best of the six on average, 1.12 at worst.  us, uncut / cut, 192 rows: 520 x 768 x 3072 (9 tiles)
// 51 / 33, 200 x 2304 x 3072 (18) 52 / 36, 520 x 768 x 2048 38 / 28, 520 x 4096 x 14336 (48) 218 / 86; 1095 x 4096 x 1024 (96) 26 / 29, 2200 x
// 3072 x 768 (144) 24 / 31.
constexpr double kIter[5] = {0, 0, 1.45 * 0.85, 1.45 * 0.93, 1.45};
constexpr double kUncut[5][3] = {{}, {}, {10.9, 0.83, 0.26}, {11.8, 0.86, 0.37}, {12.5, 0.88, 0.42}};
constexpr double kCut[5][5] = {{}, {}, {2.8, 1.29, 3.8, 3.8, 0.42}, {1.7, 1.33, 4.8, 4.2, 0.61}, {0.7, 1.46, 5.2, 4.3, 0.71}};
double call_cost(int tiles, int wpx, int KT, int r1, bool* cut) {
  const int G = 8 * wpx, rest = tiles % G;
  if (tiles < G) {
    const double *u = kUncut[r1], *c = kCut[r1];
    const int share = (tiles + 7) / 8;  // the most tiles of an XCD
    const double uncut = u[0] + KT * (u[1] + u[2] * tiles / 256);
    const double split = c[0] + c[1] * KT * share / wpx + c[2] * wpx / share + (wpx % share ? c[3] : 0) + c[4] * tiles / 8;
    *cut = split < uncut;
    return std::min(split, uncut);
  }
  const double full = (double)rest / G, idle = rest == 0 ? 0 : 0.75 * kIter[r1] * KT * (1 - full);
  const double split = rest == 0 ? 0 : 6 + KT * (0.2 + 0.7 * std::max(0.0, full - 0.3));
  *cut = rest != 0 && split < idle;
  return 6 + kIter[r1] * KT * tiles / G + std::min(split, idle);
}

// The row tile (R1): a smaller one pays where it saves rows past M (1095 rows are five tiles either way) or fills the last round.
// Measured, us, 256 / 224 / 192 rows: gate|up 28672 x 4096 of 520 / 1095 / 1700 / 3333 rows 130 / 128 / 122, 207 / 203 / 243, 291 / 304 / 347, 555 / 585 /
// 662; down 4096 x 14336 of 900 / 1095 / 2200 rows 101 / 114 / 114, 124 / 121 / 116, 216 / 207 / 215.
int row_tile(int M, int tiles_n, int KT) {
  int best = 4;
  double least = 0;
  for (int r1 = 4; r1 >= 2; --r1) {
    bool cut;
    const int bm = 128 + 32 * r1, tiles = (M + bm - 1) / bm * tiles_n;
    const double us = call_cost(tiles, grid_wpx(tiles, KT), KT, r1, &cut);
    if (r1 == 4 || us < least) best = r1, least = us;
  }
  return best;
}

// How a call is cut: its row tiles, grid, stream-K tiles (none without a workspace) and rounds of whole tiles
int plan(Params& p, bool swiglu) {
  p.tiles_n = (p.N + 255) / 256, p.KT = p.K / 64;
  const int r1 = p.lda < (1 << 20) ? row_tile(p.M, p.tiles_n, p.KT) : 4, bm = 128 + 32 * r1;
  p.tiles_m = (p.M + bm - 1) / bm;
  const int tiles = p.tiles_m * p.tiles_n;
  p.wpx = grid_wpx(tiles, p.KT);
  const int G = 8 * p.wpx;
  bool cut;
  call_cost(tiles, p.wpx, p.KT, r1, &cut);
  if (!p.ws) cut = false;
  p.dp_rounds = cut ? std::max(0, tiles / G - 1) : (tiles + G - 1) / G;
  p.sk_tiles = cut ? tiles - p.dp_rounds * G : 0;
  p.gm = std::max(1, env_int("LWC_G8_GM", 8));
  p.nt = (long long)p.M * p.N * (swiglu ? 1 : 2) > 256LL << 20;
  return r1;
}

}  // namespace g8p
}  // namespace lwc

// Workgroups the kernel launches (= partial slots / flags the workspace must hold): 8 x (CUs / 8).
extern "C" int lwc_gemm8p_slots() { return 8 * (lwc::g8p::device_cus() / 8); }

// epi 0: C = A W^T; 1: C = A W^T + R; 2: C[:, :N/2] = silu(gate) * up over 32-row interleaved W (N % 64 == 0);
// 3: C = A W^T + bias (R = bias [N]); 4: C = gelu(A W^T + bias) (exact erf GELU).
// Requires K % 64 == 0, N % 8 == 0, lda / ldc % 8 == 0 (16-byte rows); ws >= slots * 65536 floats,
// flags >= slots ints, zero on the first call (the kernel leaves them zero).
extern "C" int lwc_gemm8p(const void* A, const void* W, void* C, const void* R, float* ws, int* flags, int M, int N,
                          int K, int lda, int ldc, int epi, hipStream_t s) {
  using namespace lwc::g8p;
  if (K % 64 != 0 || K < 64 || N % 8 != 0 || lda % 8 != 0 || ldc % 8 != 0) return -1;
  if ((long long)M * lda * 2 >= (1LL << 31) || 256LL * K * 2 >= (1LL << 31) || ldc >= (1 << 26)) return -1;  // 32-bit buffer offsets
  if (epi == EPI_SWIGLU && N % 64 != 0) return -1;
  if ((epi == EPI_RESIDUAL || epi == EPI_BIAS || epi == EPI_BIAS_GELU) && R == nullptr) return -1;
  if (M == 0 || N == 0) return 0;
  Params p{};
  p.A = (const lwc::bf16_t*)A, p.W = (const lwc::bf16_t*)W, p.C = (lwc::bf16_t*)C, p.R = (const lwc::bf16_t*)R, p.ws = ws, p.flags = flags;
  p.M = M, p.N = N, p.K = K, p.lda = lda, p.ldc = ldc;
  const int r1 = plan(p, epi == EPI_SWIGLU);
  switch (epi) {
    case EPI_PLAIN: return launch<EPI_PLAIN>(p, r1, s);
    case EPI_RESIDUAL: return launch<EPI_RESIDUAL>(p, r1, s);
    case EPI_SWIGLU: return launch<EPI_SWIGLU>(p, r1, s);
    case EPI_BIAS: return launch<EPI_BIAS>(p, r1, s);
    case EPI_BIAS_GELU: return launch<EPI_BIAS_GELU>(p, r1, s);
  }
  return -1;
}

// What a tile from row m0 on may read of A's block scales (for tests).
extern "C" int lwc_gemm8p_mx_bytes(int planes, int s_rows, int M, int m0) { return lwc::g8p::mx_bytes(planes, s_rows, M, m0); }

// C [M, N] = (A [M, K] . W [N, K]^T) * a_scale[row] * w_scale[column] of e4m3 A and W, or (swiglu 1, W's rows gate / up interleaved in
// blocks of 32) silu(gate) * up [M, N / 2], bf16; swiglu 2: that as e4m3 with block scales mx_out (N % 256 == 0, ldc % 16 == 0, bytes).  a_mx: A's
// block scales in place of a_scale (swiglu 0).  Scale planes of s_rows rows (gemm8g.hip).  Requires K % 128 == 0, N % 8 == 0 (SwiGLU: 64), lda % 16 == 0
// (bytes), ldc % 8 == 0, operands at 16 bytes; ws and flags as lwc_gemm8p's, or null: K is not cut then. 
extern "C" int lwc_gemm8p_fp8(const void* A, const void* W, void* C, const float* a_scale, const float* w_scale, const void* a_mx,
                              void* mx_out, int s_rows, float* ws, int* flags, int M, int N, int K, int lda, int ldc, int swiglu, hipStream_t s) {
  using namespace lwc::g8p;
  if (K % 128 != 0 || K < 128 || N % (swiglu ? 64 : 8) != 0 || lda % 16 != 0 || ldc % 8 != 0 || (!a_scale && !a_mx) || !w_scale) return -1;
  if ((long long)M * lda >= (1LL << 31) || 256LL * K >= (1LL << 31) || ldc >= (1 << 26)) return -1;  // 32-bit buffer offsets
  if (swiglu < 0 || swiglu > 2 || (swiglu && a_mx)) return -1;
  if (swiglu == 2 && (N % 256 != 0 || !mx_out || s_rows < M || ldc % 16 != 0)) return -1;
  if (a_mx && (s_rows < M || (long long)(K / 128) * s_rows * 4 >= (1LL << 31))) return -1;
  if (M == 0 || N == 0) return 0;
  Params p{};
  p.A = (const lwc::bf16_t*)A, p.W = (const lwc::bf16_t*)W, p.C = (lwc::bf16_t*)C, p.ws = ws, p.flags = flags;
  p.a_scale = a_scale, p.w_scale = w_scale, p.a_mx = (const uint8_t*)a_mx, p.mx_out = (uint8_t*)mx_out, p.s_rows = s_rows;
  p.M = M, p.N = N, p.K = K / 2, p.lda = lda / 2, p.ldc = ldc;
  const int r1 = plan(p, swiglu);
  if (swiglu == 2) return launch<EPI_FP8_MX_OUT>(p, r1, s);
  if (swiglu) return launch<EPI_FP8_SWIGLU>(p, r1, s);
  return a_mx ? launch<EPI_FP8_MX>(p, r1, s) : launch<EPI_FP8>(p, r1, s);
}
