// Grouped fp8 and bf16 GEMM of few rows per group (gfx950): the calls of the 256-row kernel (gemm8g.hip: the same operands, epilogues
// and MX form) while the weights, not the matrix cores, bound them.
//
// That kernel keeps one workgroup per CU with 32 KiB of weights on their way, and hands its CU over with nothing in
// flight: the experts of a decode step read their weights at 2.7 to 3.6 TB/s.  Here a tile is 64, 128 or 192 rows of a group
// by 128 weight rows, as in gemm2w.hip (LDS layout and operand order are the same): two workgroups per CU, each with three (64
// rows) or two steps of 128 bytes of every row in flight.  Rows past the group's end are neither loaded nor multiplied.
// (192 rows of an A with MX scales need 82 KiB: those workgroups have a CU to themselves, and gemm8g.hip
// sends none here that would need a second round.)
// More steps in flight for calls that give a CU one workgroup (six, five, four) gain nothing and cost dear where a second round
// follows, us, so / here: fp8, 8 experts of 16 rows [4096, 8192] (256 workgroups) 66 / 65, [4608, 8192] (288) 89 / 77; dense
// 700 rows x 6144 x 4096 (288) 50 / 31.
// Measured, 8 experts, us, 256-row kernel (in four phases per K tile; in its two some 6 % less) -> here ([28672, 4096] SwiGLU to MX, [4096, 14336] from MX; 154
// and 77 at the rate of a plain read): 4 rows an expert 257 -> 182, 144 -> 81; 32 rows 259 -> 189, 145 -> 84; 64 rows 264 -> 200, 150 -> 90; 128 rows
// 270 -> 217, 155 -> 115.  Dense calls of few tiles likewise: 512 rows x 4096 x K 4096 from MX 45 -> 21.
// bf16, 8 experts of 16 rows: [14336, 4096] 194 (the 128-row kernel with split K, its clear and its conversion 204), [4096, 7168] 82
// (103).
#include <algorithm>

#include "common.h"

namespace lwc {
namespace g2g {

typedef int v8i32 __attribute__((ext_vector_type(8)));

constexpr int kPlain = 0, kSwiglu = 1, kMxOut = 2, kMxA = 3, kBf16 = 4, kBf16Swiglu = 5;  // as in gemm8g.hip

struct Params {
  const uint8_t* A;      // [rows_a, lda] e4m3 or bf16 (lda, K in bytes)
  const uint8_t* W;      // [G][N, K]
  bf16_t* C;
  const int* row_off;
  const int* a_rows;
  const float* a_scale;
  const float* w_scale;
  int G, N, K, lda, ldc, rows_a, rows;
  int slots, n_tiles;
  const uint8_t* a_mx;
  uint8_t* mx_out;
  int s_rows;
  int turned;  // a tile's walk over K starts at a step of its own
};

LWC_DEVICE float4v mfma8(const uint4v& a0, const uint4v& a1, const uint4v& b0, const uint4v& b1, const float4v& c, int sb) {
  const v8i32 av = {(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w, (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
  const v8i32 bv = {(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w, (int)b1.x, (int)b1.y, (int)b1.z, (int)b1.w};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 0, 0, 0, 127, 0, sb);
}
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
LWC_DEVICE float4v mfma16(const uint4v& a, const uint4v& b, const float4v& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
LWC_DEVICE float silu8(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }
template <int CP = 0>
LWC_DEVICE void dma16(const __amdgpu_buffer_rsrc_t& r, uint8_t* dst, uint32_t vo, int so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, vo, so, 0, CP);
}
LWC_DEVICE void dma4(const __amdgpu_buffer_rsrc_t& r, uint8_t* dst, uint32_t vo, int so) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, vo, so, 0, 0);
}
template <int N>
LWC_DEVICE void wait_rows() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// all but the last n steps' loads (n < NST of S each), and all LDS reads
template <int S, int NST>
LWC_DEVICE void wait_steps(int n) {
  if constexpr (NST > 1) {
    if (n >= NST - 1) {
      wait_rows<(NST - 1) * S>();
      return;
    }
    wait_steps<S, NST - 1>(n);
  } else {
    wait_rows<0>();
  }
}

// NT: the weights of groups of one tile pass the caches by (weights_pass, common.h).
template <int MODE, int TM, int NST, bool NT>
__global__ void __launch_bounds__(256, 2) gemm2g_kernel(const Params p) {
  constexpr bool MXA = MODE == kMxA, BF = MODE == kBf16 || MODE == kBf16Swiglu;
  constexpr int TN = 128, kA = TM * 128, kS = kA + TN * 128, kStage = kS + (MXA ? 1024 : 0);  // rows, weights, scales
  constexpr int IA = TM / 32, IW = TN / 32, MI = TM / 32;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, q = lane >> 4, wr = wid >> 1, wc = wid & 1;

  // XCD x owns weight tiles x, x + 8, ... and walks all of them for one row tile before the next: the row tiles of an expert
  // read its weights from that XCD's L2
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, nj = (p.n_tiles + 7) / 8;
  const int ntile = local % nj * 8 + xcd;
  if (ntile >= p.n_tiles) return;
  int slot = local / nj, g = 0, m_begin = 0, m_end = 0;
  bool once = false;  // the weights are read by this tile alone
  for (; g < p.G; ++g) {
    const int r0 = p.row_off ? p.row_off[g] : 0, r1 = p.row_off ? p.row_off[g + 1] : p.rows, nt = (r1 - r0 + TM - 1) / TM;
    if (slot < nt) {
      m_begin = r0 + slot * TM;
      m_end = min(r1, m_begin + TM);
      once = nt == 1;
      break;
    }
    slot -= nt;
  }
  if (g >= p.G) return;  // a slot that the routing left over
  const int n0 = ntile * TN;

  uint32_t voA[IA], voW[IW];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int row = (i * 4 + wid) * 8 + (lane >> 3), r = m_begin + row;
    voA[i] = r < m_end ? (uint32_t)((p.a_rows ? p.a_rows[r] : r) * p.lda + (((lane & 7) ^ ((row >> 1) & 7)) << 4)) : 0x7fffffffu;
  }
  const int rows_n = min(p.N - n0, TN);
#pragma unroll
  for (int i = 0; i < IW; ++i) {
    const int row = (i * 4 + wid) * 8 + (lane >> 3);
    voW[i] = row < rows_n ? (uint32_t)(row * p.K + (((lane & 7) ^ ((row >> 3 & 3) * 2 + (row >> 1 & 1))) << 4)) : 0x7fffffffu;
  }
  const __amdgpu_buffer_rsrc_t rA = uniform_rsrc(p.A, p.rows_a * p.lda);
  const __amdgpu_buffer_rsrc_t rW = uniform_rsrc(p.W + ((size_t)g * p.N + n0) * p.K, rows_n * p.K);
  // kMxA: the rows' scales of a step, four bytes (its blocks of 32) a row
  const uint32_t voS = m_begin + tid < m_end ? (uint32_t)((m_begin + tid) * 4) : 0x7fffffffu;
  const __amdgpu_buffer_rsrc_t rS = uniform_rsrc(p.a_mx, MXA ? (p.K / 128) * p.s_rows * 4 : 0);
  const int nk = p.K / 128, live = m_end - m_begin;
  const int k0 = p.turned ? (int)((unsigned)(3 * (ntile >> 3) + 15 * g) % (unsigned)nk) : 0;
  auto stage = [&](uint8_t* buf, int step, auto policy) {
    const int kt = step + k0 < nk ? step + k0 : step + k0 - nk;
#pragma unroll
    for (int i = 0; i < IA; ++i) dma16(rA, buf + (i * 4 + wid) * 1024, voA[i], kt * 128);
#pragma unroll
    for (int i = 0; i < IW; ++i) dma16<decltype(policy)::value>(rW, buf + kA + (i * 4 + wid) * 1024, voW[i], kt * 128);
    if constexpr (MXA) dma4(rS, buf + kS + wid * 256, voS, kt * p.s_rows * 4);
  };
  // the wave's row tiles are every other one, so that the rows a short group has divide between the waves
  const int pos0 = (q ^ (r16 >> 1)) << 4, pos1 = pos0 ^ 64;
  const int offA = (wr * 16 + r16) * 128;
  const int offW = kA + (wc * 64 + 8 * (r16 >> 2) + (r16 & 3)) * 128;
  int src_row[MI];  // the lane's rows (past the end: the tile's first)
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m_begin + (2 * i + wr) * 16 + r16;
    src_row[i] = m < m_end ? m : m_begin;
  }
  float4v acc[MI][2][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[i][c][h] = float4v{0.f, 0.f, 0.f, 0.f};

  // (a walk over K of its own for either: with a branch in each step 1 x 4096 x 14336 48.4 -> 49.9 us)
  auto walk = [&](auto policy) {
#pragma unroll
    for (int k = 0; k < NST; ++k)
      if (k < nk) stage(smem + k * kStage, k, policy);
    int at = 0;
    for (int kt = 0; kt < nk; ++kt) {
      uint8_t* buf = smem + at;
      at = at == (NST - 1) * kStage ? 0 : at + kStage;
      wait_steps<IA + IW + (MXA ? 1 : 0), NST>(nk - 1 - kt);  // this step's rows have landed, later ones may be in flight
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      uint4v a[2][MI], w[2][2][2];
      int sc[MI];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int pos = s ? pos1 : pos0;
#pragma unroll
        for (int i = 0; i < MI; ++i) a[s][i] = *reinterpret_cast<const uint4v*>(buf + offA + pos + i * 4096);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int h = 0; h < 2; ++h) w[s][c][h] = *reinterpret_cast<const uint4v*>(buf + offW + pos + c * 4096 + h * 512);
      }
      if constexpr (MXA) {
#pragma unroll
        for (int i = 0; i < MI; ++i) sc[i] = buf[kS + ((2 * i + wr) * 16 + r16) * 4 + q];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();  // every wave holds the step's operands: its buffer takes a later step
      asm volatile("" ::: "memory");
      if (kt + NST < nk) stage(buf, kt + NST, policy);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < MI; ++i)
        if ((2 * i + wr) * 16 < live) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              if constexpr (BF) acc[i][c][h] = mfma16(w[1][c][h], a[1][i], mfma16(w[0][c][h], a[0][i], acc[i][c][h]));
              else acc[i][c][h] = mfma8(w[0][c][h], w[1][c][h], a[0][i], a[1][i], acc[i][c][h], MXA ? sc[i] : 127);
            }
        }
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (NT) {
    if (once) walk(std::integral_constant<int, kNT>{});
    else walk(std::integral_constant<int, 0>{});
  } else {
    walk(std::integral_constant<int, 0>{});
  }

  const int col0 = n0 + wc * 64 + 8 * q;
  float ws[2][8];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) ws[c][e] = !BF && col0 + 32 * c < p.N ? p.w_scale[(size_t)g * p.N + col0 + 32 * c + e] : 0.f;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m_begin + (2 * i + wr) * 16 + r16;
    const float as = MXA || BF ? 1.f : p.a_scale[p.a_rows ? p.a_rows[src_row[i]] : src_row[i]];
    float x[2][8];
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[c][e] = BF ? acc[i][c][e >> 2][e & 3] : acc[i][c][e >> 2][e & 3] * (as * ws[c][e]);
    if constexpr (MODE == kPlain || MODE == kMxA || MODE == kBf16) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
        if (m < m_end && col0 + 32 * c < p.N) *reinterpret_cast<uint4v*>(p.C + (size_t)m * p.ldc + col0 + 32 * c) = pack8(x[c]);
    } else {  // the wave's first 32 columns are gate, the other 32 the matching up columns
      const int col = (n0 + wc * 64) / 2 + 8 * q;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = silu8(x[0][e]) * x[1][e];
      const uint4v packed = pack8(y);
      if constexpr (MODE == kSwiglu || MODE == kBf16Swiglu) {
        if (m < m_end && col < p.N / 2) *reinterpret_cast<uint4v*>(p.C + (size_t)m * p.ldc + col) = packed;
      } else {  // e4m3 rows, one e8m0 scale per row and block of 32: four lanes hold a block
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
          if (q == 0) p.mx_out[((size_t)(col >> 7) * p.s_rows + m) * 4 + (col >> 5 & 3)] = (uint8_t)(e + 127);
        }
      }
    }
  }
}

template <int MODE, int TM, int NST, bool NT>
int launch(Params p, int rows, hipStream_t s) {
  constexpr int kLds = NST * ((TM + 128) * 128 + (MODE == kMxA ? 1024 : 0));
  static_assert(2 * kLds <= 160 * 1024 || (MODE == kMxA && TM == 192), "two workgroups share a CU's LDS");
  static const hipError_t attr =
      hipFuncSetAttribute((const void*)gemm2g_kernel<MODE, TM, NST, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  (void)attr;
  p.slots = (rows + TM - 1) / TM + p.G;
  p.n_tiles = (p.N + 127) / 128;
  const long long grid = 8LL * ((p.n_tiles + 7) / 8) * p.slots;
  if (grid >= (1LL << 31)) return -1;
  gemm2g_kernel<MODE, TM, NST, NT><<<(unsigned)grid, 256, kLds, s>>>(p);
  return (int)hipGetLastError();
}

}  // namespace g2g
}  // namespace lwc

extern "C" int lwc_gemm2s(const void*, const void*, void*, const int*, const int*, int, int, int, int, int, int, int, int, hipStream_t);

// bf16 weights whose rows lie 8 KiB or a multiple apart, as many tiles of 256 columns as fill their rounds of 256 CUs: gemm2s.hip's
// weight streams.  us, here / there, uneven groups, N x K x groups of 3 / 16 / 40 / 100 rows: 14336 x 4096 x 8 (1.75 rounds) 184 /
// 153, 195 / 162, 196 / 171, 208 / 207; 4096 x 4096 x 32 (2) 213 / 189, 210 / 187, 215 / 201, 239 / 316; 28672 x 8192 x 2 (0.88) 211 / 168, 208 /
// 167, 203 / 184, 207 / 235; 28672 x 4096 x 8 (3.5) 365 / 355, 361 / 358, 372 / 376, 388 / 440; 3072 x 4096 x 64 (3) 296 / 278, 304 / 307, 316
// / 314; but 22016 x 4096 x 4 (1.34) 150 / 161, and with other K 8192 x 7168 x 8 159 / 159, 4096 x 7168 x 8 (0.5) 71 / 95, 5632 x 2048 x
// 64 262 / 288
// Rows of a tile there, 0 for the small tiles (K in bytes).
extern "C" int lwc_gemm2s_rows(int rows, int G, int N, int K) {
  const int per = (rows + G - 1) / G;
  const long long wide = (long long)((N + 255) / 256) * G, rounds = (wide + 255) / 256;
  if (K % 8192 != 0 || per > 48 || 20 * wide < 17 * 256 * rounds) return 0;
  return per > 16 ? 192 : 64;
}

// The operands of lwc_gemm8g_fp8 (checked there), row_off null for a dense call, or of lwc_gemm8g_bf16 (K and lda in bytes);
// mode 3: A carries MX scales; 4, 5: bf16.  rows: all groups' rows.
extern "C" int lwc_gemm2g(const void* A, const void* W, void* C, const int* row_off, const int* a_rows,
                              const float* a_scale, const float* w_scale, int G, int N, int K, int lda, int ldc, int rows_a,
                              int rows, int mode, const void* a_mx, void* mx_out, int s_rows, hipStream_t s) {
  using namespace lwc::g2g;
  if ((!row_off && G != 1) || K % 128 != 0 || K < 128 || N % 8 != 0 || rows <= 0) return -1;
  Params p{(const uint8_t*)A, (const uint8_t*)W, (lwc::bf16_t*)C, row_off, a_rows, a_scale, w_scale, G, N, K, lda, ldc, rows_a,
                 rows, 0, 0, (const uint8_t*)a_mx, (uint8_t*)mx_out, s_rows, 0};
  // The tile that most groups' rows fit, with room for an uneven routing: a second tile reads the weights again, and where the
  // columns give every CU a workgroup already some CUs walk K once more.  us at 64 / 128 / 192 rows a tile, 32 rows a group: bf16
  // [4096, 14336] x 8 (256 columns) 164 / 166 / 172, one expert with four times the rows 238 / 190 / 193, with 130 rows 254 /
  // 292 / 193; two workgroups a CU, fp8 [4096, 6400] x 16 (512) at 40 rows 79 / 80 / 80, one with twice the rows 96 / 82 / 82
  // (256-row kernel 86).  Fewer columns, where a second tile finds an idle CU: fp8 [2048, 7168] x 8 (128) at 40 rows 34 / 40 / 44, twice
  // 34 / 42 / 46.  More, where it is one of many: bf16 [14336, 4096] x 8 (896) 204 / 203 / 205, four times 190 / 193 / 202.
  // Dense (no table): tiles of 64 rows while they give a CU two workgroups at most, else of 128.
  const int per = (rows + G - 1) / G;
  const long long nt = (N + 127) / 128, cols = nt * G;
  // 128 rows of a stride whose low bits are zero lie on few memory channels, and all tiles walk K in step: starting each tile's
  // walk at another step of K spreads them.  fp8, 8 experts, us, before -> after: [28672, 4096] to MX at 64 / 128 / 160 rows 203 /
  // 214 / 221 -> 170 / 186 / 198, [4096, 8192] at 176 74 -> 71; odd multiples of 2048 bytes gain nothing (14336: 82 / 94 -> 85 / 95).
  // With many rows the tiles of a row tile no longer share its rows' way through L2: what an XCD's 64 workgroups have in use, the
  // rows of so many groups, has to fit its 4 MiB, unless every workgroup has a CU to itself.
  // bf16 experts walk K from its start: the next layer's router reads their sums, and in another order of them rows whose second
  // and third expert nearly tie change experts (2 of 1280 rows behind one such layer; one moved by a tenth of its norm), for
  // [14336, 4096] x 8 of 8 rows at 199 us instead of 165.  fp8 rows are rounded to e4m3 in front of every product, which moves
  // them more than an order does.
  const long long nj = (nt + 7) / 8, groups = std::min<long long>(G, (64 + nj - 1) / nj);
  p.turned = mode != kBf16 && mode != kBf16Swiglu && (K % 4096 == 0 || K % 2048 != 0) &&
             ((groups * per * K <= 4 << 20 && per <= (K <= 4096 ? 160 : 144)) || (row_off && cols <= 256 && per <= 192));
  if ((mode == kBf16 || mode == kBf16Swiglu) && row_off)
    if (const int rt = lwc_gemm2s_rows(rows, G, N, K)) {
      const int rc = lwc_gemm2s(A, W, C, row_off, a_rows, G, N, K, lda, ldc, rows_a, mode == kBf16Swiglu, rt, s);
      if (rc != -1) return rc;
    }
  int tm = per <= (cols <= 128 ? 44 : 16) ? 64 : per <= 104 && !(cols > 128 && cols <= 256) ? 128 : 192;
  if (!row_off) tm = nt * ((rows + 63) / 64) <= 512 ? 64 : 128;
  // (160 rows a group on average: with more, 180 or 192 in each group, gate|up loses 1.5 % by it)
  const bool past = per <= (row_off ? 160 : tm) && lwc::weights_pass((long long)G * N * K);
#define LWC_G2G(M) \
  case M:          \
    if (past) return tm == 64 ? launch<M, 64, 3, true>(p, rows, s) : tm == 128 ? launch<M, 128, 2, true>(p, rows, s) : launch<M, 192, 2, true>(p, rows, s); \
    return tm == 64 ? launch<M, 64, 3, false>(p, rows, s) : tm == 128 ? launch<M, 128, 2, false>(p, rows, s) : launch<M, 192, 2, false>(p, rows, s);
  switch (mode) {
    LWC_G2G(kPlain)
    LWC_G2G(kSwiglu)
    LWC_G2G(kMxOut)
    LWC_G2G(kMxA)
    LWC_G2G(kBf16)
    LWC_G2G(kBf16Swiglu)
  }
#undef LWC_G2G
  return -1;
}
