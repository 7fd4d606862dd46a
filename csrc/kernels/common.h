// Shared device helpers for the gfx950 (CDNA4, MI355X) kernels of llm_weighted_consensus_amd.
//
// Conventions used by every kernel in csrc/kernels:
//   * wave64 everywhere: lane = threadIdx.x & 63, block sizes are multiples of 64;
//   * bf16 is carried as raw uint16 bits in memory and widened to f32 in registers;
//     loads/stores are 16 B per lane (8 bf16) wherever the row length allows it;
//   * every launcher takes a hipStream_t so the torch binding layer can put the kernel
//     on the caller's current stream (and hence inside a captured hipGraph).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>
#include <type_traits>

#define LWC_HOST_DEVICE __host__ __device__ __forceinline__
#define LWC_DEVICE __device__ __forceinline__

namespace lwc {

typedef uint16_t bf16_t;
typedef short short8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

LWC_DEVICE float bf2f(bf16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

// Round-to-nearest-even f32 -> bf16 (NaN stays NaN: hipcc lowers this to v_cvt_pk_bf16_f32).
LWC_DEVICE bf16_t f2bf(float f) {
  __hip_bfloat16 b = __float2bfloat16(f);
  return *reinterpret_cast<bf16_t*>(&b);
}

// (As one conversion of a pair: put together from two single ones, of which the compiler makes each an instruction, a shift and an or, a
// pair took four instructions instead of one.)
LWC_DEVICE uint32_t pack_bf16x2(float lo, float hi) {
  typedef float float2v __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(float2v{lo, hi}, bf16x2));
}

// 16-byte vector of 8 bf16 <-> 8 floats.
LWC_DEVICE void unpack8(const uint4v& v, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(v[i] << 16);
    f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
  }
}
LWC_DEVICE uint4v pack8(const float (&f)[8]) {
  uint4v v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack_bf16x2(f[2 * i], f[2 * i + 1]);
  return v;
}
// f as hi + lo, each rounded to bf16
LWC_DEVICE void split8(const float (&f)[8], short8& hi, short8& lo) {
  const uint4v h = pack8(f);
  float r[8];
  unpack8(h, r);
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = f[e] - r[e];
  hi = __builtin_bit_cast(short8, h);
  lo = __builtin_bit_cast(short8, pack8(r));
}

LWC_DEVICE float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
LWC_DEVICE float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Block-wide sum for blockDim.x <= 1024; `scratch` must hold >= 16 floats.
LWC_DEVICE float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = lane < nw ? scratch[lane] : 0.f;
  return wave_sum(r);
}
LWC_DEVICE float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = lane < nw ? scratch[lane] : -INFINITY;
  return wave_max(r);
}

// Weights that a call reads once, in one tile of rows, are loaded with the nt bit where there are at least 32 MiB of them: a model of
// such layers does not stay in the last-level cache (256 MiB) from one call to the next, and loads that claim no place there run at up
// to 6.6 TB/s instead of 5.9.  us, without / with it, weights from memory: gemm1s 61 x 28672 x 4096 42.3 / 39.3, 4096 x 4096 (32 MiB) 11.7
// / 11.0; gemm2w 16 x 128256 x 4096 182 / 158 (more rows: past_caches there), 61 x 4096 x 14336 26.9 / 25.1; gemm2s 8 x 16 rows x 14336 x
// 4096 166 / 152; gemm2g bf16 [4096, 7168] x 8 of 16 rows 79 / 70, fp8 [28672, 4096] x 8 of 16 and 128 rows 158 / 139 and 187 / 184, [4096,
// 14336] x 8 of 128 108 / 94.
// A second tile of rows then reads from memory too (gemm2w 1000 x 128256 x 4096 1019 / 1420, gemm2g fp8 8 x 250 rows x 28672 x 4096 313 / 402), so a
// group of several tiles takes its weights through the caches among others that do not.  us, without / with it for all / for groups of
// one tile, 28672 x 4096 fp8, 8 groups: 210, 205, 200, 198, 90, 60, 40, 20 rows 236 / 277 / 231, two of 300 among 20s 228 / 246 / 216; bf16
// 14336 x 4096 245 / 285 / 244 and 229 / 254 / 218, 4096 x 14336 331 / 343 / 311 and 283 / 302 / 278.
// Weights that would have been in the cache lose: 24 MiB of 3072 x 1024 4 %, a single 10240 x 8192 called again and again 46 / 73.  Partial
// reads of a line too (skinny.hip, 1 x 128256 x 4096 163 / 180).
constexpr int kNT = 2;  // a buffer load's nt bit
constexpr int weights_pass(long long bytes) { return bytes >= 32LL << 20; }

// x Phi(x), the erf form of GELU, as max(x, 0) - |x| Phi(-|x|), with log2 Phi(-a) a polynomial over 0 <= a <= 5.6 (least squares at
// Chebyshev nodes, weights moved towards the minimax of |x| times the error; beyond 5.6 the last term stays at 6e-8).  One exp2 and
// eleven other instructions per element, where erf by Abramowitz & Stegun 7.1.26 took one exp, one rcp and fourteen: a tile of 256 x
// 256 spends 0.4 us on each.  Error in fp32 arithmetic over N(0, 1) and a grid of [-6, 6]: at most 2.4e-7, rms 8.6e-8 (with erf
// 4.7e-7 and 8.8e-8), and of the value at most 2.2e-5 for |x| < 4 (with erf 9.3e-4).  NaN stays NaN (minimum, not min).
LWC_DEVICE float gelu_erf(float x) {
  const float a = __builtin_elementwise_minimum(fabsf(x), 5.6f);
  float l = fmaf(-1.437473542864609e-06f, a, 5.503627471625805e-05f);
  l = fmaf(l, a, -0.0008901672554202378f);
  l = fmaf(l, a, 0.008395220153033733f);
  l = fmaf(l, a, -0.05382503569126129f);
  l = fmaf(l, a, -0.45850393176078796f);
  l = fmaf(l, a, -1.1512768268585205f);
  l = fmaf(l, a, -0.9999866485595703f);
  return fmaf(-a, __builtin_amdgcn_exp2f(l), fmaxf(x, 0.f));
}

// Reductions over the 4 lanes {l, l^16, l^32, l^48} holding one query row's tokens: two VALU
// half-swaps (v_permlane32_swap / v_permlane16_swap, gfx950) instead of LDS ds_bpermute round trips.
LWC_DEVICE float row_max4(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
LWC_DEVICE float row_sum4(float v) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}


// A buffer resource built from explicitly wave-uniform parts (readfirstlane of the base address and the
// size).  Built straight from kernel arguments / tile indices, the compiler sometimes cannot prove the
// resource uniform and wraps EVERY buffer access through it in a readfirstlane "waterfall" loop (~10
// instructions and a branch per access, inside GEMM main loops too).
// e8m0 exponent of an MX block with max |x| = amax: the smallest e with amax * 2^-e <= 448 (e4m3's largest
// finite), from amax's own exponent and mantissa (448 = 0.875 * 2^9), so no rounding pushes a value past 448
LWC_DEVICE int mx_exp(float amax) {
  const int ea = __builtin_amdgcn_frexp_expf(amax);
  const float m = __builtin_amdgcn_frexp_mantf(amax);
  return min(127, max(-127, ea - 9 + (m > 0.875f ? 1 : 0)));
}

// max over each 16-lane DPP row (quad xor 1, quad xor 2, half-row mirror, row mirror)
LWC_DEVICE float row16_max(float x) {
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, false)));
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, false)));
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xF, 0xF, false)));
  return fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x140, 0xF, 0xF, false)));
}

// sum over each 16-lane DPP row, the same way
LWC_DEVICE float row16_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, false));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xF, 0xF, false));
  return x + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x140, 0xF, 0xF, false));
}

LWC_DEVICE __amdgpu_buffer_rsrc_t uniform_rsrc(const void* base, int bytes) {
  const uint64_t a = (uint64_t)base;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), (short)0,
                                           __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// Bijective XCD-aware remap of a linear workgroup id (cdna_hip_programming.md §5 "XCD swizzle
// must be bijective"): consecutive remapped ids land on the same XCD so neighbouring tiles share L2.
LWC_DEVICE int xcd_remap(int orig, int nwg) {
  const int q = nwg / 8, r = nwg % 8, xcd = orig % 8;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + orig / 8;
}

// ---- rows of different lengths over the CUs ----
// The place of workgroup w of n among the items sorted by work, most first, so that every CU gets about as much.  Workgroup w
// starts on CU w % 256 as long as that has room: the rounds of 256 that are resident walk the order back and forth, the last
// one forwards; after them the next longest goes to the CU that is done first.
LWC_DEVICE int ranked_place(int w, int n, int rounds) {
  const int k = w / 256, resident = min((n + 255) / 256, rounds);
  return k < resident && ((resident - 1 - k) & 1) ? 256 * k + 255 - w % 256 : w;
}

// The row of rank `rank` among rows 0 .. B - 1 (0: the largest key(i); equal ones in their order), found bit by bit of the keys
// (0 .. max_key; larger ones count as that) from ballots: each wave for itself, without a sort, a barrier or LDS, 0.3 us.  Beyond
// 64 rows the n = ceil(B / 64) sets of every n-th one are ranked each for itself and take turns, the order of all but for
// neighbours (with all of them at once, two and more keys a lane, the decode attention spilled 43 registers).  from: the lane
// whose key it is, so that what the key is made of need not be read again.
template <typename Key>
LWC_DEVICE int ranked_row(int B, int rank, int lane, int max_key, Key key_of, int& from) {
  const int n = (B + 63) / 64, set = rank % n, i = set + n * lane;
  rank /= n;
  const int key = i < B ? min(key_of(i), max_key) : 0;
  unsigned long long mask = __ballot(i < B);
  for (int bit = __ballot(key >> 4) ? 31 - __clz(max_key) : 3; bit >= 0; --bit) {
    const unsigned long long ones = __ballot((key >> bit) & 1) & mask;
    const int c = __popcll(ones);
    const bool in = rank < c;
    rank -= in ? 0 : c;
    mask = in ? ones : mask & ~ones;
  }
  const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
  from = (int)__builtin_ctzll(__ballot(((mask >> lane) & 1) && below == rank));
  return set + n * from;
}

}  // namespace lwc

#define LWC_CHECK_LAUNCH() (void)hipGetLastError()
