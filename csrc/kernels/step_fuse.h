// What the projections of a decode step of few rows do besides their product, so that no kernel runs between them and
// the attention (csrc/kernels/skinny.hip, gemm2w.hip, gemm1s.hip): a kernel of a few rows takes 4 to 5 us however little it does.
//
//   * RMSNorm whose weight is folded into the projection behind it: rmsnorm(x) W^T = (x W^T) / rms(x), so the projection
//     that writes the residual stream leaves the sums of squares of its columns and the next one scales its rows;
//   * RoPE of k and the paged cache's rows: the qkv projection holds both halves of a head in one tile, rotates them and
//     writes k and v where the attention reads them (q leaves un-rotated: the attention rotates it as it loads it).
//
// Measured (us, weights from memory): qkv 6144 x 4096 behind a norm and in front of a RoPE kernel, 4.7 each: 1 row 13.0 -> 14.1
// with both, 16 rows 18.4 -> 15.9, 61 rows 17.4 -> 19.9; gate|up 28672 x 4096 behind a norm, 61 rows 53 -> 54.3; the residual
// projections, whose partials the norm is made of, unchanged.
#pragma once
#include "common.h"
#include "step_fuse_args.h"

namespace lwc {

// A row's slot and the angles of n columns of a k head, read ahead of the product (behind it, one after the other, they
// held the finished tile back).
template <int n>
struct RopeAhead {
  int slot, position;
  float cs[n], sn[n];
};
template <int n>
LWC_DEVICE void rope_kv_row(const RopeKV& r, RopeAhead<n>& a, int row, int h) {
  if (h < r.Hq) return;
  a.slot = r.slots[row];
  a.position = r.positions[row];
}
template <int n>
LWC_DEVICE void rope_kv_angles(const RopeKV& r, RopeAhead<n>& a, int h, int c) {
  if (h < r.Hq || h >= r.Hq + r.Hkv) return;
  const size_t at = (size_t)a.position * (r.D / 2) + c;
  typedef float vec __attribute__((ext_vector_type(n < 4 ? n : 4)));
#pragma unroll
  for (int e = 0; e < n; e += 4) {
    *reinterpret_cast<vec*>(a.cs + e) = *reinterpret_cast<const vec*>(r.cos + at + e);
    *reinterpret_cast<vec*>(a.sn + e) = *reinterpret_cast<const vec*>(r.sin + at + e);
  }
}

// where a slot's row of v head h begins; entry c lies at 4 c
LWC_DEVICE bf16_t* rope_v_row(const RopeKV& r, int slot, int h) {
  const size_t blk = slot / r.BS;
  const int off = slot % r.BS;
  return r.vc + (blk * r.Hkv + (h - r.Hq - r.Hkv)) * r.BS * r.D + (size_t)(off >> 2) * r.D * 4 + (off & 3);
}

// n consecutive columns of a row in each half of head h (q heads, k heads, v heads): x at column c, y at c + D / 2.  q goes
// to C as it is; k, rounded to bf16 as a projection of its own would round it, is rotated and cached; v is cached.
template <int n>
LWC_DEVICE void rope_kv_store(const RopeKV& r, const RopeAhead<n>& ahead, bf16_t* C, int ldc, int row, int h, int c,
                              const float (&x)[n], const float (&y)[n]) {
  typedef uint32_t vec __attribute__((ext_vector_type(n / 2)));
  const int half = r.D / 2;
  auto put = [](bf16_t* dst, const float (&v)[n]) {
    vec o;
#pragma unroll
    for (int e = 0; e < n / 2; ++e) o[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
    *reinterpret_cast<vec*>(dst) = o;
  };
  if (h < r.Hq) {
    bf16_t* dst = C + (size_t)row * ldc + h * r.D + c;
    put(dst, x);
    put(dst + half, y);
    return;
  }
  if (ahead.slot < 0) return;
  const size_t blk = ahead.slot / r.BS;
  const int off = ahead.slot % r.BS;
  if (h < r.Hq + r.Hkv) {
    float a[n], b[n];
#pragma unroll
    for (int e = 0; e < n; ++e) {
      const float x1 = bf2f(f2bf(x[e])), x2 = bf2f(f2bf(y[e]));
      a[e] = x1 * ahead.cs[e] - x2 * ahead.sn[e];
      b[e] = x2 * ahead.cs[e] + x1 * ahead.sn[e];
    }
    bf16_t* dst = r.kc + ((blk * r.Hkv + (h - r.Hq)) * r.BS + off) * r.D + c;
    put(dst, a);
    put(dst + half, b);
    return;
  }
  bf16_t* dst = rope_v_row(r, ahead.slot, h) + 4 * c;
#pragma unroll
  for (int e = 0; e < n; ++e) {
    dst[4 * e] = f2bf(x[e]);
    dst[4 * (e + half)] = f2bf(y[e]);
  }
}

}  // namespace lwc
