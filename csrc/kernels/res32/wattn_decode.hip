// Decode rows of the sliding-window attention: the launchers (the kernel is in wattn_decode_kernel.h; the wide
// instantiation is compiled in a file of its own, wattn_decode_wide.hip, with its own code generation flags).
#include "wattn_decode_kernel.h"

// Sizes the decode kernel is built for.  vk: the caller's value pages repeat the first Dv entries of the key rows (a
// latent that is key and value at once); only then does the wide kernel apply (it reads its values from the key rows).
extern "C" int r32_window_attn_decode_ok(int D, int Dv, int vk) {
  const bool small = (D == 32 || D == 64 || D == 128 || D == 192) && (Dv == 32 || Dv == 64 || Dv == 128);
  return small || (vk && ((D == 576 && Dv == 512) || (D == 320 && Dv == 256)));
}

extern "C" int r32_window_attn_decode_wide_launch(const WAttnDecodeParams* p, int D, int gx, int gy, int gz, int chunks_per_group,
                                                  hipStream_t s);

// out[b, h, :] = sum_s exp(m_s - M) o_s / sum_s exp(m_s - M) l_s  (splits that saw no key have l = 0, and no o)
// sink (or null): exp(sink_h) joins the denominator.
// Lane s of every wave weighs split s (S <= 64), so the loop over the splits only has loads that do not wait for one
// another: at 64 splits of one row the step (both kernels) took 59 us with the
// weights formed inside the loop, 26 now.
__global__ void window_attn_reduce_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                          const float* __restrict__ sink, bf16_t* __restrict__ out, int ldo, int H, int S,
                                          int Dv) {
  const int b = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
  float m = -1e30f, l = 0.f;
  if (lane < S) {
    const float* ml = part_ml + (((size_t)b * H + h) * S + lane) * 2;
    m = ml[0];
    l = ml[1];
  }
  const bool seen = l > 0.f;
  const int top = S > 1 ? 1 << (31 - __builtin_clz(S - 1)) : 0;  // (the splits' lanes meet in lane 0: none, where there is one)
  auto first = [](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, x))); };
  float M = seen ? m : -1e30f;
  for (int o = top; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
  M = first(M);
  if (sink) M = fmaxf(M, sink[h]);
  const float w = seen ? expf(m - M) : 0.f;
  float L = seen ? w * l : 0.f;
  for (int o = top; o > 0; o >>= 1) L += __shfl_xor(L, o, 64);
  L = first(L);
  if (sink) L += expf(sink[h] - M);
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  const unsigned long long live = __ballot(seen);
  const int n = live ? 64 - __builtin_clzll(live) : 0;  // splits fill from the first
  const float* po = part_o + ((size_t)b * H + h) * S * Dv;
  const int dv = 2 * threadIdx.x;
  float2 acc = {0.f, 0.f};
  if (dv < Dv)
#pragma unroll 8
    for (int s = 0; s < n; ++s) {
      const float ws = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), s));
      const float2 o = *reinterpret_cast<const float2*>(po + (size_t)s * Dv + dv);
      acc.x += ws != 0.f ? ws * o.x : 0.f;  // (a split without keys has left its row as it was)
      acc.y += ws != 0.f ? ws * o.y : 0.f;
    }
  if (dv < Dv) {
    out[(size_t)b * ldo + (size_t)h * Dv + dv] = f2bf(acc.x * inv);
    out[(size_t)b * ldo + (size_t)h * Dv + dv + 1] = f2bf(acc.y * inv);
  }
}

template <int ND>
int launch_decode_nv(const WAttnDecodeParams& p, int nv, dim3 grid, hipStream_t s) {
  switch (nv) {
    case 2: window_attn_decode_kernel<ND, 2><<<grid, 64, 0, s>>>(p); break;
    case 4: window_attn_decode_kernel<ND, 4><<<grid, 64, 0, s>>>(p); break;
    case 8: window_attn_decode_kernel<ND, 8><<<grid, 64, 0, s>>>(p); break;
    default: return -1;
  }
  return (int)hipGetLastError();
}

// Splits for a decode step of B sequences whose windows hold at most max_keys keys: about 2048 waves (two per SIMD, the
// registers' limit).  Measured, cold, with contexts of 500 to 1500 keys of 128, 8 kv heads: at 64 sequences 2 splits 63 us, 4
// (2048 waves) 67, 6 67, 8 67, 16 72; at 8 sequences of 1000 2 splits 31, 4 22, 8 19, 16 and 32 20.  (1024 waves: 0.82 to 0.98 of the time for
// equal contexts of 128 entries, a step of 64 rows level; up to 1.15 for 100 to 3000 keys, 64 entries up to 1.48.)
// Wide rows (D = 320, 576): workgroups of four waves, about 512 of them, or of eight (more than 16 heads), at most 256 of them
// (one per CU: at 64 sequences of 500 to 1500 keys x 32 heads x 576 / 512 2 / 4 / 8 splits take 81 / 54 / 63 us), at least 128 keys each (their
// partials are large).
extern "C" int r32_window_attn_decode_splits(int B, int G, int Hg, int max_keys, int D) {
  const bool wide = D > 192;
  const int chunks = (Hg + 15) / 16;
  const int waves = B * G * (wide && chunks > 1 ? (chunks + 1) / 2 : chunks);  // wide rows: workgroups
  int s = wide && chunks > 1 ? 256 / waves : ((wide ? 512 : 2048) + waves - 1) / waves;
  const int by_keys = wide ? (max_keys + 32 + 127) / 128 : (max_keys + 32 + 63) / 64;
  if (s > by_keys) s = by_keys;
  if (s > 64) s = 64;
  return s < 1 ? 1 : s;
}

// Head chunks that share a workgroup: two where one wide row serves more than 16 heads.
static int chunks_per_group(int Hg, int D) { return D > 192 && Hg > 16 ? 2 : 1; }

// The lowest and highest of a sequence's heads whose q and bias the decode kernel loads, over all its workgroups and waves.
extern "C" void r32_window_attn_decode_heads(int H, int G, int D, int* lo, int* hi) {
  const int Hg = H / G, nc = chunks_per_group(Hg, D), chunks = (Hg + 15) / 16;
  *lo = H, *hi = -1;
  for (int y = 0; y < G * ((chunks + nc - 1) / nc); ++y)
    for (int cw = 0; cw < nc; ++cw)
      for (int r16 = 0; r16 < 16; ++r16) {
        const int h = loaded_head(head_chunk(y, cw, nc, Hg), r16);
        if (h < *lo) *lo = h;
        if (h > *hi) *hi = h;
      }
}

// part_o: fp32 [B * H * S * Dv], part_ml: fp32 [B * H * S * 2] scratch of the caller.
extern "C" int r32_window_attn_decode(const float* q, const void* k_cache, const void* v_cache, long long kb_stride,
                                      long long vb_stride, int block_size, const int* positions, const int* block_tables,
                                      int bt_width, const float* bias, const float* sink, int window, int chunk, float cap, float* part_o,
                                      float* part_ml, int S, void* out, int ldo, int B, int H, int G, int D,
                                      int Dv, int vk, hipStream_t s) {
  if (B <= 0) return 0;
  if (!r32_window_attn_decode_ok(D, Dv, vk) || H % G != 0 || S < 1 || (block_size & (block_size - 1)) != 0) return -1;
  WAttnDecodeParams p;
  p.q = q; p.k_cache = (const bf16_t*)k_cache; p.v_cache = (const bf16_t*)v_cache; p.kb_stride = kb_stride;
  p.vb_stride = vb_stride; p.block_size = block_size; p.positions = positions; p.block_tables = block_tables;
  p.bs_shift = -1;
  for (int b = 0; b < 20; ++b)
    if ((1 << b) == block_size) p.bs_shift = b;
  p.bt_width = bt_width; p.bias = bias; p.window = window; p.chunk = chunk; p.cap = cap; p.part_o = part_o; p.part_ml = part_ml; p.H = H; p.G = G;
  p.S = S;
  p.min_keys = D > 192 ? 128 : 64;
  const int Hg = H / G;
  const dim3 grid(B, G * ((Hg + 15) / 16), S);
  int rc = -1;
  if (D > 192) {  // one wide row for all heads: a low-rank attention's cached latent + rotated part
    const int chunks = (Hg + 15) / 16, nc = chunks_per_group(Hg, D);
    rc = r32_window_attn_decode_wide_launch(&p, D, B, G * ((chunks + nc - 1) / nc), S, nc, s);
  } else {
    switch (D / 32) {
      case 1: rc = launch_decode_nv<1>(p, Dv / 16, grid, s); break;
      case 2: rc = launch_decode_nv<2>(p, Dv / 16, grid, s); break;
      case 4: rc = launch_decode_nv<4>(p, Dv / 16, grid, s); break;
      case 6: rc = launch_decode_nv<6>(p, Dv / 16, grid, s); break;
    }
  }
  if (rc != 0) return rc;
  window_attn_reduce_kernel<<<dim3(B, H), Dv <= 128 ? 64 : Dv / 2, 0, s>>>(part_o, part_ml, sink, (bf16_t*)out, ldo, H, S, Dv);
  return (int)hipGetLastError();
}
