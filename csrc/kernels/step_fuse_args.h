// The operands of step_fuse.h, for the launchers and the binding layer alike.
#pragma once
#include <cstdint>

namespace lwc {

// ss [M, P] fp32: partial sums of squares of the rows (P % 4 == 0, rows 16-byte aligned)
struct RowSumsq {
  float* ss = nullptr;
  int P = 0;
  float eps = 0.f;
};

// K cache [NB, Hkv, BS, D], V cache [NB, Hkv, BS / 4, D, 4]; slots[row] < 0: the row is not cached
struct RopeKV {
  const int* positions = nullptr;
  const int* slots = nullptr;
  const float* cos = nullptr;  // [max_pos, D / 2]
  const float* sin = nullptr;
  uint16_t* kc = nullptr;
  uint16_t* vc = nullptr;
  int Hq = 0, Hkv = 0, D = 0, BS = 0;
};

inline bool rope_kv_ok(const RopeKV& r, int N) {
  return r.positions && r.slots && r.cos && r.sin && r.kc && r.vc && r.D % 64 == 0 && r.D > 0 && r.BS % 4 == 0 && r.BS > 0 &&
         r.Hq > 0 && r.Hkv > 0 && (r.Hq + 2 * r.Hkv) * r.D == N;
}

}  // namespace lwc
