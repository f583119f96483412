// Shapes of the table of Green's functions (bubble.h): which frequencies and grains a
// pass holds, and how many bytes the table takes.  Host arithmetic only.
#pragma once
#include <algorithm>
#include <cstddef>

namespace tups {

constexpr size_t kGreenTabBytes = (size_t)256 << 20;  // of one pass
constexpr size_t kGreenElem = 16;                     // bytes of an element (complex128)

struct GreenShape {
  int lo = 0, len = 0;
  int ng2 = 1;      // grains in all
  int grains = 1;   // grains of one pass
  bool split = false;
  int plain = 0;    // slot of the lattice point itself
  size_t slots() const { return split ? 2 * (size_t)grains + 1 : (size_t)grains; }
  size_t bytes(int nc) const { return slots() * nc * len * kGreenElem; }
  int passes() const { return (ng2 + grains - 1) / grains; }
};

// the shape over the enlarged box of f_range, with at most `budget` bytes for the grains of a pass
inline GreenShape green_shape(int nc, int nf, int nw, int ngrain, int f_range, size_t budget = kGreenTabBytes) {
  GreenShape t;
  // k + q and q - k reach (f_range + 1) Nf + Nw - 1 on top, the self-energy's k - q down to 2 - Nw
  t.lo = std::min(1 - f_range * nf, 2 - nw);
  t.len = (f_range + 1) * nf + nw - t.lo;
  t.ng2 = ngrain * ngrain;
  const size_t per = (size_t)nc * t.len * kGreenElem;
  t.split = per * t.ng2 > budget && t.ng2 > 1;
  if (t.split) {
    t.grains = (int)std::min<size_t>(t.ng2, std::max<size_t>(1, budget / per / 2));
    t.plain = 2 * t.grains;
  } else {
    t.grains = t.ng2;
    const int half = (ngrain + 1) / 2 - 1;
    t.plain = half * ngrain + half;
  }
  return t;
}

// what to reserve for work at f_range: the full iteration's calc_chi builds the table over the
// box itself (f_range 0) when the enlarged one takes several passes, and that can be the larger
// of the two (the slots of a pass are rounded to each shape's own rows)
inline size_t green_reserve_bytes(int nc, int nf, int nw, int ngrain, int f_range, size_t budget = kGreenTabBytes) {
  return std::max(green_shape(nc, nf, nw, ngrain, f_range, budget).bytes(nc),
                  green_shape(nc, nf, nw, ngrain, 0, budget).bytes(nc));
}

}  // namespace tups
