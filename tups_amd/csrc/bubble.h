// Table of Green's functions and the Green's-function pairs ("bubbles") formed
// from it, shared by calc_chi, the self-energy and the susceptibilities.
#pragma once
#include "green.h"
#include "green_shape.h"
#include "internal.h"

namespace tups {

// G(grain; k, nu) for the momenta k = (ky - 1) Nx + kx - 1 and the frequencies
// lo .. lo + len - 1 (1-based, outside 1..Nf with Sigma_H): tab[(slot Nc + k) len +
// nu - lo].  Slot s holds grain s = (gy - 1) Ng + gx - 1; when all of them would
// exceed kGreenTabBytes, a pass holds `grains` of them from g0 on, then their
// mirror images Ng^2 - 1 - g, then the lattice point itself (plain): green_shape.h.
struct GreenTab : GreenShape {
  const double2* tab = nullptr;
};

// the weight families: groups of NW weights wt[(group Nc + k) NW + i], and per weight
// where its sum goes, dst[3 i]: array pair, place, second place (-1: none)
enum { kBubbleChi = 0, kBubbleAux = 1, kBubbleChiAux = 2, kBubbleSus = 3 };

// reserves the table for this Ngrain and every shape that work at f_range builds (outside any capture)
int green_tab_reserve(tups_ctx* c, int ngrain, int f_range);
// forms pass `pass` of the table (one pass unless split) on the context's stream; an error
// when the reserved table does not hold it
int green_tab_build(tups_ctx* c, const GreenParams& g, int f_range, int pass, GreenTab* out);

// destination of one array pair: element q qs + o os + place us, o the frequency of the enlarged box
struct BubbleOut {
  double2 *ph = nullptr, *pp = nullptr;
  long long qs = 0;
  int os = 0, us = 0;
};
// the bubbles of weight family `set` over the enlarged box of f_range for every q
// slot, from the table when `built` holds it, else building its passes
int launch_bubbles(tups_ctx* c, const GreenParams& g, int f_range, int set, const BubbleOut* out, const GreenTab* built);
// the two users' launches in the full iteration (chi.hip, sde.hip)
int launch_chi_aux_device(tups_ctx* c, const GreenParams& g, const BubbleOut& aux, const GreenTab* tab);
BubbleOut sde_aux_out(tups_ctx* c, int f_range);
// the weight families to the device (with the other tables)
int upload_bubble_weights(tups_ctx* c);

}  // namespace tups
