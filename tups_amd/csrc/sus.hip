// Susceptibilities of the four channels from the resident vertices, FP64.
//
// Reference: calc_sus, SRC/parquet_sus.f90:18-362, with calc_GG_ph / calc_GG_pp
// (:528-643), fillpickNu_range (:708-731) and the external form factors
// fill_FF_sdwave (SRC/parquet_formfactors.f90:792-815: 1, cos px - cos py,
// sin px, sin px sin py).  Two steps:
//  1. per q slot the Green's-function pairs of the enlarged box (bubble.hip)
//       GG_ph(l, nu; ff) = 1/Ng^2 sum_{k, g} FF_sd(k, ff) FF(k, l) G(g; k, nu) G(g; k + q, nu + w - 1)
//       GG_pp(l, nu; ff) = 1/Ng^2 sum_{k, g} FF_sd(k, ff) FF(k, l) G(g; k, nu) G(Ng + 1 - g; q - k, Nf - nu + w);
//  2. sus_contract: per (q, channel) sus(ff) = sum_{L1, L2} V(L1, L2) GG(L1) GG(L2) / (Nx^2 Ny^2 beta^2),
//     V = F inside the box and, for the pairs not both inside, the bare vertex
//     (U, -U, 2U, 0 for d, m, s, t) / FF11^2 on the l = 1 block plus the
//     reducible vertex Phi at the clamped frequencies.  Lanes run along L1 (so
//     the vertex columns are read coalesced), each with the four form factors'
//     partial sums; one LDS reduction per workgroup.
// The loop's G_r_LL hold Phi when the reference calls calc_sus (before G = F - G,
// SRC/loop.f90:193-222); after a device iteration they hold Gamma = F - Phi, and
// Phi is read back as F - Gamma.
#include "bubble.h"

#include <cmath>

namespace tups {

namespace {

struct SusArgs {
  const double2* fv[4];
  const double2* gam[4];  // Phi (after_update = 0) or Gamma = F - Phi (after_update = 1)
  double2* gg;            // [q][2 (ph, pp)][4 ff][nent]
  double2* out;           // [r][ff][q]
  int nf, nl, nz, nq, ext, f_range, after_update;
  double bare[4], inv_ff11_sq, norm;
};

// grid: (nq, 4 channels)
__global__ __launch_bounds__(256) void sus_contract(SusArgs a) {
  __shared__ double2 red[4][256];
  const int q = blockIdx.x, r = blockIdx.y;
  const int nf = a.nf, ext = a.ext, nent = a.nl * ext;
  const size_t nz = a.nz, base = (size_t)q * nz * nz;
  const double2* gq = a.gg + ((size_t)q * 8 + (r < 2 ? 0 : 4)) * nent;  // [ff][nent]
  const double2* F = a.fv[r] + base;
  const double2* G = a.gam[r] + base;
  const double bare = a.bare[r] * a.inv_ff11_sq;
  double2 part[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) part[f] = make_double2(0.0, 0.0);
  for (int i1 = threadIdx.x; i1 < nent; i1 += 256) {
    const int l1 = i1 / ext, n1 = i1 - l1 * ext - a.f_range * nf + 1;
    const bool in1 = n1 >= 1 && n1 <= nf;
    const size_t row = (size_t)l1 * nf + (n1 < 1 ? 1 : (n1 > nf ? nf : n1)) - 1;  // pickNu
    double2 acc[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] = make_double2(0.0, 0.0);
    for (int i2 = 0; i2 < nent; ++i2) {
      const int l2 = i2 / ext, n2 = i2 - l2 * ext - a.f_range * nf + 1;
      const bool in2 = n2 >= 1 && n2 <= nf;
      const size_t col = (size_t)l2 * nf + (n2 < 1 ? 1 : (n2 > nf ? nf : n2)) - 1;
      const size_t idx = row + nz * col;
      double2 v;
      if (in1 && in2) {
        v = F[idx];
      } else {
        v = G[idx];
        if (a.after_update) {  // Phi = F - Gamma
          const double2 fv = F[idx];
          v = make_double2(fv.x - v.x, fv.y - v.y);
        }
        if (l1 == 0 && l2 == 0) v.x += bare;
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const double2 t = cmul(v, gq[(size_t)f * nent + i2]);
        acc[f].x += t.x;
        acc[f].y += t.y;
      }
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const double2 t = cmul(gq[(size_t)f * nent + i1], acc[f]);
      part[f].x += t.x;
      part[f].y += t.y;
    }
  }
#pragma unroll
  for (int f = 0; f < 4; ++f) red[f][threadIdx.x] = part[f];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        red[f][threadIdx.x].x += red[f][threadIdx.x + h].x;
        red[f][threadIdx.x].y += red[f][threadIdx.x + h].y;
      }
    __syncthreads();
  }
  if (threadIdx.x < 4) {
    const double2 s = red[threadIdx.x][0];
    a.out[((size_t)r * 4 + threadIdx.x) * a.nq + q] = make_double2(s.x * a.norm, s.y * a.norm);
  }
}

}  // namespace

}  // namespace tups

using namespace tups;

extern "C" int tups_calc_sus(tups_ctx* c, double u, int32_t f_range, int32_t after_update, double* sus_out) {
  TUPS_CHECK(c && sus_out, TUPS_EINVAL, "null argument");
  const tups_sizes& s = c->sz;
  TUPS_CHECK(s.full_ibz, TUPS_EINVAL, "the susceptibilities need every IBZ q of the box (nq = 0 at create)");
  TUPS_CHECK(f_range >= 0 && f_range <= 8, TUPS_EINVAL, "f_range must be in 0..8");
  // the header's limit; no buffer grows with Nx
  TUPS_CHECK(s.nx * s.ny <= 256, TUPS_EINVAL, "the susceptibilities support Nx <= 16");
  int rc = ensure_tables(c);
  if (rc) return rc;
  GreenParams g{};
  if ((rc = green_params(c, &g))) return rc;
  if ((rc = green_tab_reserve(c, g.ngrain, f_range))) return rc;
  SusArgs a{};
  a.ext = (2 * f_range + 1) * s.nf;
  const size_t nent = (size_t)s.nl * a.ext;
  const size_t need = ((size_t)s.nq * 8 * nent + 16 * (size_t)s.nq) * sizeof(double2);
  if (c->sus_ws_bytes < need) {
    if (c->sus_ws) TUPS_HIP(hipFree(c->sus_ws));
    c->sus_ws = nullptr;
    c->sus_ws_bytes = 0;
    TUPS_HIP(hipMalloc(&c->sus_ws, need));
    c->sus_ws_bytes = need;
  }
  a.gg = static_cast<double2*>(c->sus_ws);
  a.out = a.gg + (size_t)s.nq * 8 * nent;
  for (int r = 0; r < 4; ++r) {
    a.fv[r] = c->fvert[r];
    a.gam[r] = c->gamma[r];
  }
  a.nf = s.nf;
  a.nl = s.nl;
  a.nz = s.nz;
  a.nq = s.nq;
  a.f_range = f_range;
  a.after_update = after_update ? 1 : 0;
  a.bare[0] = u;
  a.bare[1] = -u;
  a.bare[2] = 2.0 * u;
  a.bare[3] = 0.0;
  const double f11 = c->tab.ff[0];
  a.inv_ff11_sq = 1.0 / (f11 * f11);
  a.norm = 1.0 / ((double)s.nx * s.nx * s.ny * s.ny * c->beta * c->beta);
  if ((rc = timer_begin(c))) return rc;
  const BubbleOut out[2] = {{a.gg, a.gg + 4 * nent, (long long)(8 * nent), 1, a.ext}, {}};
  if ((rc = launch_bubbles(c, g, f_range, kBubbleSus, out, nullptr))) return rc;
  hipLaunchKernelGGL(sus_contract, dim3((unsigned)s.nq, 4), dim3(256), 0, c->stream, a);
  TUPS_HIP(hipGetLastError());
  if ((rc = timer_end(c, TUPS_K_SUS))) return rc;
  TUPS_HIP(hipMemcpyAsync(sus_out, a.out, 16 * (size_t)s.nq * sizeof(double2), hipMemcpyDeviceToHost, c->stream));
  TUPS_HIP(hipStreamSynchronize(c->stream));
  return TUPS_OK;
}
