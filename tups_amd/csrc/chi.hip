// Bubbles chi_ph, chi_pp in form-factor space for every q slot:
// calc_chi (SRC/parquet_chi.f90:438-523) with get_green_coarse
// (SRC/parquet_util.f90:1303-1327), Ek_grain (SRC/parquet_util.f90:143-164)
// and the index maps index_FaddB / index_minusF (SRC/parquet_util.f90:1345-1381).
//
//   chi_X(l1, l2, nu) = sum_k P_X(k, nu) FF(k, l1) FF(k, l2), X = ph, pp
// over the Green's-function pairs P of bubble.hip, with the Hartree value Sigma_H(k)
// outside the box 1..Nf.  Only the Nl x Nl blocks of the block-diagonal bubble are
// formed (the resident TUPS_CHI layout), each pair (l1, l2) once.
#include "bubble.h"

#include <cmath>

namespace tups {

// Sigma and Sigma_H to the device (Sigma_H defaults to Sigma at the last box
// frequency, SRC/parquet_chi.f90:103-110); synchronous w.r.t. the host buffers
int upload_sigma(tups_ctx* c, const double* sigma, const double* sigma_h, GreenParams* g, double mu, int ngrain) {
  const tups_sizes& s = c->sz;
  const int nc = s.nx * s.ny;
  const size_t nt = (size_t)nc * s.nf;
  TUPS_CHECK(sigma, TUPS_EINVAL, "null Sigma");
  TUPS_CHECK(ngrain >= 1 && ngrain <= 64, TUPS_EINVAL, "ngrain must be in 1..64");
  if (!c->d_sigma) TUPS_HIP(hipMalloc((void**)&c->d_sigma, nt * sizeof(double2)));
  if (!c->d_sigh) TUPS_HIP(hipMalloc((void**)&c->d_sigh, (size_t)nc * sizeof(double2)));
  if (!c->d_sigma_old) TUPS_HIP(hipMalloc((void**)&c->d_sigma_old, nt * sizeof(double2)));
  c->sigma_old_valid = false;
  std::vector<double> sh(2 * (size_t)nc);
  if (sigma_h) {
    std::copy(sigma_h, sigma_h + 2 * (size_t)nc, sh.begin());
  } else {
    for (int kx = 1; kx <= s.nx; ++kx)
      for (int ky = 1; ky <= s.ny; ++ky) {
        const size_t src = ((size_t)(kx - 1) * s.ny + (ky - 1)) * s.nf + (s.nf - 1);
        const size_t dst = (size_t)(kx - 1) + (size_t)s.nx * (ky - 1);
        sh[2 * dst] = sigma[2 * src];
        sh[2 * dst + 1] = sigma[2 * src + 1];
      }
  }
  TUPS_HIP(hipMemcpyAsync(c->d_sigma, sigma, nt * sizeof(double2), hipMemcpyHostToDevice, c->stream));
  TUPS_HIP(hipMemcpyAsync(c->d_sigh, sh.data(), (size_t)nc * sizeof(double2), hipMemcpyHostToDevice, c->stream));
  if (!c->d_gstate) TUPS_HIP(hipMalloc((void**)&c->d_gstate, sizeof(GtauState)));
  TUPS_HIP(hipMemcpyAsync(&c->d_gstate->mu, &mu, sizeof(double), hipMemcpyHostToDevice, c->stream));
  TUPS_HIP(hipStreamSynchronize(c->stream));
  g->sigma = c->d_sigma;
  g->sigh = c->d_sigh;
  g->nx = s.nx;
  g->nf = s.nf;
  g->ngrain = ngrain;
  g->mu = mu;
  g->beta = c->beta;
  g->mu_dev = nullptr;
  c->green_mu = mu;
  c->green_ngrain = ngrain;
  c->sigh_default = sigma_h == nullptr;
  c->green_set = true;
  return TUPS_OK;
}

// where calc_chi's results go
static BubbleOut chi_out(tups_ctx* c) {
  const tups_sizes& s = c->sz;
  return {c->chi[0], c->chi[1], (long long)s.nl * s.nl * s.nf, s.nl * s.nl, 1};
}

// The boxes that calc_chi takes.  No buffer of the bubbles grows with Nx any more; the line is
// where the k-space bubble of a frequency filled the LDS, and larger boxes stay refused.
static int chi_box_ok(const tups_ctx* c) {
  TUPS_CHECK(c->sz.nx <= 70, TUPS_EINVAL, "calc_chi supports Nx <= 70");
  return TUPS_OK;
}

// calc_chi from the Sigma already on the device (g); tab: the table when it is built already
int launch_chi_device(tups_ctx* c, const GreenParams& g, const GreenTab* tab) {
  if (int rc = chi_box_ok(c)) return rc;
  if (int rc = timer_begin(c)) return rc;
  const BubbleOut out[2] = {chi_out(c), {}};
  if (int rc = launch_bubbles(c, g, 0, kBubbleChi, out, tab)) return rc;
  if (int rc = timer_end(c, TUPS_K_CALC_CHI)) return rc;
  return TUPS_OK;
}

// calc_chi and, for the self-energy at f_range 0, calc_chi_aux over the same pairs
int launch_chi_aux_device(tups_ctx* c, const GreenParams& g, const BubbleOut& aux, const GreenTab* tab) {
  if (int rc = chi_box_ok(c)) return rc;
  if (int rc = timer_begin(c)) return rc;
  const BubbleOut out[2] = {chi_out(c), aux};
  if (int rc = launch_bubbles(c, g, 0, kBubbleChiAux, out, tab)) return rc;
  if (int rc = timer_end(c, TUPS_K_CALC_CHI)) return rc;
  return TUPS_OK;
}

int launch_calc_chi(tups_ctx* c, const double* sigma, const double* sigma_h, double mu, int ngrain) {
  GreenParams g{};
  if (int rc = chi_box_ok(c)) return rc;
  TUPS_CHECK(ngrain >= 1 && ngrain <= 64, TUPS_EINVAL, "ngrain must be in 1..64");
  if (int rc = green_tab_reserve(c, ngrain, 0)) return rc;
  if (int rc = upload_sigma(c, sigma, sigma_h, &g, mu, ngrain)) return rc;
  return launch_chi_device(c, g, nullptr);
}

}  // namespace tups
