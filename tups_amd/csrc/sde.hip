// Self-energy from the Schwinger-Dyson equation in form-factor space, FP64.
//
// Reference: calc_SDE, SRC/parquet_SDE.f90:27-258 (its use_U2 second-order term
// calc_order_2nd, :263-340, is added from the device Grt by gtau.hip), with
// calc_chi_aux (:346-432), calc_LChi (:436-497), calc_PhChi
// (:501-537), calc_PPChi (:540-575) and symmetrize_array
// (SRC/parquet_util.f90:1215-1272).  Three kernels:
//  1. per IBZ q, the auxiliary bubbles over the Green's-function pairs of bubble.hip
//       chi_aux_X(l4, nu) = sum_k P_X(k, nu) FF(k, l4)
//     over the enlarged box nu in (-f_range Nf, (f_range + 1) Nf]; for f_range > 0
//     sde_aux_fold adds those outside the box to its edges, where pickNu_range
//     clamps the vertex to, so that every vertex column is read once;
//  2. sde_vchi: per (q, L3), PL = LChi + PhChi and PP = PPChi, i.e. the
//     resident reducible vertices contracted with the bubbles (one pass over
//     the four G_r arrays, coalesced along L3);
//  3. sde_sigma: per IBZ (k, nu) the sum over q slots and the star of each q with
//     the Green's functions at k + Sq, -k + Sq, k - Sq from the table of bubble.hip,
//     scaled by -U / beta^2 / Nc^2 / 2 and written to every point of k's star (the
//     stars partition the zone, so each Sigma entry is written once).
#include <algorithm>

#include "bubble.h"

namespace tups {

struct SdeArgs {
  const double2* tab;       // plain Green's functions: [k tlen + nu - tlo]
  int tlo, tlen;
  const double2* gam[4];    // reducible vertices G_r_LL (Nz, Nz, Nq)
  const double2* lam_d;     // L_d (Nf, Nf, Nw)
  const double2* lam_m;
  const double* ffi;        // FF_inv[(s Nl + l) Nc + (ky-1) Nx + kx-1]
  const int* signs;
  const int* qw;            // bosonic index of each q (1-based)
  const int* ibz;           // IBZ momenta: x[0..nibz), then y[0..nibz) (1-based)
  double2* caux_ph;         // [q][l4 ext + f_range Nf + nu - 1]
  double2* caux_pp;
  double2* wph;             // [q][l4 Nf + nu - 1]: the bubbles folded onto the box (caux itself at f_range 0)
  double2* wpp;
  double2* out_ph;          // [q]: sum of the l = 1 ph bubble outside the box (f_range > 0)
  double2* sum;             // [chunk][km Nf + nu - 1]: partial sums of sde_sigma
  double2* pl;              // [q][L3]: LChi + PhChi
  double2* pp;              // [q][L3]: PPChi
  double2* sigma_out;       // (Nx Ny Nf)
  int nx, nf, nl, nz, nq, nibz, nxi, ext, f_range, use_u2, chunks;
  double u, inv_ff11_sq, pref;
};

// list_symmetries (SRC/parquet_util.f90:1140-1207): bit s-1 set when operation s
// generates a point of the star of the IBZ point (kx, ky)
__device__ __forceinline__ unsigned star_ops(int kx, int ky, int nxi) {
  if ((kx == 1 && ky == 1) || (kx == nxi && ky == nxi)) return 0x01u;
  if (kx == nxi && ky == 1) return 0x11u;
  if (kx == nxi && ky > 1 && ky < nxi) return 0x01u | 0x02u | 0x10u | 0x80u;
  if (kx > 1 && ky < nxi) {
    if (ky == 1) return 0x01u | 0x04u | 0x10u | 0x20u;
    if (ky == kx) return 0x0fu;
    return 0xffu;
  }
  return 0u;
}

// symmetry_operation on 1-based momentum indices (SRC/parquet_util.f90:896-978)
__device__ __forceinline__ void sym_apply(int s, int ix, int iy, int nx, int& ox, int& oy) {
  const int x = ix - 1, y = iy - 1;
  int a = x, b = y;
  switch (s) {
    case 2: a = x; b = -y; break;
    case 3: a = -x; b = y; break;
    case 4: a = -x; b = -y; break;
    case 5: a = y; b = x; break;
    case 6: a = y; b = -x; break;
    case 7: a = -y; b = -x; break;
    case 8: a = -y; b = x; break;
    default: break;
  }
  ox = (a < 0 ? a + nx : a) + 1;  // |a|, |b| < Nx
  oy = (b < 0 ? b + nx : b) + 1;
}

// the bubbles outside the box onto its first and last frequency; grid: nq
__global__ __launch_bounds__(256) void sde_aux_fold(SdeArgs a) {
  const int q = blockIdx.x, nf = a.nf, fr = a.f_range * nf;
  for (int i = threadIdx.x; i < 2 * a.nl * nf; i += 256) {
    const int x = i / (a.nl * nf), e = i - x * a.nl * nf, l = e / nf, n = e - l * nf;
    const double2* c = (x ? a.caux_pp : a.caux_ph) + (size_t)q * a.nl * a.ext + (size_t)l * a.ext;
    double2 s = c[fr + n], lo = make_double2(0.0, 0.0), hi = lo;
    if (n == 0)
      for (int o = 0; o < fr; ++o) {
        lo.x += c[o].x;
        lo.y += c[o].y;
      }
    if (n == nf - 1)
      for (int o = fr + nf; o < a.ext; ++o) {
        hi.x += c[o].x;
        hi.y += c[o].y;
      }
    s.x += lo.x + hi.x;
    s.y += lo.y + hi.y;
    (x ? a.wpp : a.wph)[(size_t)q * a.nl * nf + e] = s;
  }
  if (threadIdx.x == 0) {
    const double2* c = a.caux_ph + (size_t)q * a.nl * a.ext;
    double2 s = make_double2(0.0, 0.0);
    for (int o = 0; o < fr; ++o) {
      s.x += c[o].x + c[fr + nf + o].x;
      s.y += c[o].y + c[fr + nf + o].y;
    }
    a.out_ph[q] = s;
  }
}

// grid: (ceil(Nz / R), nq); R lanes along L3 = (l3, nu) x 256 / R parts of the columns
// (R = 64, or the power of two that holds a smaller Nz), added in order.  HBM-bound:
// the four vertices once, 467 us at Nx = 8, Nf = 64, Nl = 5 (6.7 TB/s; 551 us with 256
// lanes along L3, of which Nz = 320 fills 5 of 8); Nx = 6, Nf = 22, Nl = 9, f_range = 1:
// 49 us (308 us with every clamped column read again).
__global__ __launch_bounds__(256) void sde_vchi(SdeArgs a, int rlog) {
  __shared__ double2 red[2][256];
  const int q = blockIdx.y, R = 1 << rlog, parts = 256 >> rlog;
  const int r = threadIdx.x & (R - 1), part = threadIdx.x >> rlog;
  const int i3 = blockIdx.x * R + r;
  const int nf = a.nf, nz = a.nz, w = a.qw[q];
  double2 pl = make_double2(0.0, 0.0), pp = make_double2(0.0, 0.0);
  if (i3 < nz) {
    const size_t base = (size_t)q * nz * nz + i3;
    const double2* wph = a.wph + (size_t)q * nz;
    const double2* wpp = a.wpp + (size_t)q * nz;
#pragma unroll 2
    for (int col = part; col < nz; col += parts) {
      const size_t idx = base + (size_t)col * nz;
      const double2 gd = ld_stream(a.gam[0] + idx), gm = ld_stream(a.gam[1] + idx);
      const double2 gs = ld_stream(a.gam[2] + idx), gt = ld_stream(a.gam[3] + idx);
      double2 t = cmul(make_double2(gd.x - 3.0 * gm.x, gd.y - 3.0 * gm.y), wph[col]);
      pl.x += t.x;
      pl.y += t.y;
      t = cmul(make_double2(gs.x + gt.x, gs.y + gt.y), wpp[col]);
      pp.x += t.x;
      pp.y += t.y;
    }
    if (i3 < nf) {  // LChi: the l = 1 block only
      const double2* cph = a.caux_ph + (size_t)q * a.nl * a.ext + a.f_range * nf;
      for (int o = part; o < nf; o += parts) {
        const double2 xp = cph[o];
        const size_t li = (size_t)i3 + (size_t)nf * o + (size_t)nf * nf * (w - 1);
        const double2 ld = a.lam_d[li], lm = a.lam_m[li];
        double cr = (ld.x - lm.x) * a.inv_ff11_sq;
        const double ci = (ld.y - lm.y) * a.inv_ff11_sq;
        if (a.use_u2) cr -= 2.0 * a.u * a.inv_ff11_sq;
        pl.x += cr * xp.x - ci * xp.y;
        pl.y += cr * xp.y + ci * xp.x;
      }
      if (part == 0 && a.f_range > 0 && !a.use_u2) {
        const double2 xp = a.out_ph[q];
        pl.x += 2.0 * a.u * a.inv_ff11_sq * xp.x;
        pl.y += 2.0 * a.u * a.inv_ff11_sq * xp.y;
      }
    }
  }
  red[0][threadIdx.x] = pl;
  red[1][threadIdx.x] = pp;
  __syncthreads();
  if (part > 0 || i3 >= nz) return;
  for (int p = 1; p < parts; ++p) {
    const double2 x = red[0][(p << rlog) + r], y = red[1][(p << rlog) + r];
    pl.x += x.x;
    pl.y += x.y;
    pp.x += y.x;
    pp.y += y.y;
  }
  a.pl[(size_t)q * nz + i3] = pl;
  a.pp[(size_t)q * nz + i3] = pp;
}

// the sum of one IBZ (k, nu) to every point of k's star
__device__ __forceinline__ void write_star(const SdeArgs& a, int km, int k0, double2 sum) {
  const int kx = a.ibz[km], ky = a.ibz[a.nibz + km];
  const unsigned ops = star_ops(kx, ky, a.nxi);
  const double2 v = make_double2(a.pref * sum.x, a.pref * sum.y);
  for (int s = 1; s <= 8; ++s)
    if ((ops >> (s - 1)) & 1u) {
      int sx, sy;
      sym_apply(s, kx, ky, a.nx, sx, sy);
      a.sigma_out[((size_t)(sx - 1) * a.nx + (sy - 1)) * a.nf + (k0 - 1)] = v;
    }
}

// 64 lanes of IBZ (k, nu), nu fastest, x 8 or 16 waves over the q slots of a chunk: the
// reads of pl, pp and of the Green's-function table run along nu, and the vertex parts
// of a q are read once for its star.  Bound by the L1 reads of the three Green's
// functions per (q, star operation).  Nx = 16, Nf = 64, Nl = 1: 86 us
// (728 us with G formed for each use).
// grid: (ceil(NIBZ Nf / 64), chunks); with one chunk it writes Sigma itself
constexpr int sigma_waves(int nl) { return nl == 1 ? 16 : 8; }  // the vertex parts of a q take 8 Nl doubles
template <int NL, int LANES>
__global__ __launch_bounds__(64 * sigma_waves(NL)) void sde_sigma(SdeArgs a) {
  constexpr int W = sigma_waves(NL) * 64 / LANES;
  __shared__ double2 red[W][LANES];
  const int lane = threadIdx.x & (LANES - 1);
  const int part = LANES == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x / LANES;
  const int nf = a.nf, nx = a.nx, nc = nx * nx, nz = a.nz, nw = nf / 2;
  const int t = blockIdx.x * LANES + lane;
  const bool ok = t < a.nibz * nf;
  const int km = ok ? t / nf : 0, k0 = (ok ? t - km * nf : 0) + 1;
  const int kx = a.ibz[km] - 1, ky = a.ibz[a.nibz + km] - 1;
  const double* ffi = a.ffi + ky * nx + kx;
  double ar = 0.0, ai = 0.0;
  for (int q = blockIdx.y * W + part; q < a.nq; q += W * a.chunks) {
    const int m = q / nw, w = q - m * nw + 1;  // every IBZ q of the box, in order
    const int qx = a.ibz[m], qy = a.ibz[a.nibz + m];
    const unsigned ops = star_ops(qx, qy, a.nxi);
    const double2* pl = a.pl + (size_t)q * nz;
    const double2* pp = a.pp + (size_t)q * nz;
    double2 x[NL], y[NL], xm[NL], ym[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      x[l] = pl[l * nf + k0 - 1];
      y[l] = pp[l * nf + k0 - 1];
      const double sg = (double)a.signs[l];
      const double2 u = pl[l * nf + nf - k0], v = pp[l * nf + nf - k0];
      xm[l] = make_double2(sg * u.x, -sg * u.y);
      ym[l] = make_double2(sg * v.x, -sg * v.y);
    }
    const double2* tp = a.tab + (k0 + w - 1 - a.tlo);   // G(., nu + w - 1)
    const double2* tm = a.tab + (nf - k0 + w - a.tlo);  // G(., Nf - nu + w)
    const double2* tr = a.tab + (k0 - w + 1 - a.tlo);   // G(., nu - w + 1)
#pragma unroll(NL == 1 ? 4 : 1)
    for (int s = 1; s <= 8; ++s) {
      if (!((ops >> (s - 1)) & 1u)) continue;
      int sx, sy;
      sym_apply(s, qx, qy, nx, sx, sy);
      int px = kx + sx - 1, py = ky + sy - 1, mx = sx - 1 - kx, my = sy - 1 - ky;
      px -= px >= nx ? nx : 0;
      py -= py >= nx ? nx : 0;
      mx += mx < 0 ? nx : 0;
      my += my < 0 ? nx : 0;
      const int rx = mx ? nx - mx : 0, ry = my ? nx - my : 0;
      const double2 gkq = tp[(size_t)(py * nx + px) * a.tlen];
      const double2 gqmk = tm[(size_t)(my * nx + mx) * a.tlen];
      double2 sx1 = make_double2(0.0, 0.0), sy1 = sx1, sxm = sx1, sym = sx1;
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        const double fi = ffi[(size_t)((s - 1) * NL + l) * nc];
        sx1.x += fi * x[l].x;
        sx1.y += fi * x[l].y;
        sy1.x += fi * y[l].x;
        sy1.y += fi * y[l].y;
        sxm.x += fi * xm[l].x;
        sxm.y += fi * xm[l].y;
        sym.x += fi * ym[l].x;
        sym.y += fi * ym[l].y;
      }
      double2 c = cmul(gkq, sx1);
      ar += c.x;
      ai += c.y;
      c = cmul(gqmk, sy1);
      ar += c.x;
      ai += c.y;
      if (w == 1) continue;
      c = cmul(tr[(size_t)(ry * nx + rx) * a.tlen], sxm);
      ar += c.x;
      ai += c.y;
      c = cmul(make_double2(gkq.x, -gkq.y), sym);
      ar += c.x;
      ai += c.y;
    }
  }
  red[part][lane] = make_double2(ar, ai);
  __syncthreads();
  if (part > 0 || !ok) return;
  for (int p = 1; p < W; ++p) {
    ar += red[p][lane].x;
    ai += red[p][lane].y;
  }
  if (a.chunks == 1)
    write_star(a, km, k0, make_double2(ar, ai));
  else
    a.sum[(size_t)blockIdx.y * a.nibz * nf + t] = make_double2(ar, ai);
}

// the chunks' sums in order; grid: ceil(NIBZ Nf / 64)
__global__ __launch_bounds__(64) void sde_star(SdeArgs a) {
  const int n = a.nibz * a.nf, t = blockIdx.x * 64 + threadIdx.x;
  if (t >= n) return;
  double2 s = make_double2(0.0, 0.0);
  for (int c = 0; c < a.chunks; ++c) {
    const double2 v = a.sum[(size_t)c * n + t];
    s.x += v.x;
    s.y += v.y;
  }
  write_star(a, t / a.nf, t % a.nf + 1, s);
}

// chunks of the q slots of sde_sigma: enough workgroups for the chip, at least four q
// slots for each of their waves (a chunk costs a partial sum and, from two on, the
// extra launch, which a small box does not earn back)
static int sde_chunks(const tups_sizes& s) {
  const int wg = (s.nibz * s.nf + 63) / 64;
  return std::max(1, std::min({512 / wg, s.nq / 64, 32}));
}

// sizes of the SDE workspace's parts, in elements
struct SdeParts {
  size_t aux, v, fold, out, sum, sigma;
  size_t total() const { return 2 * aux + 2 * v + 2 * fold + out + sum + sigma; }
};
static SdeParts sde_parts(const tups_sizes& s, int f_range) {
  SdeParts p;
  p.aux = (size_t)s.nq * s.nl * (2 * (size_t)f_range + 1) * s.nf;
  p.v = (size_t)s.nq * s.nz;
  p.fold = f_range > 0 ? p.v : 0;
  p.out = f_range > 0 ? s.nq : 0;
  const int ch = sde_chunks(s);
  p.sum = ch > 1 ? (size_t)ch * s.nibz * s.nf : 0;
  p.sigma = (size_t)s.nx * s.ny * s.nf;
  return p;
}

// workspace and table of the SDE for ngrain and f_range (allocated outside any stream
// capture, and before a call changes anything: what is refused here leaves the context as it was)
int sde_reserve(tups_ctx* c, int ngrain, int f_range) {
  const tups_sizes& s = c->sz;
  TUPS_CHECK(ngrain >= 1 && ngrain <= 64, TUPS_EINVAL, "ngrain must be in 1..64");
  TUPS_CHECK(f_range >= 0 && f_range <= 8, TUPS_EINVAL, "f_range must be in 0..8");
  const size_t need = sde_parts(s, f_range).total() * sizeof(double2);
  if (c->sde_ws_bytes < need) {
    drop_graphs(c);  // captured graphs hold the old workspace
    if (c->sde_ws) TUPS_HIP(hipFree(c->sde_ws));
    c->sde_ws = nullptr;
    c->sde_ws_bytes = 0;
    TUPS_HIP(hipMalloc(&c->sde_ws, need));
    c->sde_ws_bytes = need;
  }
  return green_tab_reserve(c, ngrain, f_range);
}

// Sigma output of the last SDE launch with this f_range (inside the workspace)
double2* sde_output(tups_ctx* c, int f_range) {
  const SdeParts p = sde_parts(c->sz, f_range);
  return static_cast<double2*>(c->sde_ws) + (p.total() - p.sigma);
}

// where calc_chi_aux's results go
BubbleOut sde_aux_out(tups_ctx* c, int f_range) {
  const tups_sizes& s = c->sz;
  const int ext = (2 * f_range + 1) * s.nf;
  double2* ws = static_cast<double2*>(c->sde_ws);
  return {ws, ws + sde_parts(s, f_range).aux, (long long)s.nl * ext, 1, ext};
}

// the SDE from the Sigma on the device (g); the workspace must be reserved.  tab: the
// table when it is built already; aux_done: so are the auxiliary bubbles
int launch_sde_device(tups_ctx* c, const GreenParams& g, const GreenTab* tab, bool aux_done, int f_range, double u,
                      int use_u2) {
  const tups_sizes& s = c->sz;
  SdeArgs a{};
  const int nc = s.nx * s.ny;
  a.ext = (2 * f_range + 1) * s.nf;
  const SdeParts p = sde_parts(s, f_range);
  double2* ws = static_cast<double2*>(c->sde_ws);
  a.caux_ph = ws;
  a.caux_pp = ws + p.aux;
  a.pl = ws + 2 * p.aux;
  a.pp = a.pl + p.v;
  a.wph = f_range > 0 ? a.pp + p.v : a.caux_ph;
  a.wpp = f_range > 0 ? a.wph + p.fold : a.caux_pp;
  a.out_ph = a.pp + p.v + 2 * p.fold;
  a.sum = a.out_ph + p.out;
  a.sigma_out = a.sum + p.sum;
  a.chunks = sde_chunks(s);
  for (int r = 0; r < 4; ++r) a.gam[r] = c->gamma[r];
  a.lam_d = c->lam[0];
  a.lam_m = c->lam[1];
  a.ffi = c->d_ffik;
  a.signs = c->d_signs;
  a.qw = c->d_qw;
  a.ibz = c->d_ibz;
  a.nx = s.nx;
  a.nf = s.nf;
  a.nl = s.nl;
  a.nz = s.nz;
  a.nq = s.nq;
  a.nibz = s.nibz;
  a.nxi = (s.nx + 2) / 2;
  a.f_range = f_range;
  a.use_u2 = use_u2 ? 1 : 0;
  a.u = u;
  const double f11 = c->tab.ff[0];
  a.inv_ff11_sq = 1.0 / (f11 * f11);
  a.pref = -u / c->beta / c->beta / nc / nc / 2.0;
  if (int rc = timer_begin(c)) return rc;
  GreenTab t;
  if (tab)
    t = *tab;
  else if (int rc = green_tab_build(c, g, f_range, 0, &t))
    return rc;
  if (!aux_done) {
    const BubbleOut out[2] = {{}, sde_aux_out(c, f_range)};
    if (int rc = launch_bubbles(c, g, f_range, kBubbleAux, out, &t)) return rc;
  }
  a.tab = t.tab + (size_t)t.plain * nc * t.len;  // in the table whichever pass is in it
  a.tlo = t.lo;
  a.tlen = t.len;
  if (f_range > 0) {
    hipLaunchKernelGGL(sde_aux_fold, dim3((unsigned)s.nq), dim3(256), 0, c->stream, a);
    TUPS_HIP(hipGetLastError());
  }
  const int rlog = s.nz <= 16 ? 4 : s.nz <= 32 ? 5 : 6;
  hipLaunchKernelGGL(sde_vchi, dim3((unsigned)((s.nz + (1 << rlog) - 1) >> rlog), (unsigned)s.nq), dim3(256), 0, c->stream,
                     a, rlog);
  TUPS_HIP(hipGetLastError());
  const int wg = (s.nibz * s.nf + 63) / 64;
  // with few (k, nu) and no chunks, 16 to a workgroup spreads them over four times the CUs
  const bool few = a.chunks == 1 && wg <= 64;
  auto sigma = s.nl == 1   ? (few ? sde_sigma<1, 16> : sde_sigma<1, 64>)
               : s.nl == 5 ? (few ? sde_sigma<5, 16> : sde_sigma<5, 64>)
                           : (few ? sde_sigma<9, 16> : sde_sigma<9, 64>);
  hipLaunchKernelGGL(sigma, dim3((unsigned)(few ? (s.nibz * s.nf + 15) / 16 : wg), (unsigned)a.chunks),
                     dim3(64 * sigma_waves(s.nl)), 0, c->stream, a);
  TUPS_HIP(hipGetLastError());
  if (a.chunks > 1) {
    hipLaunchKernelGGL(sde_star, dim3((unsigned)wg), dim3(64), 0, c->stream, a);
    TUPS_HIP(hipGetLastError());
  }
  if (int rc = timer_end(c, TUPS_K_SDE)) return rc;
  return TUPS_OK;
}

// SigmaOld <- Sigma (SRC/loop.f90:152), Sigma <- the SDE output, and with the default
// rule Sigma_H(k) = Sigma(k, Nf) (SRC/parquet_chi.f90:103-110): the device state for the
// convergence check and the next iteration
__global__ __launch_bounds__(256) void sigma_commit(const double2* __restrict__ src, double2* __restrict__ sigma,
                                                    double2* __restrict__ sigma_old, double2* __restrict__ sigh,
                                                    int nx, int nf, int sigh_default) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t nt = (size_t)nx * nx * nf;
  if (i >= nt) return;
  const double2 v = src[i];
  sigma_old[i] = sigma[i];
  sigma[i] = v;
  if (sigh_default && (int)(i % nf) == nf - 1) {
    const size_t k = i / nf;  // (kx - 1) Ny + ky - 1
    const size_t kx = k / nx, ky = k % nx;
    sigh[kx + (size_t)nx * ky] = v;
  }
}

int launch_sigma_commit(tups_ctx* c, int f_range) {
  const tups_sizes& s = c->sz;
  const size_t nt = (size_t)s.nx * s.ny * s.nf;
  hipLaunchKernelGGL(sigma_commit, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, c->stream,
                     sde_output(c, f_range), c->d_sigma, c->d_sigma_old, c->d_sigh, s.nx, s.nf,
                     c->sigh_default ? 1 : 0);
  TUPS_HIP(hipGetLastError());
  return TUPS_OK;
}

int launch_sde(tups_ctx* c, const double* sigma, const double* sigma_h, double mu, int ngrain, int f_range, double u,
               int use_u2, double* sigma_out) {
  const tups_sizes& s = c->sz;
  TUPS_CHECK(sigma_out, TUPS_EINVAL, "null output");
  GreenParams g{};
  if (int rc = sde_reserve(c, ngrain, f_range)) return rc;
  if (int rc = upload_sigma(c, sigma, sigma_h, &g, mu, ngrain)) return rc;
  if (int rc = launch_sde_device(c, g, nullptr, false, f_range, u, use_u2)) return rc;
  if (use_u2) {
    TUPS_CHECK(c->grt_valid && c->gt_ngrain == ngrain, TUPS_ESTATE,
               "use_u2 needs Grt on the device for this ngrain (tups_gkw_grt first)");
    if (int rc = launch_order_2nd(c, u, sde_output(c, f_range))) return rc;
  }
  const size_t nt = (size_t)s.nx * s.ny * s.nf;
  TUPS_HIP(hipMemcpyAsync(sigma_out, sde_output(c, f_range), nt * sizeof(double2), hipMemcpyDeviceToHost, c->stream));
  TUPS_HIP(hipStreamSynchronize(c->stream));
  return TUPS_OK;
}

}  // namespace tups
