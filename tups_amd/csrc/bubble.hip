// Green's-function pairs summed over the zone with form-factor weights, FP64:
//
//   P_ph(k, nu) = 1/Ng^2 sum_g G(g; k, nu) G(g; k + q, nu + w - 1)
//   P_pp(k, nu) = 1/Ng^2 sum_g G(g; k, nu) G(Ng + 1 - g; q - k, Nf - nu + w)
//   out_i(nu, q) = sum_k W_i(k) P(k, nu)
// with W = FF_l1 FF_l2 for calc_chi (SRC/parquet_chi.f90:438-523), FF_l for
// calc_chi_aux (SRC/parquet_SDE.f90:346-432) and FF_sdwave FF_l for calc_GG_ph /
// calc_GG_pp (SRC/parquet_sus.f90:528-643); get_green_coarse
// (SRC/parquet_util.f90:1303-1327) with Sigma_H outside the box.
//
// G depends on q not at all, so it is formed once per (grain, k, nu)
// (green_table) instead of three times per (q, k, nu): the cosines and the
// division were nearly all of the former kernels' time.  In the pair kernel a lane
// is one (q, nu) with nu fastest, so the three reads of a (grain, k) are contiguous
// runs of the table (0.4 to 8 MB, served by L1 and L2), k and with it every weight
// is uniform over the wave (scalar operands), and the sums stay in registers: no
// LDS between the product and the projection.  Four waves (with 16 lanes, for small
// grids, 16 parts) take every fourth k and are added in order at the end.  Bound by
// the issue of the 8 + 4 NW FP64 operations
// per (grain, k) and, at few weights, by the L1 reads.  calc_chi and calc_chi_aux
// together at Nx = 16, Nf = 64, Nl = 1 (1440 q): 63 us (1224 + 664 us); calc_GG at
// Nx = 8, Nf = 64, Nl = 5, Ngrain = 4: 75 us (2681 us); the table 4 to 5 us.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "bubble.h"

namespace tups {

// grid: ceil(slots Nc len / 256)
__global__ __launch_bounds__(256) void green_table(GreenParams gp, double2* tab, int lo, int len, int grains, int g0,
                                                   int split, int slots) {
  const GreenParams g = green_resolve(gp);
  const int nc = g.nx * g.nx, ng = g.ngrain, ng2 = ng * ng;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)slots * nc * len) return;
  const int o = (int)(i % len), rest = (int)(i / len);
  const int k = rest % nc, slot = rest / nc;
  const int kx = k % g.nx + 1, ky = k / g.nx + 1;
  int gr = slot;
  if (split) {
    if (slot == 2 * grains) {
      tab[i] = green_plain(g, kx, ky, lo + o);
      return;
    }
    gr = slot < grains ? g0 + slot : ng2 - 1 - (g0 + slot - grains);
    if (gr < 0 || gr >= ng2) return;  // the last pass may be shorter
  }
  tab[i] = green_coarse(g, gr % ng + 1, gr / ng + 1, kx, ky, lo + o);
}

struct BubbleArgs {
  const double2* tab;
  const double* wt;
  const int* dst;
  const int* qm;
  const int* qw;
  const int* ibz;
  double2 *ph[2], *pp[2];
  long long qs[2];
  int os[2], us[2];
  int lo, len, nx, nf, nq, nibz, ext, f_range, nwt, grains, mirror, mslot, accumulate;
  double inv_g2;
};

// grid: (ceil(nq ext / LANES), weight groups); LANES lanes of (q, nu) x 256 / LANES parts of k
template <int NW, int LANES>
__global__ __launch_bounds__(256) void bubble_kernel(BubbleArgs a) {
  constexpr int STEP = NW < 4 ? NW : 4;  // weights reduced at a time
  constexpr int PARTS = 256 / LANES;
  __shared__ double2 red[PARTS - 1][2 * STEP][LANES];
  const int lane = threadIdx.x & (LANES - 1);
  const int part = LANES == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x / LANES;
  const int grp = blockIdx.y;
  const long long t = (long long)blockIdx.x * LANES + lane;
  const bool ok = t < (long long)a.nq * a.ext;
  const int q = ok ? (int)(t / a.ext) : 0, o = ok ? (int)(t - (long long)q * a.ext) : 0;
  const int nx = a.nx, nc = nx * nx, m = a.qm[q];
  const int qx = a.ibz[m] - 1, qy = a.ibz[a.nibz + m] - 1, w = a.qw[q];
  const int nu = o - a.f_range * a.nf + 1;
  const double2* t1 = a.tab + (nu - a.lo);
  const double2* t2 = a.tab + (nu + w - 1 - a.lo);
  const double2* t3 = a.tab + (a.nf - nu + w - a.lo);
  double2 ph[NW], pp[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) ph[i] = pp[i] = make_double2(0.0, 0.0);
  const double* wt = a.wt + (size_t)grp * nc * NW;
  for (int k = part; k < nc; k += PARTS) {
    const int ky = k / nx, kx = k - ky * nx;
    int ax = kx + qx, ay = ky + qy, bx = qx - kx, by = qy - ky;
    ax -= ax >= nx ? nx : 0;
    ay -= ay >= nx ? nx : 0;
    bx += bx < 0 ? nx : 0;
    by += by < 0 ? nx : 0;
    const int kq = ay * nx + ax, qk = by * nx + bx;
    double2 sph = make_double2(0.0, 0.0), spp = make_double2(0.0, 0.0);
#pragma unroll 2
    for (int s = 0; s < a.grains; ++s) {
      const int sm = a.mirror >= 0 ? a.mirror - s : a.mslot + s;
      const double2 g1 = t1[(size_t)(s * nc + k) * a.len];
      const double2 g2 = t2[(size_t)(s * nc + kq) * a.len];
      const double2 g3 = t3[(size_t)(sm * nc + qk) * a.len];
      sph.x += g1.x * g2.x - g1.y * g2.y;
      sph.y += g1.x * g2.y + g1.y * g2.x;
      spp.x += g1.x * g3.x - g1.y * g3.y;
      spp.y += g1.x * g3.y + g1.y * g3.x;
    }
    sph.x *= a.inv_g2;
    sph.y *= a.inv_g2;
    spp.x *= a.inv_g2;
    spp.y *= a.inv_g2;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const double f = wt[(size_t)k * NW + i];
      ph[i].x += f * sph.x;
      ph[i].y += f * sph.y;
      pp[i].x += f * spp.x;
      pp[i].y += f * spp.y;
    }
  }
#pragma unroll
  for (int i0 = 0; i0 < NW; i0 += STEP) {
    if (part > 0)
#pragma unroll
      for (int i = 0; i < STEP; ++i)
        if (i0 + i < NW) {
          red[part - 1][2 * i][lane] = ph[i0 + i];
          red[part - 1][2 * i + 1][lane] = pp[i0 + i];
        }
    __syncthreads();
    if (part == 0 && ok)
#pragma unroll
      for (int i = 0; i < STEP; ++i) {
        const int gi = grp * NW + i0 + i;
        if (i0 + i >= NW || gi >= a.nwt) continue;
        double2 x = ph[i0 + i], y = pp[i0 + i];
#pragma unroll
        for (int r = 0; r < PARTS - 1; ++r) {
          x.x += red[r][2 * i][lane].x;
          x.y += red[r][2 * i][lane].y;
          y.x += red[r][2 * i + 1][lane].x;
          y.y += red[r][2 * i + 1][lane].y;
        }
        const int kind = a.dst[3 * gi], off = a.dst[3 * gi + 1] * a.us[kind], off2 = a.dst[3 * gi + 2] * a.us[kind];
        const long long at = (long long)q * a.qs[kind] + (long long)o * a.os[kind];
        double2 *dph = a.ph[kind] + at, *dpp = a.pp[kind] + at;
        if (a.accumulate) {
          x.x += dph[off].x;
          x.y += dph[off].y;
          y.x += dpp[off].x;
          y.y += dpp[off].y;
        }
        dph[off] = x;
        dpp[off] = y;
        if (off2 >= 0) {
          dph[off2] = x;
          dpp[off2] = y;
        }
      }
    __syncthreads();
  }
}

// the widths that bubble_kernel exists for; a narrow layout has at most kNarrowWidth of
// more than 2 kNarrowWidth weights in a group
static const int kBubbleWidths[] = {1, 2, 5, 10, 15, 20, 23};
constexpr int kNarrowWidth = 5;

static GreenShape tab_shape(const tups_ctx* c, int ngrain, int f_range) {
  return green_shape(c->sz.nc, c->sz.nf, c->sz.nw, ngrain, f_range);
}

int upload_bubble_weights(tups_ctx* c) {
  const Tables& t = c->tab;
  const int nl = t.nl, nc = t.nc, nx = t.nx;
  struct Weight {
    std::vector<double> w;
    int kind, u, u2;
  };
  std::vector<Weight> chi, aux, sus;
  for (int l2 = 0; l2 < nl; ++l2) {
    const double* f2 = t.ff.data() + (size_t)l2 * nc;
    // the blocks are symmetric in (l1, l2)
    for (int l1 = 0; l1 <= l2; ++l1) {
      Weight x{std::vector<double>(nc), 0, l1 + nl * l2, l1 == l2 ? -1 : l2 + nl * l1};
      for (int k = 0; k < nc; ++k) x.w[k] = t.ff[(size_t)l1 * nc + k] * f2[k];
      chi.push_back(std::move(x));
    }
    aux.push_back({std::vector<double>(f2, f2 + nc), 1, l2, -1});
    for (int f = 0; f < 4; ++f) {  // fill_FF_sdwave (SRC/parquet_formfactors.f90:792-815)
      Weight x{std::vector<double>(nc), 0, f * nl + l2, -1};
      const double pi = 3.14159265358979323846;
      for (int k = 0; k < nc; ++k) {
        const double px = 2.0 / nx * pi * (k % nx), py = 2.0 / nx * pi * (k / nx);
        const double e = f == 0 ? 1.0 : f == 1 ? std::cos(px) - std::cos(py) : f == 2 ? std::sin(px) : std::sin(px) * std::sin(py);
        x.w[k] = e * f2[k];
      }
      sus.push_back(std::move(x));
    }
  }
  std::vector<Weight> both(chi);
  both.insert(both.end(), aux.begin(), aux.end());
  const std::vector<Weight>* sets[4] = {&chi, &aux, &both, &sus};
  std::vector<double> wt;
  std::vector<int> dst;
  for (int kk = 0; kk < 8; ++kk) {
    const bool wide = kk >= 4;
    const std::vector<Weight>& v = *sets[kk & 3];
    BubbleSet& b = c->bubble_set[wide][kk & 3];
    b.count = (int)v.size();
    b.wt = wt.size();
    b.dst = (int)dst.size();
    // a group costs its NW weights and the products it forms again, worth about four a grain;
    // the wide layout is for many of them
    long long best = -1;
    for (int w : kBubbleWidths) {
      if (!wide && w > kNarrowWidth && b.count > 2 * kNarrowWidth) continue;
      const long long g = (b.count + w - 1) / w, cost = g * (w + (wide ? 64 : 4));
      if (best < 0 || cost < best) {
        best = cost;
        b.nw = w;
        b.groups = (int)g;
      }
    }
    wt.resize(wt.size() + (size_t)b.groups * nc * b.nw, 0.0);
    for (int i = 0; i < b.count; ++i) {
      for (int n = 0; n < nc; ++n) wt[b.wt + ((size_t)(i / b.nw) * nc + n) * b.nw + i % b.nw] = v[i].w[n];
      dst.insert(dst.end(), {v[i].kind, v[i].u, v[i].u2});
    }
  }
  // one block: the weights, their places, and room for the table at Ngrain 1 and f_range 0
  const size_t o_dst = wt.size() * sizeof(double);
  const size_t o_tab = (o_dst + dst.size() * sizeof(int) + 255) / 256 * 256;
  const size_t n_tab = tab_shape(c, 1, 0).bytes(nc);
  if (c->green_tab_owned) (void)hipFree(c->green_tab);
  if (c->d_bubble_wt) (void)hipFree(c->d_bubble_wt);
  c->green_tab = nullptr;
  c->green_tab_owned = false;
  c->green_tab_bytes = 0;
  c->d_bubble_wt = nullptr;
  TUPS_HIP(hipMalloc((void**)&c->d_bubble_wt, o_tab + n_tab));
  char* base = (char*)c->d_bubble_wt;
  c->d_bubble_dst = (int*)(base + o_dst);
  c->green_tab = (double2*)(base + o_tab);
  c->green_tab_bytes = n_tab;
  std::vector<char> img(o_tab);
  std::memcpy(img.data(), wt.data(), o_dst);
  std::memcpy(img.data() + o_dst, dst.data(), dst.size() * sizeof(int));
  TUPS_HIP(hipMemcpyAsync(base, img.data(), o_dst + dst.size() * sizeof(int), hipMemcpyHostToDevice, c->stream));
  TUPS_HIP(hipStreamSynchronize(c->stream));
  return TUPS_OK;
}

int green_tab_reserve(tups_ctx* c, int ngrain, int f_range) {
  const tups_sizes& s = c->sz;
  const size_t need = green_reserve_bytes(s.nc, s.nf, s.nw, ngrain, f_range);
  if (c->green_tab_bytes < need) {
    drop_graphs(c);  // captured graphs hold the old table
    if (c->green_tab_owned) TUPS_HIP(hipFree(c->green_tab));
    c->green_tab = nullptr;
    c->green_tab_owned = false;
    c->green_tab_bytes = 0;
    const hipError_t e = hipMalloc((void**)&c->green_tab, need);
    if (e != hipSuccess) {
      c->green_tab = nullptr;
      set_error(std::string("Green's-function table: hipMalloc of ") + std::to_string(need) + " bytes failed: " +
                hipGetErrorString(e));
      return TUPS_ENOMEM;
    }
    c->green_tab_bytes = need;
    c->green_tab_owned = true;
  }
  return TUPS_OK;
}

int green_tab_build(tups_ctx* c, const GreenParams& g, int f_range, int pass, GreenTab* out) {
  static_cast<GreenShape&>(*out) = tab_shape(c, g.ngrain, f_range);
  out->tab = c->green_tab;
  const int slots = (int)out->slots();
  const size_t n = out->slots() * c->sz.nc * out->len;
  TUPS_CHECK(out->bytes(c->sz.nc) <= c->green_tab_bytes, TUPS_ESTATE, "Green's-function table larger than reserved");
  const size_t nb = (n + 255) / 256;
  TUPS_CHECK(nb < ((size_t)1 << 31), TUPS_EINVAL, "Green's-function table grid too large");
  hipLaunchKernelGGL(green_table, dim3((unsigned)nb), dim3(256), 0, c->stream, g, c->green_tab, out->lo, out->len,
                     out->grains, pass * out->grains, out->split ? 1 : 0, slots);
  TUPS_HIP(hipGetLastError());
  return TUPS_OK;
}

int launch_bubbles(tups_ctx* c, const GreenParams& g, int f_range, int set, const BubbleOut* out, const GreenTab* built) {
  const tups_sizes& s = c->sz;
  // Narrow groups of weights where forming the products again costs little (one grain) or
  // falls to CUs that would be idle; us a call of calc_chi, narrow | wide at (Nx, Nf, Nl, Ngrain):
  // (4, 16, 5, 1) 27 | 31, (8, 16, 5, 1) 30 | 36, (6, 22, 9, 1) 34 | 41, (8, 64, 9, 1) 106 | 116,
  // (4, 32, 9, 2) 32 | 43; (8, 64, 5, 2) 86 | 74, (8, 32, 9, 4) 153 | 102.
  const long long n64 = ((long long)s.nq * (2 * f_range + 1) * s.nf + 63) / 64;
  const long long work = (long long)s.nc * g.ngrain * g.ngrain;  // products of a lane
  const bool wide = g.ngrain > 1 && (work > 256 || n64 * c->bubble_set[0][set].groups > 512);
  const BubbleSet& bs = c->bubble_set[wide][set];
  BubbleArgs a{};
  a.wt = c->d_bubble_wt + bs.wt;
  a.dst = c->d_bubble_dst + bs.dst;
  a.qm = c->d_qm;
  a.qw = c->d_qw;
  a.ibz = c->d_ibz;
  for (int k = 0; k < 2; ++k) {
    a.ph[k] = out[k].ph;
    a.pp[k] = out[k].pp;
    a.qs[k] = out[k].qs;
    a.os[k] = out[k].os;
    a.us[k] = out[k].us;
  }
  a.nx = s.nx;
  a.nf = s.nf;
  a.nq = s.nq;
  a.nibz = s.nibz;
  a.ext = (2 * f_range + 1) * s.nf;
  a.f_range = f_range;
  a.nwt = bs.count;
  a.inv_g2 = 1.0 / g.ngrain / g.ngrain;
  // A grid of less than half a workgroup a CU (one, with long sums) takes 16 lanes a
  // workgroup and splits a lane's products over 16 parts; 64 | 16 lanes at (Nx, Nf, Nl, Ngrain):
  // (4, 16, 5, 16) 334 | 97 us, (8, 16, 5, 4) 105 | 48, (8, 24, 9, 8) 211 | 187, (8, 24, 9, 1) 59 | 73.
  const bool few = (n64 * bs.groups <= 128 && work >= 64) || (n64 * bs.groups <= 256 && work >= 4096);
  const long long nb = few ? ((long long)s.nq * a.ext + 15) / 16 : n64;
  TUPS_CHECK(nb < (1LL << 31), TUPS_EINVAL, "bubble grid too large");
  const dim3 grid((unsigned)nb, (unsigned)bs.groups);
  GreenTab t;
  int passes = 1;
  for (int p = 0; p < passes; ++p) {
    if (built && p == 0) {
      t = *built;
    } else if (int rc = green_tab_build(c, g, f_range, p, &t)) {
      return rc;
    }
    passes = t.passes();
    a.tab = t.tab;
    a.lo = t.lo;
    a.len = t.len;
    a.grains = std::min(t.grains, t.ng2 - p * t.grains);
    a.mirror = t.split ? -1 : t.ng2 - 1;
    a.mslot = t.grains;
    a.accumulate = p > 0 ? 1 : 0;
    void (*fn)(BubbleArgs);
    switch (bs.nw) {
      case 1: fn = few ? bubble_kernel<1, 16> : bubble_kernel<1, 64>; break;
      case 2: fn = few ? bubble_kernel<2, 16> : bubble_kernel<2, 64>; break;
      case 5: fn = few ? bubble_kernel<5, 16> : bubble_kernel<5, 64>; break;
      case 10: fn = few ? bubble_kernel<10, 16> : bubble_kernel<10, 64>; break;
      case 15: fn = few ? bubble_kernel<15, 16> : bubble_kernel<15, 64>; break;
      case 20: fn = few ? bubble_kernel<20, 16> : bubble_kernel<20, 64>; break;
      default: fn = few ? bubble_kernel<23, 16> : bubble_kernel<23, 64>; break;
    }
    hipLaunchKernelGGL(fn, grid, dim3(256), 0, c->stream, a);
    TUPS_HIP(hipGetLastError());
  }
  return TUPS_OK;
}

}  // namespace tups
