// Closed form of the BSE ladder, direct (FP64) and by FP32 factors with FP64
// iterative refinement.
//
// For fixed Gamma the damped update of BSE(ite) (SRC/parquet_BSE.f90:62-132),
//   Phi = c_r f alpha (Gamma chi F + F chi Gamma) + (1 - f)(F - Gamma),
// has the fixed point F = (I - kappa_r Gamma chi)^-1 Gamma, kappa_r = 2 c_r alpha
// (push-through identity: Gamma chi F = F chi Gamma there), where Phi = F - Gamma
// for every damping f.  Both modes solve A X = Gamma, A = I - kappa_r Gamma chi,
// per (q, r) and return Phi = X - Gamma: the converged ladder in one call.  The
// reference has no such solve; it iterates the update.
//
// Direct mode (TUPS_BSE_CLOSED_LU), from D = 128 the block form: A = P^-1 L U by
// 64-column blocks with partial pivoting, a launch over all matrices per phase
// (closed_panel, closed_diag, closed_row, closed_trail), the block rows scaled
// by the inverses of their diagonal blocks (closed_scale), then the right-hand
// sides by panels of 64 columns (closed_lu_solve).  Work per (q, r): (8/3 + 8)
// D^3 real flops.  Below D = 128 closed_solve: Gauss-Jordan elimination with
// partial pivoting on the augmented matrix [A | Gamma] (D x 2D, complex128), one
// workgroup per matrix, 12 D^3 flops.  Per panel of CL_NB columns:
//   1. LU of the panel rows k0..D-1 with row pivoting (rows swapped over all
//      columns from k0 on, so the right-hand side follows the equations);
//   2. Y = L11^-1 Z on the panel rows for every trailing column Z;
//   3. rows below the panel: Z -= L21 Y                    (MFMA);
//   4. X = U11^-1 Y on the panel rows;
//   5. rows above the panel: Z -= P_above X                (MFMA);
// after the last panel the right-hand block holds the solution.
//
// Refinement mode (TUPS_BSE_CLOSED_IR): the same in FP32 (MFMA) on fp32(A); the
// block form keeps the factors, below D = 128 the elimination of [fp32(A) | I]
// gives the inverse.  With A32^-1 standing for either,
//   X  = fp64(A32^-1 fp32(Gamma))
//   repeat: R = Gamma - A X = Gamma - X + kappa (Gamma chi) X   (FP64 MFMA)
//           stop when max over (q, r) of |R|_F / |Gamma|_F <= tol
//           X += fp64(A32^-1 fp32(R))
// FP64 is used only for A's assembly, the residual and the update of X.  Each
// step shrinks the error by about cond(A) 2^-24.  A tolerance for full double
// precision (kIrFull) asks for one step beyond the X that meets it; the X that is
// returned is in every case one whose own residual meets the tolerance.  Work per
// (q, r): 8/3 D^3 FP32 (factors) + 8 D^3 FP32 per solve + 8 D^3 FP64 per residual.
#include "internal.h"
#include "lds_dma.h"

#include <cmath>
#include <cstring>
#include <type_traits>

namespace tups {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int CL_NB = 16;  // panel width (closed_solve), sub-panel width (block form)
constexpr int CL_T = 64;   // update tile (rows and columns)
constexpr int CL_BB = 64;  // block width of the block form

__device__ __forceinline__ double2 mkc(double x, double y) { return make_double2(x, y); }
__device__ __forceinline__ float2 mkc(float x, float y) { return make_float2(x, y); }

// Precision of an elimination or product: complex type, MFMA accumulator and
// the 16 x 16 x 4 MFMA output layout (element e of lane l sits at column l % 16
// and the row given by orow(l / 16, e)).
template <class R>
struct Prec;
template <>
struct Prec<double> {
  using C = double2;
  using V = d4;
  __device__ static V fma_add(double a, double b, V acc) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
  }
  __device__ static V fma_sub(double a, double b, V acc) {  // A negated by the MFMA modifier
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 1);
  }
  __device__ static int orow(int lk, int e) { return lk + 4 * e; }
};
template <>
struct Prec<float> {
  using C = float2;
  using V = f4;
  __device__ static V fma_add(float a, float b, V acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
  }
  __device__ static V fma_sub(float a, float b, V acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(-a, b, acc, 0, 0, 0);
  }
  __device__ static int orow(int lk, int e) { return 4 * lk + e; }
};

template <class C>
__device__ __forceinline__ C cmul(C a, C b) {
  return mkc(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <class C>
__device__ __forceinline__ C csub(C a, C b) {
  return mkc(a.x - b.x, a.y - b.y);
}
template <class C>
__device__ __forceinline__ C cinv(C a) {
  // 1 / a with the larger component scaled out (Smith's method), two divisions
  if (fabs(a.x) >= fabs(a.y)) {
    const auto r = a.y / a.x, id = 1 / (a.x + a.y * r);
    return mkc(id, -r * id);
  }
  const auto r = a.x / a.y, id = 1 / (a.y + a.x * r);
  return mkc(r * id, -id);
}

// Largest 64-bit key over the wave (unsigned order), in every lane: DPP steps
// leave the row maxima in every lane of a row, row_bcast carries them to lane
// 63, which is read out.
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long key) {
  unsigned hi = (unsigned)(key >> 32), lo = (unsigned)key;
  auto step = [&](auto ctrl, auto rmask) {
    constexpr int CT = decltype(ctrl)::value, RM = decltype(rmask)::value;
    const unsigned nhi = (unsigned)__builtin_amdgcn_update_dpp((int)hi, (int)hi, CT, RM, 0xf, false);
    const unsigned nlo = (unsigned)__builtin_amdgcn_update_dpp((int)lo, (int)lo, CT, RM, 0xf, false);
    if (nhi > hi || (nhi == hi && nlo > lo)) {
      hi = nhi;
      lo = nlo;
    }
  };
  step(std::integral_constant<int, 0xb1>{}, std::integral_constant<int, 0xf>{});   // quad_perm [1,0,3,2]
  step(std::integral_constant<int, 0x4e>{}, std::integral_constant<int, 0xf>{});   // quad_perm [2,3,0,1]
  step(std::integral_constant<int, 0x141>{}, std::integral_constant<int, 0xf>{});  // row_half_mirror
  step(std::integral_constant<int, 0x140>{}, std::integral_constant<int, 0xf>{});  // row_mirror
  step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // row_bcast:15 to rows 1, 3
  step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});  // row_bcast:31 to rows 2, 3
  hi = (unsigned)__builtin_amdgcn_readlane((int)hi, 63);
  lo = (unsigned)__builtin_amdgcn_readlane((int)lo, 63);
  return ((unsigned long long)hi << 32) | lo;
}

// Pivot key of a candidate: the bits of |.|_1 (a non-negative double, so its
// bits order as unsigned integers) with the low 10 bits replaced by 1023 -
// off (off < 1024, the row's offset in the panel), so the largest key is the
// largest magnitude (to 2^-42) and, among equal ones, the lowest row; 0 for
// no candidate and for NaN.
__device__ __forceinline__ unsigned long long pivot_key(double m, int off) {
  if (!(m >= 0.0)) return 0ull;
  return ((unsigned long long)__double_as_longlong(m) & ~0x3ffull) | (unsigned long long)(1023 - off);
}
__device__ __forceinline__ unsigned long long pivot_key(float m, int off) { return pivot_key((double)m, off); }
__device__ __forceinline__ double pivot_mag(unsigned long long key) {
  return __longlong_as_double((long long)(key & ~0x3ffull));
}

// f(std::integral_constant<int, I>{}) for I = B .. E - 1, each I a compile-time
// constant (register arrays indexed by it stay in registers)
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// consecutive workgroups go round-robin over the 8 XCDs: a contiguous range each
__device__ __forceinline__ int closed_xcd_remap(int bid, int nblk) {
  const int xcd = bid & 7, idx = bid >> 3;
  const int per = nblk >> 3, rem = nblk & 7;
  return xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

struct ClosedArgs {
  const double2* gam[4];
  double2* out[4];
  const double2* chi[2];
  void* W;      // column-major, double2 (direct) or float2 (refinement): [mat][2D columns][D rows] for
                // closed_solve, [mat][D columns][D rows] for the block form
  void* T;      // block form: [mat][block][2][CL_BB][CL_BB], L_kk^-1 and U_kk^-1
  int* perm;    // block form: [mat][D + 1]: row i of L U is row perm[i] of A; then whether any row moved
  int blk;      // the block form
  double2* gx;  // refinement mode: [mat][D][D] Gamma chi in FP64
  float2* g32;  // and fp32(Gamma), the first right-hand side of the inverse
  int* info;    // first failing pivot (1-based column) over all matrices, 0 if none
  int D, nf, nl, q0, nqb;
  double kappa[4];
};

__global__ void closed_clear(int* info) { *info = 0; }

// [I - kappa Gamma chi | Gamma] (direct mode) or [fp32(I - kappa Gamma chi) | I]
// (refinement mode, A formed in FP64 and rounded); the block form takes the left block
// only, its right-hand sides come from Gamma itself.  One workgroup per (nu,
// matrix) forms the Nl columns (l2, nu) of the left block from the Nl columns
// (l1, nu) of Gamma, each read once: (Gamma chi)(row, (l2, nu)) =
// sum_l1 Gamma(row, (l1, nu)) chi_nu(l1, l2), and writes the columns (l1, nu)
// of the right block from the same reads; in refinement mode also Gamma chi itself,
// which the residuals multiply with, and the rounded Gamma.  grid: (Nf, 4 nqb); one
// thread per row.
constexpr int CL_NL_MAX = 9;
template <class T, bool IR>
__global__ __launch_bounds__(256) void closed_build_nu(ClosedArgs a) {
  const int x = blockIdx.x, mat = blockIdx.y;
  const int r = mat / a.nqb, q = a.q0 + (mat - r * a.nqb);
  const int D = a.D, nf = a.nf, nl = a.nl;
  const double2* G = a.gam[r] + (size_t)D * D * q;
  T* W = static_cast<T*>(a.W) + (size_t)mat * (a.blk ? 1 : 2) * D * D;
  auto put = [](double re, double im) -> T {
    if constexpr (IR) return make_float2((float)re, (float)im);
    else return make_double2(re, im);
  };
  const int nu = x;
  const double2* cb = a.chi[r >> 1] + (size_t)nf * nl * nl * q + (size_t)nu * nl * nl;  // chi_nu(l1, l2) at l1 + nl l2
  const double kap = a.kappa[r];
  for (int row = threadIdx.x; row < D; row += 256) {
    double2 g[CL_NL_MAX];
#pragma unroll
    for (int l1 = 0; l1 < CL_NL_MAX; ++l1)
      if (l1 < nl) {
        const int j = l1 * nf + nu;
        g[l1] = G[(size_t)j * D + row];
        // the right-hand side: Gamma's column j (the identity's for the FP32 inverse)
        if constexpr (IR) {
          if (!a.blk) W[(size_t)(D + j) * D + row] = put(row == j ? 1.0 : 0.0, 0.0);
          a.g32[((size_t)mat * D + j) * D + row] = put(g[l1].x, g[l1].y);
        } else if (!a.blk) {
          W[(size_t)(D + j) * D + row] = g[l1];
        }
      }
    for (int l2 = 0; l2 < nl; ++l2) {
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int l1 = 0; l1 < CL_NL_MAX; ++l1)
        if (l1 < nl) {
          const double2 c = cb[l1 + nl * l2];
          sr += g[l1].x * c.x - g[l1].y * c.y;
          si += g[l1].x * c.y + g[l1].y * c.x;
        }
      const int j = l2 * nf + nu;
      W[(size_t)j * D + row] = put((row == j ? 1.0 : 0.0) - kap * sr, -kap * si);
      if constexpr (IR) a.gx[((size_t)mat * D + j) * D + row] = make_double2(sr, si);
    }
  }
}

// Z(r, c) -= sum_t W(r, k0 + t) W(k0 + t, c) for r in [r0, r1), c in [c0, c1),
// t < nb (nb <= CL_NB, the panel of closed_solve), by 64 x 64 tiles held in registers
// with both factors in LDS; four waves of 2 x 2 blocks of 16 x 16 x 4 MFMAs.
// A fragments: lane l holds A[l % 16][l / 16]; B: B[l / 16][l % 16].
template <class R>
__device__ void closed_update(typename Prec<R>::C* W, int D, int r0, int r1, int c0, int c1, int k0, int nb,
                              typename Prec<R>::C (*As)[CL_T + 1], typename Prec<R>::C (*Bs)[CL_T + 1]) {
  using P = Prec<R>;
  using C = typename P::C;
  using V = typename P::V;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  const C zero = mkc((R)0, (R)0);
  for (int tr = r0; tr < r1; tr += CL_T)
    for (int tc = c0; tc < c1; tc += CL_T) {
      V ar[2][2], ai[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = tr + wr + i * 16 + P::orow(lk, e), col = tc + wc + j * 16 + li;
            const C z = (row < r1 && col < c1) ? W[(size_t)col * D + row] : zero;
            ar[i][j][e] = z.x;
            ai[i][j][e] = z.y;
          }
      // thread tid moves A(row tid % 64, t (tid / 64) + 4 v) and B(t tid % 16, column
      // tid / 16 + 16 v), v < 4, all loads before the first store
      C pa[4], pb[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = tid & (CL_T - 1), ka = (tid >> 6) + 4 * v;
        pa[v] = (tr + row < r1 && ka < nb) ? W[(size_t)(k0 + ka) * D + tr + row] : zero;
        const int kb = tid % CL_NB, col = tid / CL_NB + 16 * v;
        pb[v] = (tc + col < c1 && kb < nb) ? W[(size_t)(tc + col) * D + k0 + kb] : zero;
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        As[(tid >> 6) + 4 * v][tid & (CL_T - 1)] = pa[v];
        Bs[tid % CL_NB][tid / CL_NB + 16 * v] = pb[v];
      }
      __syncthreads();
#pragma unroll
      for (int kk = 0; kk < CL_NB; kk += 4) {
        C fa[2], fb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[i] = As[kk + lk][wr + i * 16 + li];
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[j] = Bs[kk + lk][wc + j * 16 + li];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            // Z - A B: re -= ar br - ai bi, im -= ar bi + ai br
            ar[i][j] = P::fma_sub(fa[i].x, fb[j].x, ar[i][j]);
            ar[i][j] = P::fma_add(fa[i].y, fb[j].y, ar[i][j]);
            ai[i][j] = P::fma_sub(fa[i].x, fb[j].y, ai[i][j]);
            ai[i][j] = P::fma_sub(fa[i].y, fb[j].x, ai[i][j]);
          }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int row = tr + wr + i * 16 + P::orow(lk, e), col = tc + wc + j * 16 + li;
            if (row < r1 && col < c1) W[(size_t)col * D + row] = mkc(ar[i][j][e], ai[i][j][e]);
          }
    }
  __syncthreads();  // the updated Z is visible to the whole workgroup
}

// Z(k0 + i, c) <- sum_t M[i][t] Z(k0 + t, c) for i, t < nb and every column c in
// [c0, c1): one thread per column, M (NB x NB, identity-padded) in LDS.
template <class R>
__device__ void panel_rows_apply(typename Prec<R>::C* W, int D, int k0, int nb, int c0, int c1,
                                 const typename Prec<R>::C (*M)[CL_NB]) {
  using C = typename Prec<R>::C;
  for (int col = c0 + (int)threadIdx.x; col < c1; col += 256) {
    C* zc = W + (size_t)col * D + k0;
    C z[CL_NB];
#pragma unroll
    for (int i = 0; i < CL_NB; ++i) z[i] = i < nb ? zc[i] : mkc((R)0, (R)0);
#pragma unroll 1
    for (int i = 0; i < CL_NB; ++i) {
      R yr = 0, yi = 0;
#pragma unroll
      for (int t = 0; t < CL_NB; ++t) {
        const C m = M[i][t];
        yr = fma(m.x, z[t].x, fma(-m.y, z[t].y, yr));
        yi = fma(m.x, z[t].y, fma(m.y, z[t].x, yi));
      }
      if (i < nb) zc[i] = mkc(yr, yi);
    }
  }
}

// One workgroup per (q, r) matrix; grid: 4 * nqb.  PHI: the direct mode's
// final Phi = X - Gamma from the right-hand block (else the right-hand block,
// the inverse, stays in W).
template <class R, bool PHI>
__global__ __launch_bounds__(256, 2) void closed_solve(ClosedArgs a) {
  using C = typename Prec<R>::C;
  __shared__ C As[CL_NB][CL_T + 1];
  __shared__ C Bs[CL_NB][CL_T + 1];
  __shared__ C Ls[CL_NB][CL_NB];
  __shared__ C Li[CL_NB][CL_NB];
  __shared__ C Ui[CL_NB][CL_NB];
  __shared__ R red_v[256];
  __shared__ int red_i[256];
  const int mat = blockIdx.x;
  const int D = a.D, D2 = 2 * D;
  C* W = static_cast<C*>(a.W) + (size_t)mat * 2 * D * D;
  const int tid = threadIdx.x;
  const C one = mkc((R)1, (R)0), zero = mkc((R)0, (R)0);
  int info = 0;
  for (int k0 = 0; k0 < D; k0 += CL_NB) {
    const int nb = min(CL_NB, D - k0);
    // 1. panel LU, rows k0..D-1, columns k0..k0+nb-1
    for (int c = k0; c < k0 + nb; ++c) {
      R best = -1;
      int bi = c;
      for (int row = c + tid; row < D; row += 256) {
        const C v = W[(size_t)c * D + row];
        const R m = fabs(v.x) + fabs(v.y);
        if (m > best) {
          best = m;
          bi = row;
        }
      }
      red_v[tid] = best;
      red_i[tid] = bi;
      __syncthreads();
      for (int s = 128; s > 0; s >>= 1) {
        if (tid < s) {
          const R o = red_v[tid + s];
          const int oi = red_i[tid + s];
          if (o > red_v[tid] || (o == red_v[tid] && oi < red_i[tid])) {
            red_v[tid] = o;
            red_i[tid] = oi;
          }
        }
        __syncthreads();
      }
      const int p = red_i[0];
      const R pmax = red_v[0];
      __syncthreads();
      if (!(pmax > 0)) {  // zero or NaN pivot column: the system is singular
        if (info == 0) info = c + 1;
        continue;
      }
      if (p != c) {
        for (int col = k0 + tid; col < D2; col += 256) {
          const C x = W[(size_t)col * D + c];
          W[(size_t)col * D + c] = W[(size_t)col * D + p];
          W[(size_t)col * D + p] = x;
        }
      }
      __syncthreads();
      const C inv = cinv(W[(size_t)c * D + c]);
      for (int row = c + 1 + tid; row < D; row += 256) {
        const C l = cmul(W[(size_t)c * D + row], inv);
        W[(size_t)c * D + row] = l;
        for (int col = c + 1; col < k0 + nb; ++col)
          W[(size_t)col * D + row] = csub(W[(size_t)col * D + row], cmul(l, W[(size_t)col * D + c]));
      }
      __syncthreads();
    }
    for (int u = tid; u < CL_NB * CL_NB; u += 256) {
      const int i = u % CL_NB, j = u / CL_NB;
      Ls[i][j] = (i < nb && j < nb) ? W[(size_t)(k0 + j) * D + k0 + i] : zero;
    }
    __syncthreads();
    // inverses of the unit lower L11 and of the upper U11, padded to NB x NB with
    // the identity: thread t < NB forms column t of both
    if (tid < CL_NB) {
      const int t = tid;
      for (int i = 0; i < CL_NB; ++i) {
        C x = i == t ? one : zero;
        if (i < nb && t < nb)
          for (int s2 = t; s2 < i; ++s2) x = csub(x, cmul(Ls[i][s2], Li[s2][t]));
        Li[i][t] = x;
      }
      for (int i = CL_NB - 1; i >= 0; --i) {
        C x = i == t ? one : zero;
        if (i < nb && t < nb) {
          for (int s2 = i + 1; s2 <= t; ++s2) x = csub(x, cmul(Ls[i][s2], Ui[s2][t]));
          x = cmul(x, cinv(Ls[i][i]));
        }
        Ui[i][t] = x;
      }
    }
    __syncthreads();
    const int j0 = k0 + nb;
    // 2. Y = L11^-1 Z on the panel rows
    panel_rows_apply<R>(W, D, k0, nb, j0, D2, Li);
    __syncthreads();
    // 3. rows below the panel
    closed_update<R>(W, D, k0 + nb, D, j0, D2, k0, nb, As, Bs);
    // 4. X = U11^-1 Y on the panel rows
    panel_rows_apply<R>(W, D, k0, nb, j0, D2, Ui);
    __syncthreads();
    // 5. rows above the panel
    closed_update<R>(W, D, 0, k0, j0, D2, k0, nb, As, Bs);
  }
  if (info && tid == 0) atomicCAS(a.info, 0, info);
  if constexpr (PHI) {
    // Phi = X - Gamma
    const int r = mat / a.nqb, q = a.q0 + (mat - r * a.nqb);
    const double2* G = a.gam[r] + (size_t)D * D * q;
    double2* O = a.out[r] + (size_t)D * D * q;
    for (size_t u = tid; u < (size_t)D * D; u += 256) O[u] = csub(W[(size_t)D * D + u], G[u]);
  }
}

// X(dst[u], col) <- X(src[u], col) for u < n, every column col in [c0, c1)
// outside [e0, e1), all with the values from before the call (the rows of a
// composed sequence of row swaps).  Whole columns go at a time, PER items per
// thread: every source of a column is read before any of its rows is written.
template <class R, int PER>
__device__ void move_rows(typename Prec<R>::C* X, int ld, int c0, int c1, int e0, int e1, const int* dst,
                          const int* src, int n) {
  using C = typename Prec<R>::C;
  const int tid = threadIdx.x;
  const int nlo = e0 - c0, ncol = (c1 - c0) - (e1 - e0);
  if (n == 0 || ncol <= 0) return;
  const int cols = max(1, 256 * PER / n);  // whole columns per round
  for (int cb = 0; cb < ncol; cb += cols) {
    const int items = n * min(cols, ncol - cb);
    C val[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int it = k * 256 + tid;
      if (it < items) {
        const int cc = cb + it / n;
        const int col = cc < nlo ? c0 + cc : e1 + (cc - nlo);
        val[k] = X[(size_t)col * ld + src[it % n]];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int it = k * 256 + tid;
      if (it < items) {
        const int cc = cb + it / n;
        const int col = cc < nlo ? c0 + cc : e1 + (cc - nlo);
        X[(size_t)col * ld + dst[it % n]] = val[k];
      }
    }
    __syncthreads();
  }
}

// As move_rows for n <= 128 and no excluded columns, without workgroup
// barriers: wave w owns the columns c0 + G (w + 4 k) .. + G - 1 and lane l the
// moved rows l and l + 64; a wave's loads of a group of columns have all
// returned (vmcnt 0) before its stores to them are issued.
template <class R, int G>
__device__ void move_rows_waves(typename Prec<R>::C* X, int ld, int c0, int c1, const int* dst, const int* src,
                                int n) {
  using C = typename Prec<R>::C;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool h0 = lane < n, h1 = lane + 64 < n;
  const int s0 = h0 ? src[lane] : 0, d0 = h0 ? dst[lane] : 0;
  const int s1 = h1 ? src[lane + 64] : 0, d1 = h1 ? dst[lane + 64] : 0;
  for (int cb = c0 + G * wave; cb < c1; cb += 4 * G) {
    C x0[G], x1[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const size_t o = (size_t)min(cb + g, c1 - 1) * ld;
      if (h0) x0[g] = X[o + s0];
      if (h1) x1[g] = X[o + s1];
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (cb + g >= c1) break;
      const size_t o = (size_t)(cb + g) * ld;
      if (h0) X[o + d0] = x0[g];
      if (h1) X[o + d1] = x1[g];
    }
  }
}

// The rows that the swaps (r0 + i, piv[i]), i < nr, move (piv[i] >= r0 + i),
// for wave 0: map[x - lo] is the original row that row x holds after all the
// swaps, and the rows with map[x - lo] != x are listed, those of r0 .. r0 + nr
// - 1 first (in order), then those beyond, each once.  The count goes to *cnt.
__device__ __forceinline__ void list_moved_rows(const int* piv, int r0, int nr, const int* map, int lo, int* dst,
                                                int* src, int* cnt) {
  const int lane = threadIdx.x & 63;
  bool in = false, out = false;
  int p = 0, sin = 0, sout = 0;
  if (lane < nr) {
    sin = map[r0 + lane - lo];
    in = sin != r0 + lane;
    p = piv[lane];
    if (p >= r0 + nr) {
      sout = map[p - lo];
      out = sout != p;
      for (int j = 0; j < lane; ++j)
        if (piv[j] == p) out = false;
    }
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  const unsigned long long mi = __ballot(in), mo = __ballot(out);
  const int ni = __popcll(mi);
  if (in) {
    const int u = __popcll(mi & below);
    dst[u] = r0 + lane;
    src[u] = sin;
  }
  if (out) {
    const int u = ni + __popcll(mo & below);
    dst[u] = p;
    src[u] = sout;
  }
  if (lane == 0) *cnt = ni + __popcll(mo);
}

// LU factorisation with partial pivoting in CL_BB-wide blocks, right-looking, in place in
// W.  Per block column k0 .. k0 + nb, each a launch over every matrix:
//  A. closed_panel: its rows k0 .. D - 1 factored by one workgroup per matrix (CL_NB-wide
//     sub-panels: column by column within a sub-panel, then the sub-panel's rank-CL_NB
//     update of the rest of the block); the row swaps are applied to the other columns
//     of W and to perm;
//  B. closed_diag: L11^-1 and U11^-1 (nb x nb) from the factors, kept in T;
//  C. closed_row: the block rows of the later columns become U12 = L11^-1 Z1;
//  D. closed_trail: the rows below, Z -= L21 U12, a 64 x 64 tile per workgroup.
// The right-hand sides are no part of it: closed_lu_solve takes them through the factors
// column panel by column panel, which is where 8 of the 10.7 D^3 flops are.  A is a chain
// of column steps (a pivot search, an exchange and a rank-1 update between two barriers);
// on its own it has the registers and the VALU for itself, where beside the products of
// another workgroup every VALU instruction waits for an F64 MFMA.  D = 320, 480 q (1920
// matrices): 8.9 ms in FP64 with the scaling of the block rows, 2.9 of them A (one kernel
// per matrix doing all of it 14.2 ms; Gauss-Jordan on [A | Gamma] 28.1 ms against 8.9 + 10.0
// with the right-hand sides).
// closed_panel, RP > 0 (D - k0 <= 256 RP): a sub-panel's column steps run on registers
// (thread t holds rows s0 + t + 256 i, i < RP, of the CL_NB columns).  One barrier per
// step: before it each wave leaves its best pivot candidate (by a wave reduction) and
// that candidate's whole row in LDS, and thread c - s0 its row c; after it every thread
// picks the same winner, the two rows are exchanged from LDS and the rank-1 update runs
// on registers.  The swaps are recorded as a row map; the rows they move (none when no
// row is swapped) reach the other columns of the block at the end of the sub-panel and
// the rest of W at the end of the block.  RP = 0: every column step works on W in memory
// and swaps its rows at once.  grid: matrices
template <class R, int RP>
__global__ __launch_bounds__(256, RP == 1 ? 3 : 2) void closed_panel(ClosedArgs a, int k0) {
  using C = typename Prec<R>::C;
  constexpr int RMAX = RP > 0 ? 256 * RP : 1;  // rows of the register path
  constexpr int RQ = RP > 0 ? 1 : 0;
  __shared__ C Ls[CL_NB][CL_NB];          // L11 of a sub-panel
  __shared__ C Us[CL_NB][CL_BB - CL_NB];  // U12 beside it
  __shared__ R red_v[256 * (1 - RQ) + 1];
  __shared__ int red_i[256 * (1 - RQ) + 1];
  __shared__ unsigned long long pk[2][4 * RQ + 1];  // per-wave pivot keys, two buffers
  __shared__ C cand[2][4 * RQ + 1][CL_NB * RQ + 1];  // each wave's candidate pivot row, two buffers
  __shared__ C crow[2][CL_NB * RQ + 1];              // row c, which the pivot row replaces
  __shared__ int piv[CL_BB * RQ + 1];          // pivot row of each column of the block
  __shared__ int map_s[RMAX], map_b[RMAX];     // row sources after the sub-panel's / block's swaps
  __shared__ int mv_dst[2 * CL_BB * RQ + 1], mv_src[2 * CL_BB * RQ + 1];
  __shared__ int mv_n;
  const int mat = blockIdx.x, D = a.D, nb = min(CL_BB, D - k0);
  C* W = static_cast<C*>(a.W) + (size_t)mat * D * D;
  int* perm = a.perm + (size_t)mat * (D + 1);
  const int tid = threadIdx.x;
  const C zero = mkc((R)0, (R)0);
  int info = 0, moved = 0;
  if (k0 == 0)
    for (int x = tid; x <= D; x += 256) perm[x] = x < D ? x : 0;
  if constexpr (RP > 0)
    for (int x = k0 + tid; x < D; x += 256) map_b[x - k0] = x;
  __syncthreads();
  for (int s0 = k0; s0 < k0 + nb; s0 += CL_NB) {
    const int sb = min(CL_NB, k0 + nb - s0);
    if constexpr (RP > 0) {
      const int lane = tid & 63, wave = tid >> 6;
      for (int x = s0 + tid; x < D; x += 256) map_s[x - s0] = x;
      C v[RP][CL_NB];
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        const int row = s0 + tid + 256 * i;
#pragma unroll
        for (int j = 0; j < CL_NB; ++j) v[i][j] = (row < D && j < sb) ? W[(size_t)(s0 + j) * D + row] : zero;
      }
      // the CL_NB steps unrolled: the register columns take static indices
      static_for<0, CL_NB>([&](auto jc) {
        constexpr int j = decltype(jc)::value, buf = j & 1;
        if (j >= sb) return;
        const int c = s0 + j;
        C pc[RP];  // this thread's entries of column c
#pragma unroll
        for (int i = 0; i < RP; ++i) pc[i] = v[i][j];
        unsigned long long key = 0ull;
#pragma unroll
        for (int i = 0; i < RP; ++i) {
          const int row = s0 + tid + 256 * i;
          if (row >= c && row < D) {
            const unsigned long long k2 = pivot_key(fabs(pc[i].x) + fabs(pc[i].y), row - s0);
            if (k2 > key) key = k2;
          }
        }
        key = wave_max_u64(key);  // the wave's candidate
        const int bi = key ? s0 + 1023 - (int)(key & 0x3ff) : c;
        const int tb = (bi - s0) & 255, ib = (bi - s0) >> 8;
        if (tid == tb) {
#pragma unroll
          for (int i = 0; i < RP; ++i)
            if (i == ib) {
#pragma unroll
              for (int jj = 0; jj < CL_NB; ++jj) cand[buf][wave][jj] = v[i][jj];
            }
        }
        if (tid == j) {
#pragma unroll
          for (int jj = 0; jj < CL_NB; ++jj) crow[buf][jj] = v[0][jj];
        }
        if (lane == 0) pk[buf][wave] = key;
        __syncthreads();
        unsigned long long kmax = pk[buf][0];
        int pw = 0;
#pragma unroll
        for (int w = 1; w < 4; ++w) {
          const unsigned long long k2 = pk[buf][w];
          if (k2 > kmax) {
            kmax = k2;
            pw = w;
          }
        }
        const int p = s0 + 1023 - (int)(kmax & 0x3ff);
        if (!(pivot_mag(kmax) > 0)) {
          if (info == 0) info = c + 1;
          if (tid == 0) piv[c - k0] = c;
          return;
        }
        const C* prw = cand[buf][pw];
        const int tp = (p - s0) & 255, ip = (p - s0) >> 8;
        if (p != c) {
          if (tid == j) {
#pragma unroll
            for (int jj = 0; jj < CL_NB; ++jj) v[0][jj] = prw[jj];
          }
          if (tid == tp) {
#pragma unroll
            for (int i = 0; i < RP; ++i)
              if (i == ip) {
                pc[i] = crow[buf][j];
#pragma unroll
                for (int jj = 0; jj < CL_NB; ++jj) v[i][jj] = crow[buf][jj];
              }
          }
        }
        if (tid == 0) {
          piv[c - k0] = p;
          if (p != c) {
            const int t1 = map_s[c - s0];
            map_s[c - s0] = map_s[p - s0];
            map_s[p - s0] = t1;
            const int t2 = map_b[c - k0];
            map_b[c - k0] = map_b[p - k0];
            map_b[p - k0] = t2;
          }
        }
        const C inv = cinv(prw[j]);
#pragma unroll
        for (int i = 0; i < RP; ++i) {
          const int row = s0 + tid + 256 * i;
          if (row > c && row < D) {
            const C l = cmul(pc[i], inv);
            v[i][j] = l;
#pragma unroll
            for (int jj = j + 1; jj < CL_NB; ++jj) v[i][jj] = csub(v[i][jj], cmul(l, prw[jj]));
          }
        }
      });
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        const int row = s0 + tid + 256 * i;
        if (row < D)
#pragma unroll
          for (int j = 0; j < CL_NB; ++j)
            if (j < sb) W[(size_t)(s0 + j) * D + row] = v[i][j];
      }
      // the sub-panel's swaps on the other columns of the block
      if (wave == 0) list_moved_rows(piv + (s0 - k0), s0, sb, map_s, s0, mv_dst, mv_src, &mv_n);
      __syncthreads();
      move_rows<R, 8>(W, D, k0, k0 + nb, s0, s0 + sb, mv_dst, mv_src, mv_n);
      __syncthreads();
    } else
    for (int c = s0; c < s0 + sb; ++c) {
      R best = -1;
      int bi = c;
      for (int row = c + tid; row < D; row += 256) {
        const C v = W[(size_t)c * D + row];
        const R m = fabs(v.x) + fabs(v.y);
        if (m > best) {
          best = m;
          bi = row;
        }
      }
      red_v[tid] = best;
      red_i[tid] = bi;
      __syncthreads();
      for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) {
          const R o = red_v[tid + st];
          const int oi = red_i[tid + st];
          if (o > red_v[tid] || (o == red_v[tid] && oi < red_i[tid])) {
            red_v[tid] = o;
            red_i[tid] = oi;
          }
        }
        __syncthreads();
      }
      const int p = red_i[0];
      const R pmax = red_v[0];
      __syncthreads();
      if (!(pmax > 0)) {  // zero or NaN pivot column: the system is singular
        if (info == 0) info = c + 1;
        continue;
      }
      if (p != c) {
        if (tid == 0) {
          const int x = perm[c];
          perm[c] = perm[p];
          perm[p] = x;
        }
        moved = 1;
        for (int col = tid; col < D; col += 256) {
          const C x = W[(size_t)col * D + c];
          W[(size_t)col * D + c] = W[(size_t)col * D + p];
          W[(size_t)col * D + p] = x;
        }
      }
      __syncthreads();
      const C inv = cinv(W[(size_t)c * D + c]);
      for (int row = c + 1 + tid; row < D; row += 256) {
        const C l = cmul(W[(size_t)c * D + row], inv);
        W[(size_t)c * D + row] = l;
        for (int col = c + 1; col < s0 + sb; ++col)
          W[(size_t)col * D + row] = csub(W[(size_t)col * D + row], cmul(l, W[(size_t)col * D + c]));
      }
      __syncthreads();
    }
    if (s0 + sb < k0 + nb) {
      // the rest of the block (sb = CL_NB here): U12 = L11^-1 Z12 on the sub-panel rows by
      // substitution, a column per thread, kept in LDS as well; then Z22 -= L21 U12, each
      // wave taking strips of 16 rows with L21 and Z22 straight from memory
      const int c1 = s0 + CL_NB, nc = k0 + nb - c1;  // at most CL_BB - CL_NB columns
      if (tid < CL_NB * CL_NB) {
        const int i = tid % CL_NB, j = tid / CL_NB;
        Ls[i][j] = W[(size_t)(s0 + j) * D + s0 + i];
      }
      __syncthreads();
      if (tid < nc) {
        C* zc = W + (size_t)(c1 + tid) * D + s0;
        C z[CL_NB];
#pragma unroll
        for (int i = 0; i < CL_NB; ++i) z[i] = zc[i];
#pragma unroll
        for (int i = 1; i < CL_NB; ++i) {
          __builtin_amdgcn_sched_barrier(0);  // L11 is read row by row, not all ahead into registers
#pragma unroll
          for (int s2 = 0; s2 < i; ++s2) z[i] = csub(z[i], cmul(Ls[i][s2], z[s2]));
        }
#pragma unroll
        for (int i = 0; i < CL_NB; ++i) {
          zc[i] = z[i];
          Us[i][tid] = z[i];
        }
      }
      __syncthreads();
      {
        using P = Prec<R>;
        using V = typename P::V;
        const int lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = lane >> 4;
        for (int r0 = c1 + 16 * wave; r0 < D; r0 += 64) {
          C fa[CL_NB / 4];
          const int ar = min(r0 + li, D - 1);
#pragma unroll
          for (int ks = 0; ks < CL_NB / 4; ++ks) fa[ks] = W[(size_t)(s0 + 4 * ks + lk) * D + ar];
#pragma unroll
          for (int cb = 0; cb < (CL_BB - CL_NB) / 16; ++cb) {
            if (16 * cb >= nc) break;
            const int col = 16 * cb + li;
            C* zc = W + (size_t)(c1 + min(col, nc - 1)) * D;
            V zr, zi;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const C z = zc[min(r0 + P::orow(lk, e), D - 1)];
              zr[e] = z.x;
              zi[e] = z.y;
            }
#pragma unroll
            for (int ks = 0; ks < CL_NB / 4; ++ks) {
              const C b = Us[4 * ks + lk][col];
              zr = P::fma_sub(fa[ks].x, b.x, zr);
              zi = P::fma_sub(fa[ks].x, b.y, zi);
              zr = P::fma_add(fa[ks].y, b.y, zr);
              zi = P::fma_sub(fa[ks].y, b.x, zi);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = r0 + P::orow(lk, e);
              if (row < D && col < nc) zc[row] = mkc(zr[e], zi[e]);
            }
          }
        }
      }
      __syncthreads();
    }
  }
  if constexpr (RP > 0) {  // the block's swaps on the other columns of W and on perm
    if (tid < 64) list_moved_rows(piv, k0, nb, map_b, k0, mv_dst, mv_src, &mv_n);
    __syncthreads();
    if (mv_n) {
      moved = 1;
      const int px = tid < mv_n ? perm[mv_src[tid]] : 0;
      __syncthreads();
      if (tid < mv_n) perm[mv_dst[tid]] = px;
      move_rows_waves<R, 8>(W, D, 0, k0, mv_dst, mv_src, mv_n);
      move_rows_waves<R, 8>(W, D, k0 + nb, D, mv_dst, mv_src, mv_n);
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (info) atomicCAS(a.info, 0, info);
    if (moved) perm[D] = 1;
  }
}

// grid: matrices
template <class R>
__global__ __launch_bounds__(256, 2) void closed_diag(ClosedArgs a, int k0) {
  using C = typename Prec<R>::C;
  __shared__ C block[CL_BB][CL_BB + 1];
  __shared__ C dinv[CL_BB];  // reciprocals of U11's diagonal
  const int mat = blockIdx.x, D = a.D, nb = min(CL_BB, D - k0), nblk = (D + CL_BB - 1) / CL_BB;
  const C* W = static_cast<const C*>(a.W) + (size_t)mat * D * D;
  // column-major, leading dimension CL_BB
  C* Linv = static_cast<C*>(a.T) + ((size_t)mat * nblk + k0 / CL_BB) * 2 * CL_BB * CL_BB;
  C* Uinv = Linv + CL_BB * CL_BB;
  const int tid = threadIdx.x;
  const C one = mkc((R)1, (R)0), zero = mkc((R)0, (R)0);
  // L11^-1 and U11^-1 (identity-padded to CL_BB) in place in LDS, where the block lies
  // packed (L below, U on and above the diagonal): the inverses of the four diagonal 16 x
  // 16 blocks of each (a column per thread, in registers), then, block column by block
  // column from where the inverse is done, on MFMA
  //   Linv(a, b) = -sum_{c = b+1}^{a} Linv(a, c) L(c, b) Linv(b, b)    b = 2, 1, 0
  //   Uinv(a, b) = -sum_{c = a}^{b-1} Uinv(a, c) U(c, b) Uinv(b, b)    b = 1, 2, 3
  {
    using P = Prec<R>;
    using V = typename P::V;
    constexpr int LD = CL_BB + 1;  // a column's stride, free of bank conflicts
    C* B = &block[0][0];           // B[col LD + row]
    for (int u = tid; u < CL_BB * CL_BB; u += 256) {
      const int i = u % CL_BB, j = u / CL_BB;
      B[j * LD + i] = (i < nb && j < nb) ? W[(size_t)(k0 + j) * D + k0 + i] : (i == j ? one : zero);
    }
    __syncthreads();
    if (tid < CL_BB) dinv[tid] = cinv(B[tid * LD + tid]);
    __syncthreads();
    {
      const bool up = tid >= CL_BB;
      const int t = tid % CL_NB, off = (tid / CL_NB) % (CL_BB / CL_NB) * CL_NB;
      const C* Md = B + off * LD + off;
      C x[CL_NB];  // column t of the diagonal block's inverse
      if (tid < CL_BB) {
#pragma unroll
        for (int i = 0; i < CL_NB; ++i) {
          __builtin_amdgcn_sched_barrier(0);
          C v = i == t ? one : zero;
#pragma unroll
          for (int s2 = 0; s2 < i; ++s2)
            if (s2 >= t) v = csub(v, cmul(Md[s2 * LD + i], x[s2]));
          x[i] = v;
        }
      } else if (tid < 2 * CL_BB) {
#pragma unroll
        for (int i = CL_NB - 1; i >= 0; --i) {
          __builtin_amdgcn_sched_barrier(0);
          C v = i == t ? one : zero;
#pragma unroll
          for (int s2 = i + 1; s2 < CL_NB; ++s2)
            if (s2 <= t) v = csub(v, cmul(Md[s2 * LD + i], x[s2]));
          x[i] = cmul(v, dinv[off + i]);
        }
      }
      __syncthreads();
      if (tid < 2 * CL_BB) {
        C* out = B + (off + t) * LD + off;
#pragma unroll
        for (int i = 0; i < CL_NB; ++i)
          if (up ? i <= t : i > t) out[i] = x[i];
      }
      __syncthreads();
    }
    const int lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = lane >> 4;
    // entry (i, k) of a diagonal block's inverse, whose other triangle is not its own
    auto diag = [&](bool up, C v, int i, int k) -> C {
      if (up) return i <= k ? v : zero;
      return i > k ? v : (i == k ? one : zero);
    };
    for (int st = 0; st < CL_BB / CL_NB - 1; ++st) {
      // 2 (st + 1) blocks, up to two a wave: those of L's column 2 - st, then U's st + 1
      V yr[2], yi[2];
      int ba[2], bb[2];
      bool upp[2], has[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int job = wave + 4 * q;
        has[q] = job < 2 * (st + 1);
        upp[q] = job > st;
        bb[q] = upp[q] ? st + 1 : 2 - st;
        ba[q] = upp[q] ? job - (st + 1) : bb[q] + 1 + job;
#pragma unroll
        for (int e = 0; e < 4; ++e) yr[q][e] = yi[q][e] = 0;
        if (!has[q]) continue;
        const int cb = upp[q] ? ba[q] : bb[q] + 1, ce = upp[q] ? bb[q] - 1 : ba[q];
        for (int c = cb; c <= ce; ++c)
#pragma unroll
          for (int ks = 0; ks < CL_NB / 4; ++ks) {
            const int kk = 4 * ks + lk;
            C x = B[(c * CL_NB + kk) * LD + ba[q] * CL_NB + li];
            if (c == ba[q]) x = diag(upp[q], x, li, kk);
            const C y = B[(bb[q] * CL_NB + li) * LD + c * CL_NB + kk];
            yr[q] = P::fma_add(x.x, y.x, yr[q]);
            yi[q] = P::fma_add(x.x, y.y, yi[q]);
            yr[q] = P::fma_sub(x.y, y.y, yr[q]);
            yi[q] = P::fma_add(x.y, y.x, yi[q]);
          }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (has[q])
#pragma unroll
          for (int e = 0; e < 4; ++e)
            B[(bb[q] * CL_NB + li) * LD + ba[q] * CL_NB + P::orow(lk, e)] = mkc(yr[q][e], yi[q][e]);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) yr[q][e] = yi[q][e] = 0;
        if (!has[q]) continue;
#pragma unroll
        for (int ks = 0; ks < CL_NB / 4; ++ks) {
          const int kk = 4 * ks + lk;
          const C x = B[(bb[q] * CL_NB + kk) * LD + ba[q] * CL_NB + li];
          const C y = diag(upp[q], B[(bb[q] * CL_NB + li) * LD + bb[q] * CL_NB + kk], kk, li);
          yr[q] = P::fma_sub(x.x, y.x, yr[q]);
          yi[q] = P::fma_sub(x.x, y.y, yi[q]);
          yr[q] = P::fma_add(x.y, y.y, yr[q]);
          yi[q] = P::fma_sub(x.y, y.x, yi[q]);
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (has[q])
#pragma unroll
          for (int e = 0; e < 4; ++e)
            B[(bb[q] * CL_NB + li) * LD + ba[q] * CL_NB + P::orow(lk, e)] = mkc(yr[q][e], yi[q][e]);
      __syncthreads();
    }
    for (int u = tid; u < CL_BB * CL_BB; u += 256) {
      const int i = u % CL_BB, j = u / CL_BB;
      const C v = B[j * LD + i];
      Linv[u] = i > j ? v : (i == j ? one : zero);
      Uinv[u] = i <= j ? v : zero;
    }
  }
}

// ---- refinement products ------------------------------------------------------------

struct IrArgs {
  const double2* gam[4];
  double2* x[4];             // X_r, the solution, in the output arrays
  const float2* inv;         // [mat][2D][D]: the inverse is columns D..2D-1
  float2* y;                 // the last product with A32^-1: matrix mat at y + ys mat
  size_t ys;
  float2* rhs;               // [mat][D][D] right-hand side of the next product: fp32(Gamma), then fp32(R)
  const double2* gx;         // [mat][D][D] Gamma chi
  double* part;              // [mat][tiles][2]: sum |R|^2, sum |Gamma|^2 per tile
  double* res;               // [mat] |R|_F / |Gamma|_F
  unsigned long long* rmax;  // bits of the largest res (non-negative doubles order as integers)
  int D, q0, nqb, tiles_n;
  double kappa[4];
};

__global__ void ir_clear(unsigned long long* rmax) { *rmax = 0ull; }

// Chunks of the inner index in the products below: 16 KiB a stage (A and B), three
// stages, so two chunks are in flight while one multiplies and three workgroups share a
// CU.
template <class R>
constexpr int tile_kc() {
  return sizeof(R) == 8 ? 8 : 16;
}
constexpr int TILE_STAGES = 3;

// One factor pair of a tile product: A(row, k) = a[k lda + row], B(k, col) = b[col ldb + k],
// k < len.  16-byte aligned, lda, ldb and len even.
template <class C>
struct TileSeg {
  const C* a;
  const C* b;
  int lda, len;
};

// A 64 x 64 tile of A1 B1 + A2 B2 (s1.len a multiple of the chunk, possibly 0) by a ring of
// LDS stages filled with direct global-to-LDS loads; four waves of 2 x 2 blocks of 16 x 16
// x 4 MFMAs.  One barrier per chunk: after it every wave is done with the chunk before,
// whose stage takes the chunk two ahead.  A stage holds A as [k][row] and B as
// [column][k], its 16-byte pieces (a double2, two float2) XOR-swizzled by the column, so 8
// consecutive lanes of a fragment read cover 32 banks or more.  Rows from `rows`, columns
// from `cols` and inner indices from s2.len on load clamped addresses: such inner indices
// are zeroed in the last chunk, rows and columns dropped by the caller.
// The register-fed form without prefetch took 11.39 ms for the FP64 residual (and 4.08 ms
// more to form chi X) at D = 320, 480 q; this one 7.43 ms (68 TFLOP/s).
template <class R>
__device__ __forceinline__ void tile_product(TileSeg<typename Prec<R>::C> s1, TileSeg<typename Prec<R>::C> s2, int ldb,
                                             int rows, int cols, char* lds, typename Prec<R>::V (&ar)[2][2],
                                             typename Prec<R>::V (&ai)[2][2]) {
  using P = Prec<R>;
  using C = typename P::C;
  constexpr int KC = tile_kc<R>();
  constexpr int E = 16 / sizeof(C);           // elements of a 16-byte piece
  constexpr int RP = CL_T / E, KP = KC / E;   // pieces per row of A (one k) and per column of B
  constexpr int STAGE = 2 * KC * CL_T * (int)sizeof(C), HALF = STAGE / 2;
  static_assert(HALF == 8192 && KP == 8, "16 KiB stages of 8 pieces a column");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  const int n1 = s1.len / KC, nch = n1 + (s2.len + KC - 1) / KC;
  const unsigned lbase = lds_addr(lds);
  // this lane's pieces: of A, slots (wave + 4 v) 64 + lane -> k = slot / RP, piece slot % RP;
  // of B, slot -> column slot / 8, piece (slot % 8) ^ (column % 8).  Their byte offsets from
  // a chunk's first element: a whole chunk costs no address arithmetic beyond its base.
  unsigned oa1[2], oa2[2], ob[2];
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    const int slot = (wave + 4 * v) * 64 + lane;
    const int row = min((slot % RP) * E, rows - E);
    oa1[v] = (unsigned)(((slot / RP) * s1.lda + row) * (int)sizeof(C));
    oa2[v] = (unsigned)(((slot / RP) * s2.lda + row) * (int)sizeof(C));
    ob[v] = (unsigned)(((size_t)min(slot / KP, cols - 1) * ldb + ((slot % KP) ^ ((slot / KP) % KP)) * E) * sizeof(C));
  }
  auto issue = [&](int ch) {
    const unsigned st = lbase + (ch % TILE_STAGES) * STAGE;
    if (ch < n1) {
#pragma unroll
      for (int v = 0; v < 2; ++v) dma16(s1.a + (size_t)ch * KC * s1.lda, oa1[v], st + (wave + 4 * v) * 1024);
#pragma unroll
      for (int v = 0; v < 2; ++v) dma16(s1.b + ch * KC, ob[v], st + HALF + (wave + 4 * v) * 1024);
      return;
    }
    const int k0 = (ch - n1) * KC;
    if (k0 + KC <= s2.len) {
#pragma unroll
      for (int v = 0; v < 2; ++v) dma16(s2.a + (size_t)k0 * s2.lda, oa2[v], st + (wave + 4 * v) * 1024);
#pragma unroll
      for (int v = 0; v < 2; ++v) dma16(s2.b + k0, ob[v], st + HALF + (wave + 4 * v) * 1024);
      return;
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int slot = (wave + 4 * v) * 64 + lane;
      const int k = min(slot / RP, s2.len - 1 - k0);
      dma16(s2.a + (size_t)k0 * s2.lda, (unsigned)((k * s2.lda + min((slot % RP) * E, rows - E)) * (int)sizeof(C)),
            st + (wave + 4 * v) * 1024);
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const int slot = (wave + 4 * v) * 64 + lane;
      const int k = min(((slot % KP) ^ ((slot / KP) % KP)) * E, s2.len - E - k0);
      dma16(s2.b + k0, (unsigned)(((size_t)min(slot / KP, cols - 1) * ldb + k) * sizeof(C)),
            st + HALF + (wave + 4 * v) * 1024);
    }
  };
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) ar[i][j][e] = ai[i][j][e] = 0;
  stage_barrier();  // the stages' last readers are done
  issue(0);
  if (nch > 1) issue(1);
  for (int ch = 0; ch < nch; ++ch) {
    // this wave's four loads of chunk ch have landed (those of ch + 1 may be in flight)
    if (ch + 1 < nch)
      wait_vmcnt<4>();
    else
      wait_vmcnt<0>();
    stage_barrier();
    if (ch + 2 < nch) issue(ch + 2);
    char* st = lds + (ch % TILE_STAGES) * STAGE;
    C* sa = reinterpret_cast<C*>(st);
    char* sb = st + HALF;
    auto b_at = [&](int col, int k) {
      return reinterpret_cast<C*>(sb + (col * KP + ((k / E) ^ (col % KP))) * 16 + (k % E) * sizeof(C));
    };
    const int left = s2.len - (ch - n1) * KC;
    if (ch >= n1 && left < KC) {  // the last chunk: zeros beyond the inner range
      for (int u = tid; u < (KC - left) * CL_T; u += 256) {
        const int k = left + u / CL_T, x = u % CL_T;
        sa[k * CL_T + x] = mkc((R)0, (R)0);
        *b_at(x, k) = mkc((R)0, (R)0);
      }
      __syncthreads();
    }
#pragma unroll
    for (int kk = 0; kk < KC; kk += 4) {
      const int k = kk + lk;
      C fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = sa[k * CL_T + wr + i * 16 + li];
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = *b_at(wc + j * 16 + li, k);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          ar[i][j] = P::fma_add(fa[i].x, fb[j].x, ar[i][j]);
          ai[i][j] = P::fma_add(fa[i].x, fb[j].y, ai[i][j]);
          ar[i][j] = P::fma_sub(fa[i].y, fb[j].y, ar[i][j]);
          ai[i][j] = P::fma_add(fa[i].y, fb[j].x, ai[i][j]);
        }
    }
  }
}

// ---- the block form's solves ---------------------------------------------------------

// Block rows scaled by the inverses of their diagonal blocks, in place and negated: left of
// the diagonal -L_kk^-1 L_ki, right of it -U_kk^-1 U_kj, so that a block row of a
// triangular solve is one product, its diagonal inverse times the right-hand side
// included.  grid: nblk (nblk - 1) blocks of every matrix
template <class R>
__global__ __launch_bounds__(256, 3) void closed_scale(ClosedArgs a) {
  using P = Prec<R>;
  using C = typename P::C;
  using V = typename P::V;
  __shared__ __attribute__((aligned(16))) char stage[TILE_STAGES * 16384];
  const int D = a.D, nblk = (D + CL_BB - 1) / CL_BB, per = nblk * (nblk - 1);
  const int logical = closed_xcd_remap(blockIdx.x, gridDim.x);
  const int mat = logical / per, t = logical - mat * per;
  const int kb = t / (nblk - 1), o = t - kb * (nblk - 1), ib = o < kb ? o : o + 1;
  const int k0 = kb * CL_BB, c0 = ib * CL_BB, nb = min(CL_BB, D - k0), nc = min(CL_BB, D - c0);
  C* W = static_cast<C*>(a.W) + (size_t)mat * D * D + (size_t)c0 * D + k0;
  const C* T = static_cast<const C*>(a.T) + (((size_t)mat * nblk + kb) * 2 + (ib < kb ? 0 : 1)) * CL_BB * CL_BB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32, li = lane & 15, lk = lane >> 4;
  V ar[2][2], ai[2][2];
  tile_product<R>({T, W, CL_BB, 0}, {T, W, CL_BB, nb}, D, CL_BB, nc, stage, ar, ai);
  // every wave's loads have landed before the last barrier: the block may be replaced
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = wr + i * 16 + P::orow(lk, e), col = wc + j * 16 + li;
        if (row < nb && col < nc) W[(size_t)col * D + row] = mkc(-ar[i][j][e], -ai[i][j][e]);
      }
}

// U12 = L11^-1 Z1 for a 64-column panel right of the block, in place; grid: the panels of
// every matrix
template <class R>
__global__ __launch_bounds__(256, 3) void closed_row(ClosedArgs a, int k0) {
  using P = Prec<R>;
  using C = typename P::C;
  using V = typename P::V;
  __shared__ __attribute__((aligned(16))) char stage[TILE_STAGES * 16384];
  const int D = a.D, nblk = (D + CL_BB - 1) / CL_BB, j0 = k0 + CL_BB, per = nblk - k0 / CL_BB - 1;
  const int logical = closed_xcd_remap(blockIdx.x, gridDim.x);
  const int mat = logical / per, c0 = j0 + (logical - mat * per) * CL_T, nc = min(CL_T, D - c0);
  C* Z = static_cast<C*>(a.W) + (size_t)mat * D * D + (size_t)c0 * D + k0;
  const C* T = static_cast<const C*>(a.T) + ((size_t)mat * nblk + k0 / CL_BB) * 2 * CL_BB * CL_BB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32, li = lane & 15, lk = lane >> 4;
  V ar[2][2], ai[2][2];
  tile_product<R>({T, Z, CL_BB, 0}, {T, Z, CL_BB, CL_BB}, D, CL_BB, nc, stage, ar, ai);
  // every wave's loads have landed before the last barrier: the panel may be replaced
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = wr + i * 16 + P::orow(lk, e), col = wc + j * 16 + li;
        if (col < nc) Z[(size_t)col * D + row] = mkc(ar[i][j][e], ai[i][j][e]);
      }
}

// Z -= L21 U12 for one 64 x 64 tile below and right of the block; grid: the tiles of every
// matrix
template <class R>
__global__ __launch_bounds__(256, 3) void closed_trail(ClosedArgs a, int k0) {
  using P = Prec<R>;
  using C = typename P::C;
  using V = typename P::V;
  __shared__ __attribute__((aligned(16))) char stage[TILE_STAGES * 16384];
  const int D = a.D, j0 = k0 + CL_BB, n = (D - j0 + CL_T - 1) / CL_T, per = n * n;
  const int logical = closed_xcd_remap(blockIdx.x, gridDim.x);
  const int mat = logical / per, t = logical - mat * per;
  const int r0 = j0 + t % n * CL_T, c0 = j0 + t / n * CL_T, nr = min(CL_T, D - r0), nc = min(CL_T, D - c0);
  C* W = static_cast<C*>(a.W) + (size_t)mat * D * D;
  C* Z = W + (size_t)c0 * D + r0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32, li = lane & 15, lk = lane >> 4;
  V ar[2][2], ai[2][2];
  const TileSeg<C> s{W + (size_t)k0 * D + r0, W + (size_t)c0 * D + k0, D, CL_BB};
  tile_product<R>({s.a, s.b, D, 0}, s, D, nr, nc, stage, ar, ai);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = wr + i * 16 + P::orow(lk, e), col = wc + j * 16 + li;
        if (row >= nr || col >= nc) continue;
        C* z = Z + (size_t)col * D + row;
        *z = csub(*z, mkc(ar[i][j][e], ai[i][j][e]));
      }
}

struct LuArgs {
  const double2* gam[4];
  double2* x[4];        // the output arrays: X (MODE 0: Phi)
  const void* W;        // scaled block rows
  const void* T;        // diagonal inverses
  const int* perm;
  const float2* rhs;    // refinement: [mat][D][D]
  float2* y;            // refinement: [mat][D][D] solution of the product in FP32
  int D, q0, nqb;
};

// X = U^-1 L^-1 P B for the 64 columns of one panel of one matrix: forward, then backward,
// a block row at a time, each one tile product whose inner index runs over the block rows
// that are done and its own right-hand side.  The panel lives in the output (direct) or in
// y (refinement); a block row is stored, and waited for, before the next one reads it.
// MFMA-bound: 9.6 D^3 flops with the diagonal inverses, the factors shared through L2 by
// the panels of a matrix, which run next to each other on one XCD.  D = 320, 480 q: 10.0 ms
// in FP64 (60 TFLOP/s executed), 5.6 to 6.6 in FP32 by mode.
//   MODE 0: FP64, B = Gamma, Phi = X - Gamma    MODE 1: X = fp64(A32^-1 rhs)
//   MODE 2: X += fp64(A32^-1 rhs)
// grid: ceil(D / 64) panels of every matrix
template <int MODE>
__global__ __launch_bounds__(256, 3) void closed_lu_solve(LuArgs a) {
  using R = typename std::conditional<MODE == 0, double, float>::type;
  using P = Prec<R>;
  using C = typename P::C;
  using V = typename P::V;
  __shared__ __attribute__((aligned(16))) char stage[TILE_STAGES * 16384];
  const int D = a.D, nblk = (D + CL_BB - 1) / CL_BB;
  const int logical = closed_xcd_remap(blockIdx.x, gridDim.x);
  const int mat = logical / nblk, c0 = (logical - mat * nblk) * CL_T;
  const int r = mat / a.nqb, q = a.q0 + (mat - r * a.nqb);
  const size_t DD = (size_t)D * D, base = DD * q + (size_t)c0 * D;
  const int nc = min(CL_T, D - c0);
  const double2* G = a.gam[r] + base;
  double2* X = a.x[r] + base;
  C* buf;
  const C* src;
  if constexpr (MODE == 0) {
    buf = X;
    src = G;
  } else {
    buf = a.y + DD * mat + (size_t)c0 * D;
    src = a.rhs + DD * mat + (size_t)c0 * D;
  }
  const C* W = static_cast<const C*>(a.W) + DD * mat;
  const C* T = static_cast<const C*>(a.T) + (size_t)mat * nblk * 2 * CL_BB * CL_BB;
  const int* perm = a.perm + (size_t)mat * (D + 1);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32, li = lane & 15, lk = lane >> 4;
  auto settle = [&]() {  // the stores of this workgroup are done, for its direct loads
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
  };
  if (perm[D]) {  // the factorisation moved rows: the panel in their order first
    for (int u = tid; u < nc * D; u += 256) {
      const int col = u / D, row = u - col * D;
      buf[(size_t)col * D + row] = src[(size_t)col * D + perm[row]];
    }
    settle();
    src = buf;
  }
  V ar[2][2], ai[2][2];
  auto store = [&](int k0, int nb, bool last) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = wr + i * 16 + P::orow(lk, e), col = wc + j * 16 + li;
          if (row >= nb || col >= nc) continue;
          const size_t at = (size_t)col * D + k0 + row;
          buf[at] = mkc(ar[i][j][e], ai[i][j][e]);
          if constexpr (MODE == 1) {
            if (last) X[at] = make_double2((double)ar[i][j][e], (double)ai[i][j][e]);
          } else if constexpr (MODE == 2) {
            if (last) {
              const double2 x = X[at];
              X[at] = make_double2(x.x + (double)ar[i][j][e], x.y + (double)ai[i][j][e]);
            }
          }
        }
    settle();
  };
  for (int kb = 0; kb < nblk; ++kb) {
    const int k0 = kb * CL_BB, nb = min(CL_BB, D - k0);
    tile_product<R>({W + k0, buf, D, k0}, {T + (size_t)kb * 2 * CL_BB * CL_BB, src + k0, CL_BB, nb}, D, nb, nc, stage,
                    ar, ai);
    store(k0, nb, false);
  }
  for (int kb = nblk - 1; kb >= 0; --kb) {
    const int k0 = kb * CL_BB, nb = min(CL_BB, D - k0), k1 = k0 + nb;
    const C* Ui = T + ((size_t)kb * 2 + 1) * CL_BB * CL_BB;
    if (k1 < D)
      tile_product<R>({Ui, buf + k0, CL_BB, nb}, {W + (size_t)k1 * D + k0, buf + k1, D, D - k1}, D, nb, nc, stage, ar,
                      ai);
    else
      tile_product<R>({Ui, buf + k0, CL_BB, 0}, {Ui, buf + k0, CL_BB, nb}, D, nb, nc, stage, ar, ai);
    store(k0, nb, true);
  }
  if constexpr (MODE == 0) {
    for (int u = tid; u < nc * D; u += 256) X[u] = csub(X[u], G[u]);
  }
}

// Batched complex products of the refinement, one 64 x 64 tile per workgroup, the tiles of
// a matrix on one XCD so that they share its L2.
//   MODE 0: X  = fp64(A32^-1 fp32(Gamma))    MODE 1: X += fp64(A32^-1 fp32(R))
//           (below the block form's orders, with the inverse that closed_solve leaves)
//   MODE 2: R  = Gamma - X + kappa (Gamma chi) X in FP64, kept as fp32(R), the only form a
//           product reads, with per-tile |R|^2, |Gamma|^2 of the FP64 values
// grid: tiles_n^2 * 4 nqb
template <int MODE>
__global__ __launch_bounds__(256, 3) void ir_gemm(IrArgs a) {
  using R = typename std::conditional<MODE == 2, double, float>::type;
  using P = Prec<R>;
  using C = typename P::C;
  using V = typename P::V;
  __shared__ __attribute__((aligned(16))) char stage[TILE_STAGES * 16384];
  const int tiles = a.tiles_n * a.tiles_n;
  const int logical = closed_xcd_remap(blockIdx.x, gridDim.x);
  const int mat = logical / tiles, t = logical - mat * tiles;
  const int tr = (t / a.tiles_n) * CL_T, tc = (t % a.tiles_n) * CL_T;
  const int r = mat / a.nqb, q = a.q0 + (mat - r * a.nqb);
  const int D = a.D;
  const size_t DD = (size_t)D * D;
  const double2* G = a.gam[r] + DD * q;
  double2* X = a.x[r] + DD * q;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  V ar[2][2], ai[2][2];
  const C *A, *B;
  if constexpr (MODE == 2) {
    A = a.gx + DD * mat + tr;
    B = X + (size_t)tc * D;
  } else {
    A = a.inv + 2 * DD * mat + DD + tr;
    B = a.rhs + DD * mat + (size_t)tc * D;
  }
  tile_product<R>({A, B, D, 0}, {A, B, D, D}, D, D - tr, D - tc, stage, ar, ai);
  double rr = 0.0, gg = 0.0;
  const double kap = a.kappa[r];
  float2* Rm = a.rhs + DD * mat;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = tr + wr + i * 16 + P::orow(lk, e), col = tc + wc + j * 16 + li;
        if (row >= D || col >= D) continue;
        const size_t idx = (size_t)col * D + row;
        if (MODE == 0) {
          X[idx] = make_double2((double)ar[i][j][e], (double)ai[i][j][e]);
        } else if (MODE == 1) {
          const double2 x = X[idx];
          X[idx] = make_double2(x.x + (double)ar[i][j][e], x.y + (double)ai[i][j][e]);
          a.y[a.ys * mat + idx] = make_float2((float)ar[i][j][e], (float)ai[i][j][e]);
        } else {
          const double2 g = G[idx], x = X[idx];
          const double2 v = make_double2(g.x - x.x + kap * ar[i][j][e], g.y - x.y + kap * ai[i][j][e]);
          Rm[idx] = make_float2((float)v.x, (float)v.y);
          rr += v.x * v.x + v.y * v.y;
          gg += g.x * g.x + g.y * g.y;
        }
      }
  if (MODE == 2) {
    double (*red)[256] = reinterpret_cast<double (*)[256]>(stage);
    __syncthreads();  // the stages are free
    red[0][tid] = rr;
    red[1][tid] = gg;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (tid < s) {
        red[0][tid] += red[0][tid + s];
        red[1][tid] += red[1][tid + s];
      }
      __syncthreads();
    }
    if (tid == 0) {
      a.part[2 * ((size_t)mat * tiles + t)] = red[0][0];
      a.part[2 * ((size_t)mat * tiles + t) + 1] = red[1][0];
    }
  }
}

// per matrix |R|_F / |Gamma|_F from the tile partials (fixed order), and the
// largest over the pass; grid: ceil(4 nqb / 256)
__global__ __launch_bounds__(256) void ir_check(IrArgs a, int mats) {
  const int mat = blockIdx.x * 256 + threadIdx.x;
  if (mat >= mats) return;
  const int tiles = a.tiles_n * a.tiles_n;
  double rr = 0.0, gg = 0.0;
  for (int t = 0; t < tiles; ++t) {
    rr += a.part[2 * ((size_t)mat * tiles + t)];
    gg += a.part[2 * ((size_t)mat * tiles + t) + 1];
  }
  // a NaN residual reports as infinity, so the pass never counts as converged
  const double v = gg > 0.0 ? sqrt(rr / gg) : (rr > 0.0 ? INFINITY : 0.0);
  const double s = v == v ? v : INFINITY;
  a.res[mat] = s;
  atomicMax(a.rmax, (unsigned long long)__double_as_longlong(s));
}

// X without its last correction; grid (ceil(D^2 / 256), 4 nqb)
__global__ __launch_bounds__(256) void ir_take_back(IrArgs a) {
  const int mat = blockIdx.y;
  const int r = mat / a.nqb, q = a.q0 + (mat - r * a.nqb);
  const size_t DD = (size_t)a.D * a.D;
  const size_t u = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= DD) return;
  double2* X = a.x[r] + DD * q;
  const float2 y = a.y[a.ys * mat + u];
  const double2 x = X[u];
  X[u] = make_double2(x.x - (double)y.x, x.y - (double)y.y);
}

// Phi = X - Gamma in place (X sits in the output array); grid (ceil(D^2 / 256), 4 nqb)
__global__ __launch_bounds__(256) void ir_final(IrArgs a) {
  const int mat = blockIdx.y;
  const int r = mat / a.nqb, q = a.q0 + (mat - r * a.nqb);
  const size_t DD = (size_t)a.D * a.D;
  const size_t u = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= DD) return;
  double2* X = a.x[r] + DD * q;
  const double2 g = a.gam[r][DD * q + u], x = X[u];
  X[u] = make_double2(x.x - g.x, x.y - g.y);
}

// ---- host -------------------------------------------------------------------------

// Workspace of one pass: up to 16 GiB (1024 q at D = 320 in one launch, so
// the workgroups' tail is paid once per call), at most half of the device
// memory that is free or already held by this workspace, at least 1 GiB.
static int closed_reserve(tups_ctx* c, size_t per_q, size_t extra, int* qbatch) {
  const tups_sizes& s = c->sz;
  size_t budget = (size_t)16 << 30, fr = 0, tot = 0;
  if (hipMemGetInfo(&fr, &tot) == hipSuccess)
    budget = std::min(budget, std::max((size_t)1 << 30, (fr + c->closed_ws_bytes) / 2));
  const size_t want = budget / per_q;
  *qbatch = (int)std::max<size_t>(1, std::min<size_t>(s.nq, want));
  const size_t need = per_q * *qbatch + extra + 256;
  if (c->closed_ws_bytes < need) {
    if (c->closed_ws) TUPS_HIP(hipFree(c->closed_ws));
    c->closed_ws = nullptr;
    c->closed_ws_bytes = 0;
    TUPS_HIP(hipMalloc(&c->closed_ws, need));
    c->closed_ws_bytes = need;
  }
  return TUPS_OK;
}

static void closed_common(tups_ctx* c, ClosedArgs& a) {
  const tups_sizes& s = c->sz;
  for (int r = 0; r < 4; ++r) {
    a.gam[r] = c->gamma[r];
    a.out[r] = c->spare[r];
  }
  a.chi[0] = c->chi[0];
  a.chi[1] = c->chi[1];
  a.info = static_cast<int*>(c->closed_ws);
  a.W = static_cast<char*>(c->closed_ws) + 256;
  a.D = s.nz;
  a.nf = s.nf;
  a.nl = s.nl;
  const double cr[4] = {0.5, 0.5, -0.25, 0.25};
  for (int r = 0; r < 4; ++r) a.kappa[r] = 2.0 * cr[r] * s.alpha;
}

// variants: 0 = Gauss-Jordan in CL_NB-wide panels (closed_solve), 1 = LU by
// CL_BB-wide blocks, 2 = the same with the sub-panels on registers (D <= 512;
// above that it runs as 1); -1 = 2 from D = 128 on
static const char* const kClosedVariants[] = {"gj_panel16", "gj_block64", "gj_block64_rp"};
constexpr int kClosedRp = 2;  // rows per thread of the register sub-panel
int closed_variant_count() { return 3; }
const char* closed_variant_name(int v) { return v >= 0 && v < 3 ? kClosedVariants[v] : ""; }
static bool closed_blocked(const tups_ctx* c) {
  return c->closed_variant >= 1 || (c->closed_variant < 0 && c->sz.nz >= 128);
}
static bool closed_regs(const tups_ctx* c) {
  return closed_blocked(c) && c->closed_variant != 1 && c->sz.nz <= 256 * kClosedRp;
}
static size_t closed_blocks(size_t D) { return (D + CL_BB - 1) / CL_BB; }
// per matrix of the block form: the factors and the diagonal inverses
static size_t closed_b64_elems(size_t D) { return D * D + 2 * closed_blocks(D) * CL_BB * CL_BB; }

// the block form's parts of a workspace from `at` on; returns its end
template <class C>
static int* place_b64(ClosedArgs& a, C* at, size_t mats) {
  const size_t D = a.D;
  a.W = at;
  at += mats * D * D;
  a.T = at;
  at += mats * closed_blocks(D) * 2 * CL_BB * CL_BB;
  a.perm = reinterpret_cast<int*>(at);
  return a.perm + mats * (D + 1);
}

// the factorisation of every matrix and the scaling of its block rows
template <class R>
static int factor_b64(tups_ctx* c, const ClosedArgs& a, unsigned mats) {
  const unsigned nblk = (unsigned)closed_blocks(a.D);
  const bool regs = closed_regs(c);
  for (unsigned kb = 0; kb < nblk; ++kb) {
    const int k0 = (int)kb * CL_BB, rows = a.D - k0;
    // the register sub-panel with the rows a thread needs; it starts at most 256 kClosedRp rows
    auto panel = !regs ? closed_panel<R, 0> : rows <= 256 ? closed_panel<R, 1> : closed_panel<R, kClosedRp>;
    hipLaunchKernelGGL(panel, dim3(mats), dim3(256), 0, c->stream, a, k0);
    TUPS_HIP(hipGetLastError());
    hipLaunchKernelGGL(closed_diag<R>, dim3(mats), dim3(256), 0, c->stream, a, k0);
    TUPS_HIP(hipGetLastError());
    const unsigned left = nblk - kb - 1;
    if (!left) break;
    hipLaunchKernelGGL(closed_row<R>, dim3(left * mats), dim3(256), 0, c->stream, a, k0);
    TUPS_HIP(hipGetLastError());
    hipLaunchKernelGGL(closed_trail<R>, dim3(left * left * mats), dim3(256), 0, c->stream, a, k0);
    TUPS_HIP(hipGetLastError());
  }
  if (nblk > 1) hipLaunchKernelGGL(closed_scale<R>, dim3(nblk * (nblk - 1) * mats), dim3(256), 0, c->stream, a);
  TUPS_HIP(hipGetLastError());
  return TUPS_OK;
}

static LuArgs lu_args(const tups_ctx* c, const ClosedArgs& a) {
  LuArgs l{};
  for (int r = 0; r < 4; ++r) {
    l.gam[r] = c->gamma[r];
    l.x[r] = c->spare[r];
  }
  l.W = a.W;
  l.T = a.T;
  l.perm = a.perm;
  l.D = a.D;
  l.q0 = a.q0;
  l.nqb = a.nqb;
  return l;
}

int launch_bse_closed(tups_ctx* c) {
  const tups_sizes& s = c->sz;
  const size_t D = s.nz;
  TUPS_CHECK(s.nl <= CL_NL_MAX, TUPS_EINVAL, "closed form: at most 9 form factors");
  const bool blk = closed_blocked(c);
  const size_t per_mat = blk ? closed_b64_elems(D) * sizeof(double2) + (D + 1) * sizeof(int) : 2 * D * D * sizeof(double2);
  int qbatch = 0;
  if (int rc = closed_reserve(c, 4 * per_mat, 0, &qbatch)) return rc;
  ClosedArgs a{};
  closed_common(c, a);
  a.blk = blk ? 1 : 0;
  if (blk) place_b64<double2>(a, static_cast<double2*>(a.W), 4 * (size_t)qbatch);
  hipLaunchKernelGGL(closed_clear, dim3(1), dim3(1), 0, c->stream, a.info);
  TUPS_HIP(hipGetLastError());
  for (int q0 = 0; q0 < s.nq; q0 += qbatch) {
    a.q0 = q0;
    a.nqb = std::min(qbatch, s.nq - q0);
    const unsigned mats = 4u * (unsigned)a.nqb;
    if (int rc = timer_begin(c)) return rc;
    hipLaunchKernelGGL((closed_build_nu<double2, false>), dim3((unsigned)s.nf, mats), dim3(256), 0, c->stream, a);
    TUPS_HIP(hipGetLastError());
    if (blk) {
      if (int rc = factor_b64<double>(c, a, mats)) return rc;
      hipLaunchKernelGGL(closed_lu_solve<0>, dim3((unsigned)closed_blocks(D) * mats), dim3(256), 0, c->stream,
                         lu_args(c, a));
    } else {
      hipLaunchKernelGGL((closed_solve<double, true>), dim3(mats), dim3(256), 0, c->stream, a);
    }
    TUPS_HIP(hipGetLastError());
    if (int rc = timer_end(c, TUPS_K_BSE_CLOSED)) return rc;
  }
  int info = 0;
  TUPS_HIP(hipMemcpyAsync(&info, a.info, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  TUPS_HIP(hipStreamSynchronize(c->stream));
  TUPS_CHECK(info == 0, TUPS_ENONFINITE, "closed-form BSE: singular I - kappa Gamma chi (zero pivot column)");
  c->ir_steps = 0;
  c->ir_residual = NAN;
  return TUPS_OK;
}

// A tolerance of the refinement up to here asks for all that FP64 gives: one step leaves
// 1e-13 to 9e-13 (D = 16 to 576), between which and the tolerance chance would decide whether X
// is exact to 1e-12 or to 1e-15.  Above it X is wanted as soon as it meets the tolerance.  The step
// beyond and its residual cost 14 of 50 ms at D = 320, 480 q.
constexpr double kIrFull = 0x1p-36;

int launch_bse_closed_ir(tups_ctx* c) {
  const tups_sizes& s = c->sz;
  TUPS_CHECK(s.nl <= CL_NL_MAX, TUPS_EINVAL, "closed form: at most 9 form factors");
  const size_t D = s.nz, DD = D * D;
  const int tiles_n = (int)((D + CL_T - 1) / CL_T);
  // per matrix: [A32 | I] (2 D^2 float2) or the block form's factors and a product's solution, the
  // rounded right-hand side (D^2 float2), Gamma chi (D^2 double2), tile partials, res
  const bool blk = closed_blocked(c);
  const size_t per_mat = DD * sizeof(float2) + DD * sizeof(double2) +
                         (size_t)tiles_n * tiles_n * 2 * sizeof(double) + sizeof(double) + 64 +
                         (blk ? (DD + closed_b64_elems(D)) * sizeof(float2) + (D + 1) * sizeof(int)
                              : 2 * DD * sizeof(float2));
  int qbatch = 0;
  if (int rc = closed_reserve(c, 4 * per_mat, 256, &qbatch)) return rc;
  ClosedArgs a{};
  closed_common(c, a);
  IrArgs b{};
  for (int r = 0; r < 4; ++r) {
    b.gam[r] = c->gamma[r];
    b.x[r] = c->spare[r];
    b.kappa[r] = a.kappa[r];
  }
  b.D = a.D;
  b.tiles_n = tiles_n;
  const size_t mats_max = 4 * (size_t)qbatch;
  char* base = static_cast<char*>(a.W);
  b.gx = a.gx = reinterpret_cast<double2*>(base);
  base += mats_max * DD * sizeof(double2);
  b.rhs = a.g32 = reinterpret_cast<float2*>(base);
  base += mats_max * DD * sizeof(float2);
  a.blk = blk ? 1 : 0;
  float2* y32 = nullptr;
  if (blk) {
    y32 = reinterpret_cast<float2*>(base);
    base = reinterpret_cast<char*>(place_b64<float2>(a, y32 + mats_max * DD, mats_max));
  } else {
    a.W = base;
    b.inv = reinterpret_cast<const float2*>(base);
    base += mats_max * 2 * DD * sizeof(float2);
  }
  // the corrections: the block form's product, or the columns that the elimination has used up
  b.y = blk ? y32 : static_cast<float2*>(a.W);
  b.ys = blk ? DD : 2 * DD;
  base = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(base) + 15) / 16 * 16);
  b.part = reinterpret_cast<double*>(base);
  base += mats_max * tiles_n * tiles_n * 2 * sizeof(double);
  b.res = reinterpret_cast<double*>(base);
  base += mats_max * sizeof(double);
  b.rmax = reinterpret_cast<unsigned long long*>((reinterpret_cast<uintptr_t>(base) + 63) / 64 * 64);
  hipLaunchKernelGGL(closed_clear, dim3(1), dim3(1), 0, c->stream, a.info);
  TUPS_HIP(hipGetLastError());
  int steps_max = 0;
  double res_max = 0.0;
  for (int q0 = 0; q0 < s.nq; q0 += qbatch) {
    a.q0 = b.q0 = q0;
    a.nqb = b.nqb = std::min(qbatch, s.nq - q0);
    const unsigned mats = 4u * (unsigned)a.nqb;
    const unsigned gblk = (unsigned)(tiles_n * tiles_n) * mats;
    if (int rc = timer_begin(c)) return rc;
    hipLaunchKernelGGL((closed_build_nu<float2, true>), dim3((unsigned)s.nf, mats), dim3(256), 0, c->stream, a);
    TUPS_HIP(hipGetLastError());
    LuArgs lu{};
    const unsigned glu = (unsigned)closed_blocks(D) * mats;
    if (blk) {
      if (int rc = factor_b64<float>(c, a, mats)) return rc;
      lu = lu_args(c, a);
      lu.rhs = b.rhs;
      lu.y = y32;
      // X = A32^-1 Gamma
      hipLaunchKernelGGL(closed_lu_solve<1>, dim3(glu), dim3(256), 0, c->stream, lu);
    } else {
      hipLaunchKernelGGL((closed_solve<float, false>), dim3(mats), dim3(256), 0, c->stream, a);
      TUPS_HIP(hipGetLastError());
      hipLaunchKernelGGL(ir_gemm<0>, dim3(gblk), dim3(256), 0, c->stream, b);
    }
    TUPS_HIP(hipGetLastError());
    int steps = 0;
    // beyond: X has had a step beyond the X that met the tolerance; back: that step was taken back
    bool beyond = false, back = false;
    double res = INFINITY;
    const dim3 all((unsigned)((DD + 255) / 256), mats);
    for (;;) {
      hipLaunchKernelGGL(ir_clear, dim3(1), dim3(1), 0, c->stream, b.rmax);
      TUPS_HIP(hipGetLastError());
      hipLaunchKernelGGL(ir_gemm<2>, dim3(gblk), dim3(256), 0, c->stream, b);
      TUPS_HIP(hipGetLastError());
      hipLaunchKernelGGL(ir_check, dim3((mats + 255) / 256), dim3(256), 0, c->stream, b, (int)mats);
      TUPS_HIP(hipGetLastError());
      unsigned long long bits = 0;
      TUPS_HIP(hipMemcpyAsync(&bits, b.rmax, sizeof(bits), hipMemcpyDeviceToHost, c->stream));
      TUPS_HIP(hipStreamSynchronize(c->stream));
      std::memcpy(&res, &bits, sizeof(res));
      const bool done = res <= c->ir_tol;
      if (beyond && !done) {
        // with a badly conditioned A a step need not make X better
        hipLaunchKernelGGL(ir_take_back, all, dim3(256), 0, c->stream, b);
        TUPS_HIP(hipGetLastError());
        --steps;
        beyond = false;
        back = true;
        continue;
      }
      // done: the step beyond makes a first solve that is just good enough no less exact than
      // one that just missed the tolerance and was refined
      const bool more = done ? c->ir_tol <= kIrFull && res > 0x1p-50 : true;
      if (beyond || back || !more || steps >= c->ir_max_steps) break;
      // X += A32^-1 R
      if (blk)
        hipLaunchKernelGGL(closed_lu_solve<2>, dim3(glu), dim3(256), 0, c->stream, lu);
      else
        hipLaunchKernelGGL(ir_gemm<1>, dim3(gblk), dim3(256), 0, c->stream, b);
      TUPS_HIP(hipGetLastError());
      ++steps;
      beyond = done;
    }
    hipLaunchKernelGGL(ir_final, all, dim3(256), 0, c->stream, b);
    TUPS_HIP(hipGetLastError());
    if (int rc = timer_end(c, TUPS_K_BSE_IR)) return rc;
    steps_max = std::max(steps_max, steps);
    res_max = std::max(res_max, res);
    if (!(res <= c->ir_tol)) break;
  }
  int info = 0;
  TUPS_HIP(hipMemcpyAsync(&info, a.info, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  TUPS_HIP(hipStreamSynchronize(c->stream));
  c->ir_steps = steps_max;
  c->ir_residual = res_max;
  TUPS_CHECK(info == 0, TUPS_ENONFINITE, "refined closed-form BSE: singular fp32(I - kappa Gamma chi) (zero pivot)");
  TUPS_CHECK(res_max <= c->ir_tol, TUPS_ENOCONV,
             "refined closed-form BSE: the residual did not reach the tolerance within the step limit");
  return TUPS_OK;
}

}  // namespace tups
