// Kernels of the ocean-core time step (everything except the 2D Helmholtz
// solve, which lives in hoc_helmholtz.hip).
//
// Two launch shapes:
//   column kernels: one lane per (j, i) column, marching k; lanes are
//     consecutive in i, so every level's load is one coalesced row segment,
//     issued a few levels before it is used (march_down, march_up).
//     Used where the work is a recurrence in k (tridiagonal sweeps, prefix
//     sums, the TKE mixing-length march) and the horizontal stencil at each
//     level is fused into the same pass.
//   cell kernels: one lane per (k, j, i) for the pure 3D stencils.
//
// Column recurrences keep their forward-sweep values (c*, d*) in LDS where the
// column fits (COL_LDS_MAX; the closure's rule is narrower), in global scratch
// for deeper ones.
#include <type_traits>

#include "hoc_device.h"
#include "hoc_kernels.h"

namespace hoc {

// Columns of a column kernel's workgroup: one wave, so that a grid of few
// columns spreads over as many compute units as it can.
constexpr int COLS = 64;
// Sweeps keep a column in LDS up to here (two or more workgroups per compute
// unit); deeper columns use the global work arrays.
constexpr size_t COL_LDS_MAX = 64 * 1024;
constexpr long long CUS = 256, CU_LDS = 160 * 1024;  // compute units, LDS of one
static unsigned column_blocks(const Dims& d) { return (unsigned)((d.n2 + COLS - 1) / COLS); }

// go(zc, stage) with the two flags as compile-time constants.
template <class Go>
static void with_column_form(bool zcol, bool stage, const Go& go) {
  using T = std::true_type;
  using F = std::false_type;
  if (zcol) {
    if (stage) go(T{}, T{});
    else go(T{}, F{});
  } else {
    if (stage) go(F{}, T{});
    else go(F{}, F{});
  }
}

// ------------------------------------------------------------ geometry
// Interface thickness of dz3 (libs/core/vertical_var.py:21-32) and the
// surface stress per unit density on faces, (tau / rho0) * mask3[u|v][0]
// (libs/core/model3d_v05.py:355-356).
__global__ void k_geometry(Dims d, StepParams p, const double* __restrict__ dz3,
                           const uint8_t* __restrict__ m3u, const uint8_t* __restrict__ m3v,
                           const double* __restrict__ tau_x, const double* __restrict__ tau_y,
                           double* __restrict__ dzi, double* __restrict__ tau_u,
                           double* __restrict__ tau_v) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const int nz = d.nz;
  const long long n2 = d.n2;
  dzi[c] = dz3[c];
  for (int k = 1; k < nz; ++k) dzi[k * n2 + c] = 0.5 * (dz3[(k - 1) * n2 + c] + dz3[k * n2 + c]);
  dzi[nz * n2 + c] = dz3[(nz - 1) * n2 + c];
  tau_u[c] = (tau_x[c] / p.rho0) * mk(m3u[c]);
  tau_v[c] = (tau_y[c] / p.rho0) * mk(m3v[c]);
}

// ------------------------------------------ moving vertical coordinates
// z* and sigma (libs/core/domain.py layer_thickness / face_thickness /
// depth_at_centres, rebuilt from eta every step, model3d_v05.py:128-139):
// dz3 = dz3_ref * (1 + eta / H) in wet columns, centre depths from the
// surface, interface spacing; then the face thickness by the face rule.
__global__ void k_moving_dz(Dims d, const uint8_t* __restrict__ m2, const double* __restrict__ H,
                            const double* __restrict__ eta, const double* __restrict__ dz3_ref,
                            double* __restrict__ dz3, double* __restrict__ zc,
                            double* __restrict__ dzi) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const long long n2 = d.n2;
  const int nz = d.nz;
  const double scale = m2[c] ? 1.0 + eta[c] / (H[c] > 0.0 ? H[c] : 1.0) : 1.0;
  double above = 0.0, prev = 0.0;
  for (int k = 0; k < nz; ++k) {
    const double dz = dz3_ref[k * n2 + c] * scale;
    dz3[k * n2 + c] = dz;
    if (k == 1) above = prev;
    else if (k > 1) above = above + prev;
    zc[k * n2 + c] = above + 0.5 * dz;
    dzi[k * n2 + c] = (k == 0) ? dz : 0.5 * (prev + dz);
    prev = dz;
  }
  dzi[nz * n2 + c] = prev;
}

__global__ void k_moving_faces(Dims d, StepParams p, const uint8_t* __restrict__ m3u,
                               const uint8_t* __restrict__ m3v, const double* __restrict__ dz3,
                               double* __restrict__ dz3u, double* __restrict__ dz3v) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.n3) return;
  const long long c = t % d.n2, o = t - c;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const long long ce = at2(d, j, wrap(i, 1, d.nx)), cn = at2(d, wrap(j, 1, d.ny), i);
  dz3u[t] = mk(m3u[t]) * face_value(p.face_rule, dz3[t], dz3[o + ce]);
  dz3v[t] = mk(m3v[t]) * face_value(p.face_rule, dz3[t], dz3[o + cn]);
}

// ---------------------------------------------------------- TKE closure
// libs/core/closure.py:141-205 in three passes over [nz+1][ny][nx] interface
// fields:
//   k_closure_lengths (integral form) or k_closure_shear + k_mixing_recursive
//     (recursive form): N^2 and shear^2 (s_n2, s_sh) and the mixing lengths
//     l_k = max(l_min, sqrt(l_up l_dn)) (s_l), l_eps = max(l_min, min(l_up,
//     l_dn)) (s_le);
//   k_closure: per column, the implicit interface tridiagonal for e (c* in
//     s_c, d* in e_out), then back-substitution, floors, K_m and K_h.

// N^2 and shear^2 on interface k of column c (closure.py:43-62,150-156).
__device__ __forceinline__ void shear_n2(const Dims& d, const StepParams& p, const Geo& geo,
                                         const double* u, const double* v, const double* b,
                                         long long c, int k, double& n2k, double& sh) {
  n2k = 0.0;
  sh = 0.0;
  if (k < 1 || k >= d.nz) return;
  const ColumnGeo cg(geo, p, d, c);
  const long long n2 = d.n2;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const long long cw = at2(d, j, wrap(i, -1, d.nx));
  const long long cs = at2(d, wrap(j, -1, d.ny), i);
  const long long a = (long long)(k - 1) * n2, o = (long long)k * n2;
  const double uc_prev = 0.5 * (u[a + c] + u[a + cw]);
  const double vc_prev = 0.5 * (v[a + c] + v[a + cs]);
  const double uc = 0.5 * (u[o + c] + u[o + cw]);
  const double vc = 0.5 * (v[o + c] + v[o + cs]);
  const double wet = (cg.wet(k - 1) ? 1.0 : 0.0) * (cg.wet(k) ? 1.0 : 0.0);
  const double idz = safe_inv(cg.dzi(k));
  const double du = (uc_prev - uc) * idz;
  const double dv = (vc_prev - vc) * idz;
  const double db = (b[a + c] - b[o + c]) * idz;
  sh = (du * du + dv * dv) * wet;
  n2k = db * wet;
}

// Integral (Gaspar) mixing lengths, closure.py:65-103. A workgroup owns
// MX_COLS consecutive columns: N^2 (clamped at 0) and the interface
// thicknesses of all their interfaces are staged in LDS once, then
// MX_TPC lanes per column march the interfaces k, k + MX_TPC, ... from LDS.
// Each march is the reference's loop with two exact shortcuts: it stops
// once the budget is spent (l and the budget are then frozen), and it skips
// the interfaces above the column's first and below its last one with
// N^2 != 0 or dz != 0 (a march from a dry interface under the bottom starts
// at the bottom), since a step across them changes neither l nor the budget.
constexpr int MX_COLS = 64, MX_TPC = 8, MX_THREADS = MX_COLS * MX_TPC;

__global__ __launch_bounds__(MX_THREADS) void k_closure_lengths(
    Dims d, StepParams p, Geo geo, const double* __restrict__ e_in, const double* __restrict__ u,
    const double* __restrict__ v, const double* __restrict__ b, double* __restrict__ s_n2,
    double* __restrict__ s_sh, double* __restrict__ s_l, double* __restrict__ s_le) {
  extern __shared__ double mx_lds[];
  __shared__ int kbeg[MX_COLS], kend[MX_COLS];
  const int nz = d.nz, ni = nz + 1;
  const long long n2 = d.n2;
  double* n2p = mx_lds;                 // [ni][MX_COLS] max(N^2, 0)
  double* dzl = mx_lds + ni * MX_COLS;  // [ni][MX_COLS] interface thickness
  const long long c0 = (long long)blockIdx.x * MX_COLS;
  for (int t = threadIdx.x; t < ni * MX_COLS; t += MX_THREADS) {
    const int kk = t / MX_COLS, col = t % MX_COLS;
    const long long c = c0 + col;
    double n2k = 0.0, sh = 0.0, dz = 0.0;
    if (c < n2) {
      shear_n2(d, p, geo, u, v, b, c, kk, n2k, sh);
      dz = ColumnGeo(geo, p, d, c).dzi(kk);
      s_n2[(long long)kk * n2 + c] = n2k;
      s_sh[(long long)kk * n2 + c] = sh;
    }
    n2p[t] = nmax(n2k, 0.0);
    dzl[t] = dz;
  }
  __syncthreads();
  if (threadIdx.x < MX_COLS) {
    const int col = threadIdx.x;
    int lo = ni, hi = -1;
    for (int kk = 0; kk < ni; ++kk) {
      const bool live = n2p[kk * MX_COLS + col] != 0.0 || dzl[kk * MX_COLS + col] != 0.0;
      if (live) {
        lo = kk < lo ? kk : lo;
        hi = kk;
      }
    }
    kbeg[col] = lo;
    kend[col] = hi + 1;
  }
  __syncthreads();
  const int col = threadIdx.x % MX_COLS, k0 = threadIdx.x / MX_COLS;
  const long long c = c0 + col;
  if (c >= n2) return;
  const int lo = kbeg[col], hi = kend[col];
  const ColumnGeo cg(geo, p, d, c);
  // column depth and the depth of interface k: dz3[0] + ... + dz3[k-1], in
  // that order
  double h = 0.0, zi = 0.0;
  if (cg.col) {
    h = cg_above(geo.zs, cg.nw, cg.hb, nz);
  } else {
    for (int k = 0; k < nz; ++k) h = h + geo.dz3[(long long)k * n2 + c];
  }
  int kz = 0;
  for (int k = k0; k <= nz; k += MX_TPC) {
    if (cg.col) {
      zi = cg_above(geo.zs, cg.nw, cg.hb, k);
    } else {
      for (; kz < k; ++kz) zi = zi + geo.dz3[(long long)kz * n2 + c];
    }
    const long long o = (long long)k * n2 + c;
    const double wet =
        (k >= 1 && k < nz) ? (cg.wet(k - 1) ? 1.0 : 0.0) * (cg.wet(k) ? 1.0 : 0.0) : 0.0;
    const double budget0 = nmax(e_in[o], p.e_min);
    // upward: interface k crosses k-1, ..., 0
    double l = 0.0, bud = budget0;
    for (int kk = (k - 1 < hi - 1 ? k - 1 : hi - 1); kk >= lo && bud > 0.0; --kk) {
      const double n2j = n2p[kk * MX_COLS + col];
      const double dzj = dzl[kk * MX_COLS + col];
      const double cost = n2j * dzj * (l + 0.5 * dzj);
      double step;
      if (cost <= bud) {
        step = dzj;
        bud = bud - cost;
      } else {
        if (n2j > 0.0) {
          const double s = sqrt(nmax(l * l + 2.0 * bud / n2j, 0.0)) - l;
          step = nmin(nmax(s, 0.0), dzj);
        } else {
          step = dzj;
        }
        bud = 0.0;
      }
      l = l + step;
    }
    const double l_up = nmin(l, zi + p.z_0) * wet;
    // downward: interface k crosses k+1, ..., nz
    l = 0.0;
    bud = budget0;
    for (int kk = (k + 1 > lo ? k + 1 : lo); kk < hi && bud > 0.0; ++kk) {
      const double n2j = n2p[kk * MX_COLS + col];
      const double dzj = dzl[kk * MX_COLS + col];
      const double cost = n2j * dzj * (l + 0.5 * dzj);
      double step;
      if (cost <= bud) {
        step = dzj;
        bud = bud - cost;
      } else {
        if (n2j > 0.0) {
          const double s = sqrt(nmax(l * l + 2.0 * bud / n2j, 0.0)) - l;
          step = nmin(nmax(s, 0.0), dzj);
        } else {
          step = dzj;
        }
        bud = 0.0;
      }
      l = l + step;
    }
    const double zb = nmax(h - zi, 0.0);
    const double l_dn = nmin(l, zb + p.z_0) * wet;
    s_l[o] = nmax(p.l_min, sqrt(l_up * l_dn));
    s_le[o] = nmax(p.l_min, nmin(l_up, l_dn));
  }
}

size_t closure_lengths_lds(int nz) { return (size_t)2 * (nz + 1) * MX_COLS * sizeof(double); }

void launch_closure_lengths(const Dims& d, const StepParams& p, const Geo& geo,
                            const double* e_in, const double* u, const double* v,
                            const double* b, double* s_n2, double* s_sh, double* s_l,
                            double* s_le, hipStream_t s) {
  const unsigned nb = (unsigned)((d.n2 + MX_COLS - 1) / MX_COLS);
  k_closure_lengths<<<nb, MX_THREADS, closure_lengths_lds(d.nz), s>>>(d, p, geo, e_in, u, v, b,
                                                                      s_n2, s_sh, s_l, s_le);
}

int closure_lengths_prepare(int nz) {
  const size_t lds = closure_lengths_lds(nz);
  if (lds > 160 * 1024) return -1;
  return hipFuncSetAttribute((const void*)k_closure_lengths,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess
             ? 0
             : -2;
}

// N^2 and shear^2 alone, one lane per interface cell (the recursive form
// needs N^2 before its length recursion).
__global__ void k_closure_shear(Dims d, StepParams p, Geo geo, const double* __restrict__ u,
                                const double* __restrict__ v, const double* __restrict__ b,
                                double* __restrict__ s_n2, double* __restrict__ s_sh) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.ni) return;
  const int k = (int)(t / d.n2);
  const long long c = t % d.n2;
  double n2k, sh;
  shear_n2(d, p, geo, u, v, b, c, k, n2k, sh);
  s_n2[t] = n2k;
  s_sh[t] = sh;
}

// Recursive (NEMO nn_mxl=2) mixing length, closure.py:106-129; s_l is the
// work array of the two sweeps and ends as l_k, s_le as l_eps.
__global__ void k_mixing_recursive(Dims d, StepParams p, Geo geo, const double* __restrict__ e_in,
                                   const double* __restrict__ s_n2, double* __restrict__ s_l,
                                   double* __restrict__ s_le) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const int nz = d.nz;
  const long long n2 = d.n2;
  const ColumnGeo cg(geo, p, d, c);
  double h = 0.0;
  for (int k = 0; k < nz; ++k) h = h + cg.dz(k);
  double zi = 0.0;
  for (int k = 0; k <= nz; ++k) {
    if (k > 0) zi = zi + cg.dz(k - 1);
    const double n2c = nmax(s_n2[k * n2 + c], p.n2_min);
    const double ek = nmax(e_in[k * n2 + c], p.e_min);
    double l = sqrt(2.0 * ek / n2c);
    const double zb = nmax(h - zi, 0.0);
    l = nmin(l, nmin(zi + p.z_0, zb + p.z_0));
    if (k > 0) l = nmin(l, s_l[(k - 1) * n2 + c] + cg.dzi(k));
    s_l[k * n2 + c] = l;
  }
  for (int k = nz - 1; k >= 0; --k) {
    const double l = nmin(s_l[k * n2 + c], s_l[(k + 1) * n2 + c] + cg.dzi(k + 1));
    s_l[k * n2 + c] = l;
  }
  for (int k = 0; k <= nz; ++k) {
    const double wet = (k >= 1 && k < nz)
                           ? (cg.wet(k - 1) ? 1.0 : 0.0) * (cg.wet(k) ? 1.0 : 0.0) : 0.0;
    const double l = s_l[k * n2 + c] * wet;  // l_up = l_dn = l
    s_l[k * n2 + c] = nmax(p.l_min, sqrt(l * l));
    s_le[k * n2 + c] = nmax(p.l_min, nmin(l, l));
  }
}

// The interface tridiagonal for e and the eddy coefficients, one lane per
// column, from s_n2, s_sh, s_l = l_k and s_le = l_eps. ZC: thicknesses and wet
// flags from the column form. STAGE: c* and d* stay in LDS between the sweeps
// instead of in s_c and e_out. NT: threads of a workgroup.
// Bound: latency of the march on small grids, then memory (10 fields, 14
// unstaged) and the roots and divisions at the few waves that LDS leaves. Per
// launch, against no loads ahead and c*, d* in memory: 128 x 4 x 20 33 -> 18
// us, 128 x 128 x 30 51 -> 26, 640 x 512 x 48 326 -> 308, 1000 x 1000 x 30
// 675 -> 513; 512 x 512 x 40 212 -> 219, whose levels are exactly 2 MiB apart
// (448 x 448 x 40 175 -> 172, 576 x 576 x 40 302 -> 266); where launch_closure
// leaves it unstaged 384 x 384 x 60 210 -> 190, 512 x 512 x 60 318 -> 316, 800 x
// 800 x 60 846 -> 826.
template <bool ZC, bool STAGE, int NT>
__global__ __launch_bounds__(NT) void k_closure(
    Dims d, StepParams p, Geo geo, const double* __restrict__ e_in, double* __restrict__ Km,
    double* __restrict__ Kh, double* __restrict__ e_out, const double* __restrict__ s_n2,
    const double* __restrict__ s_sh, const double* __restrict__ s_l,
    const double* __restrict__ s_le, double* __restrict__ s_c) {
  extern __shared__ double clo_lds[];  // STAGE: [2][nz + 1][COLS], a thread's own column
  static_assert(!STAGE || NT == COLS, "a staged column per lane of one wave");
  const long long c = (long long)(NT == COLS ? xcd_linear() : blockIdx.x) * NT + threadIdx.x;
  if (c >= d.n2) return;
  const int nz = d.nz;
  const long long n2 = d.n2;
  const unsigned bc = 8u * (unsigned)c;
  const double kb = geo.kappa_b[c];
  const double dt = p.dt;
  double* lc = clo_lds + threadIdx.x;
  double* ld = lc + (size_t)(nz + 1) * COLS;
  int nwc = 0;
  InvCol ic{};
  if constexpr (ZC) {
    nwc = geo.nw[c];
    ic = inv_col(nwc, p.dzr, nwc > 0 ? geo.hb[c] : 0.0);
  }
  auto wet_at = [&](int k, uint8_t m) { return k >= 0 && k < nz && (ZC ? k < nwc : m != 0); };
  struct Level {
    double e, n2, sh, le, kh, km, dzi, dz;
    uint8_t m;
  };
  double c_prev = 0.0, d_prev = 0.0, rhs0 = 0.0;
  // K_m at interfaces k - 1 and k, the inverse thickness and the wet flag of
  // the cell above interface k, carried down the column
  double km_up = 0.0, km_0 = Km[c], inv_up = 0.0;
  bool wet_above = false;
  march_down<STAGE ? 4 : 3>(  // 3: four unstaged waves per SIMD instead of three
      nz + 1,
      [&](int k) {
        const long long o = k * n2;
        Level L;
        L.e = at_byte(e_in + o, bc);
        L.n2 = at_byte(s_n2 + o, bc);
        L.sh = at_byte(s_sh + o, bc);
        L.le = at_byte(s_le + o, bc);
        L.kh = at_byte(Kh + o, bc);
        L.km = at_byte(Km + (k < nz ? o + n2 : o), bc);
        if constexpr (!ZC) {
          const long long oc = k < nz ? o : o - n2;
          L.dzi = at_byte(geo.dzi + o, bc);
          L.dz = at_byte(geo.dz3 + oc, bc);
          L.m = at_byte(geo.m3 + oc, (unsigned)c);
        }
        return L;
      },
      [&](int k, const Level& L) {
        const bool wet_below = wet_at(k, L.m);
        const double wet = wet_above && wet_below ? 1.0 : 0.0;
        const double kmo = km_0, km_dn = L.km;
        const double prod = (kmo - p.nu_b) * L.sh - (L.kh - kb) * L.n2;
        const double diss = p.c_eps * sqrt(nmax(L.e, p.e_min)) / L.le;
        const double inv_dn = ZC ? ic.inv(k) : safe_inv(L.dz);
        double a_up = 0.0, a_dn = 0.0;
        if (k >= 1 && k < nz) {
          const double idzi = ZC ? ic.idzi(k) : safe_inv(L.dzi);
          const double klay_up = 0.5 * (km_up + kmo);
          const double klay_dn = 0.5 * (kmo + km_dn);
          a_up = dt * klay_up * inv_up * idzi;
          a_dn = dt * klay_dn * inv_dn * idzi;
        }
        double sub = -a_up, sup = -a_dn;
        double diag = 1.0 + a_up + a_dn + dt * diss;
        double rhs = L.e + dt * prod;
        if (wet <= 0.0) {
          diag = 1.0;
          sub = 0.0;
          sup = 0.0;
          rhs = p.e_min;
        }
        if (k == 0) {
          rhs = wet_below ? p.e_bb * geo.ustar2[c] : p.e_min;
          rhs0 = rhs;
        }
        const Divisor<double> by_den(k == 0 ? diag : diag - sub * c_prev);
        const double cst = by_den(sup);
        const double dst = k == 0 ? by_den(rhs) : by_den(rhs - sub * d_prev);
        if constexpr (STAGE) {
          lc[k * COLS] = cst;
          ld[k * COLS] = dst;
        } else {
          put_byte(s_c + k * n2, bc, cst);
          put_byte(e_out + k * n2, bc, dst);
        }
        c_prev = cst;
        d_prev = dst;
        km_up = km_0;
        km_0 = km_dn;
        inv_up = inv_dn;
        wet_above = wet_below;
      });

  // back-substitution, floors, eddy coefficients
  struct Back {
    double cst, dst, l;
    uint8_t m;
  };
  const Divisor<double> by_pr = uniform_divisor<double>(p.pr_t);
  double x_next = 0.0;
  bool wet_below = false;  // cell k (below interface k)
  march_up<4>(
      nz + 1,
      [&](int k) {
        const long long o = k * n2;
        Back B;
        if constexpr (STAGE) {
          B.cst = lc[k * COLS];
          B.dst = ld[k * COLS];
        } else {
          B.cst = at_byte(s_c + o, bc);
          B.dst = at_byte(e_out + o, bc);
        }
        B.l = at_byte(s_l + o, bc);
        if constexpr (!ZC) B.m = at_byte(geo.m3 + (k > 0 ? o - n2 : o), (unsigned)c);
        return B;
      },
      [&](int k, const Back& B) {
        const bool wet_above = wet_at(k - 1, B.m);
        const double x = (k == nz) ? B.dst : B.dst - B.cst * x_next;
        x_next = x;
        const double wet = wet_above && wet_below ? 1.0 : 0.0;
        double en = nmax(x, p.e_min);
        en = wet > 0.0 ? en : p.e_min;
        if (k == 0) en = rhs0;
        const double km = p.c_k * B.l * sqrt(en) * wet + p.nu_b;
        const double kh = by_pr(km - p.nu_b) + kb;
        put_byte(e_out + k * n2, bc, en);
        put_byte(Km + k * n2, bc, km);
        put_byte(Kh + k * n2, bc, kh);
        wet_below = wet_above;
      });
}

void launch_closure(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                    const double* e_in, double* Km, double* Kh, double* e_out,
                    const double* s_n2, const double* s_sh, const double* s_l,
                    const double* s_le, double* s_c) {
  const size_t lds = (size_t)2 * (d.nz + 1) * COLS * sizeof(double);
  const long long waves = column_blocks(d), per_cu = CU_LDS / (long long)lds;
  // Staged where LDS holds three workgroups per compute unit, or the whole grid
  // at once; with two of them (53 levels and more) a large grid gains less from
  // the four passes saved than it loses in waves. Staged and not: 384 x 384 x
  // 40 126 and 124 us, 640 x 512 x 48 308 and 340, 128 x 128 x 60 45 and 50,
  // 320 x 320 x 60 174 and 132, 512 x 512 x 60 370 and 316, 800 x 800 x 60 880
  // and 826.
  const bool stage = lds <= COL_LDS_MAX && (per_cu >= 3 || waves <= CUS * per_cu);
  // Unstaged, workgroups of four waves from four per compute unit on; fewer
  // spread unevenly. One wave and four: 384 x 384 x 60 190 and 210 us, 448 x
  // 448 x 40 177 and 185, 512 x 512 x 60 340 and 316, 704 x 704 x 40 434 and 421.
  const bool wide = waves >= 16 * CUS;
  with_column_form(p.zcol != 0, stage, [&](auto zc, auto sg) {
    constexpr bool ZC = decltype(zc)::value, SG = decltype(sg)::value;
    constexpr int WIDE = 4 * COLS;
    if constexpr (!SG) {
      if (wide) {
        k_closure<ZC, SG, WIDE><<<(unsigned)((d.n2 + WIDE - 1) / WIDE), WIDE, 0, s>>>(
            d, p, geo, e_in, Km, Kh, e_out, s_n2, s_sh, s_l, s_le, s_c);
        return;
      }
    }
    k_closure<ZC, SG, COLS><<<column_blocks(d), COLS, SG ? lds : 0, s>>>(
        d, p, geo, e_in, Km, Kh, e_out, s_n2, s_sh, s_l, s_le, s_c);
  });
}

// ------------------------------------------------ vertical coefficients
// tri_m (viscosity Km, bottom drag), factored, then q = A_m^-1 1
// (libs/core/model3d_v05.py:141-153); tri_b is factored by the tracer
// kernels from the K_h they read anyway. The factorization and the forward
// sweep of q are one pass over the column; STAGE: c* and d* are kept in LDS
// for the back-substitution. Memory-bound on large grids (5 fields instead of
// 8), latency-bound on small ones: 128 x 128 x 30 29 -> 16 us, 512 x 512 x 40
// 126 -> 93, 1000 x 1000 x 30 350 -> 243.
template <bool ZC, bool STAGE>
__global__ __launch_bounds__(COLS) void k_coefficients(
    Dims d, StepParams p, Geo geo, const double* __restrict__ Km, double* __restrict__ sub_m,
    double* __restrict__ den_m, double* __restrict__ cst_m, double* __restrict__ q) {
  extern __shared__ double coe_lds[];  // STAGE: [2][nz][COLS], a thread's own column
  const long long c = (long long)xcd_linear() * COLS + threadIdx.x;
  if (c >= d.n2) return;
  const int nz = d.nz;
  const long long n2 = d.n2;
  const unsigned bc = 8u * (unsigned)c;
  double* lc = coe_lds + threadIdx.x;
  double* ld = lc + (size_t)nz * COLS;
  InvCol ic{};
  int nwc = 0;
  double idzi_t;
  bool wet;
  if constexpr (ZC) {
    nwc = geo.nw[c];
    ic = inv_col(nwc, p.dzr, nwc > 0 ? geo.hb[c] : 0.0);
    idzi_t = ic.inv(0);
    wet = nwc > 0;
  } else {
    idzi_t = safe_inv(geo.dzi[c]);
    wet = geo.m3[c] != 0;
  }
  struct Level {
    double km, dz, dzi;
    uint8_t m;
  };
  double cm_prev = 0.0, d_prev = 0.0, km_t = Km[c];
  march_down<8>(
      nz,
      [&](int k) {
        const long long o = k * n2;
        Level L;
        L.km = at_byte(Km + o + n2, bc);
        if constexpr (!ZC) {
          L.dz = at_byte(geo.dz3 + o, bc);
          L.dzi = at_byte(geo.dzi + o + n2, bc);
          L.m = at_byte(geo.m3 + (k + 1 < nz ? o + n2 : o), (unsigned)c);
        }
        return L;
      },
      [&](int k, const Level& L) {
        const long long o = k * n2;
        double inv_dz, idzi_b;
        bool below = k + 1 < nz;
        if constexpr (ZC) {
          inv_dz = ic.inv(k);
          idzi_b = k + 1 == nz ? inv_dz : ic.idzi(k + 1);
          below = below && k + 1 < nwc;
        } else {
          inv_dz = safe_inv(L.dz);
          idzi_b = safe_inv(L.dzi);
          below = below && L.m != 0;
        }
        double sub, sup, den;
        matrix_row(p, k, inv_dz, km_t, L.km, idzi_t, idzi_b, wet, below, p.thv_dt_drag, cm_prev,
                   sub, sup, den);
        const Divisor<double> by_den(den);
        const double cm = by_den(sup);
        const double dst = k == 0 ? by_den(1.0) : by_den(1.0 - sub * d_prev);
        put_byte(sub_m + o, bc, sub);
        put_byte(den_m + o, bc, den);
        put_byte(cst_m + o, bc, cm);
        if constexpr (STAGE) {
          lc[k * COLS] = cm;
          ld[k * COLS] = dst;
        } else {
          put_byte(q + o, bc, dst);
        }
        d_prev = dst;
        cm_prev = cm;
        idzi_t = idzi_b;
        km_t = L.km;
        wet = below;
      });
  struct Back {
    double cm, dst;
  };
  double x = 0.0;
  march_up<8>(
      nz,
      [&](int k) {
        const long long o = k * n2;
        Back B;
        if constexpr (STAGE) {
          B.cm = lc[k * COLS];
          B.dst = ld[k * COLS];
        } else {
          B.cm = at_byte(cst_m + o, bc);
          B.dst = at_byte(q + o, bc);
        }
        return B;
      },
      [&](int k, const Back& B) {
        x = k == nz - 1 ? B.dst : B.dst - B.cm * x;
        put_byte(q + k * n2, bc, x);
      });
}

void launch_coefficients(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                         const double* Km, double* sub_m, double* den_m, double* cst_m,
                         double* q) {
  const size_t lds = (size_t)2 * d.nz * COLS * sizeof(double);
  with_column_form(p.zcol != 0, lds <= COL_LDS_MAX, [&](auto zc, auto sg) {
    constexpr bool SG = decltype(sg)::value;
    k_coefficients<decltype(zc)::value, SG><<<column_blocks(d), COLS, SG ? lds : 0, s>>>(
        d, p, geo, Km, sub_m, den_m, cst_m, q);
  });
}

// Helmholtz face coefficients Ku = sum_k dz3u min(q, q_east) mask_u and Kv
// (libs/core/model3d_v05.py:154-157), summed in k order like NumPy's
// axis-0 reduction. 128 x 128 x 30 24 -> 10 us, 512 x 512 x 40 39 -> 35.
template <bool ZC>
__global__ __launch_bounds__(COLS) void k_kukv(Dims d, StepParams p, Geo geo,
                                               const double* __restrict__ q,
                                               double* __restrict__ Ku,
                                               double* __restrict__ Kv) {
  const long long c = (long long)xcd_linear() * COLS + threadIdx.x;
  if (c >= d.n2) return;
  const int j = (int)((unsigned)c / (unsigned)d.nx), i = (int)((unsigned)c - (unsigned)j * d.nx);
  const long long ce = at2(d, j, wrap(i, 1, d.nx));
  const long long cn = at2(d, wrap(j, 1, d.ny), i);
  const long long n2 = d.n2;
  const unsigned bc = 8u * (unsigned)c, be = 8u * (unsigned)ce, bn = 8u * (unsigned)cn;
  FaceCol fu{}, fv{};
  if constexpr (ZC) {
    fu = face_col(geo, p, c, ce, 0);
    fv = face_col(geo, p, c, cn, 1);
  }
  struct Level {
    double c, e, n, du, dv;
  };
  double su = 0.0, sv = 0.0;
  march_down<3>(
      d.nz,
      [&](int k) {
        const long long o = k * n2;
        Level L;
        L.c = at_byte(q + o, bc);
        L.e = at_byte(q + o, be);
        L.n = at_byte(q + o, bn);
        if constexpr (!ZC) {
          L.du = at_byte(geo.dz3u + o, bc);
          L.dv = at_byte(geo.dz3v + o, bc);
        }
        return L;
      },
      [&](int k, const Level& L) {
        const double tu = (ZC ? fu.dz(k) : L.du) * nmin(L.c, L.e);
        const double tv = (ZC ? fv.dz(k) : L.dv) * nmin(L.c, L.n);
        su = (k == 0) ? tu : su + tu;
        sv = (k == 0) ? tv : sv + tv;
      });
  Ku[c] = su * mk(geo.mu2[c]);
  Kv[c] = sv * mk(geo.mv2[c]);
}

void launch_kukv(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                 const double* q, double* Ku, double* Kv) {
  if (p.zcol) k_kukv<true><<<column_blocks(d), COLS, 0, s>>>(d, p, geo, q, Ku, Kv);
  else k_kukv<false><<<column_blocks(d), COLS, 0, s>>>(d, p, geo, q, Ku, Kv);
}

// --------------------------------------------------- pressure potential
// Phi_k = 1/2 dz_k b_k + sum_{k'<k} dz b (libs/core/vertical_var.py:132-136);
// optionally the thickness-weighted depth mean removed (:139-145).
__global__ void k_phi(Dims d, StepParams p, Geo geo, const double* __restrict__ b,
                      double* __restrict__ phi) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const long long n2 = d.n2;
  const ColumnGeo cg(geo, p, d, c);
  double above = 0.0;
  for (int k = 0; k < d.nz; ++k) {
    const double dz = cg.dz(k);
    const double bk = b[k * n2 + c];
    phi[k * n2 + c] = 0.5 * dz * bk + above;
    const double t = dz * bk;
    above = (k == 0) ? t : above + t;
  }
  if (p.pgf_remove) {
    double tot = 0.0, wsum = 0.0;
    for (int k = 0; k < d.nz; ++k) {
      const double dz = cg.dz(k);
      const double t = dz * phi[k * n2 + c];
      tot = (k == 0) ? dz : tot + dz;
      wsum = (k == 0) ? t : wsum + t;
    }
    const double mean = wsum * safe_inv(tot);
    for (int k = 0; k < d.nz; ++k) phi[k * n2 + c] = phi[k * n2 + c] - mean;
  }
}

// ------------------------------------- transports and vertical velocity
// Of one column: the transports U0 = sum dz3u u, V0 = sum dz3v v (TR) and
// w_k = -sum_{k'>=k} div(dz3u u, dz3v v), w_nz = 0, summed from the bottom
// (libs/core/vertical_var.py:109-121 with model3d_v05.py:232-235) (WW), in one
// march down that reads u and v once: the divergences wait in LDS (STAGE: a
// thread's own [nz] values, COLS apart) or in w for the sum upwards.
template <bool ZC, bool STAGE, bool TR, bool WW>
__device__ __forceinline__ void transports_column(const Dims& d, const StepParams& p,
                                                  const Geo& geo, const double* __restrict__ u,
                                                  const double* __restrict__ v,
                                                  double* __restrict__ U0,
                                                  double* __restrict__ V0,
                                                  double* __restrict__ w, double* lds,
                                                  long long c) {
  const int j = (int)((unsigned)c / (unsigned)d.nx), i = (int)((unsigned)c - (unsigned)j * d.nx);
  const long long ce = at2(d, j, wrap(i, 1, d.nx)), cn = at2(d, wrap(j, 1, d.ny), i);
  const long long cw = at2(d, j, wrap(i, -1, d.nx)), cs = at2(d, wrap(j, -1, d.ny), i);
  const unsigned bc = 8u * (unsigned)c, bw = 8u * (unsigned)cw, bs = 8u * (unsigned)cs;
  const long long n2 = d.n2;
  const int nz = d.nz;
  FaceCol fe{}, fw{}, fn{}, fs{};
  int nwc = 0;
  if constexpr (ZC) {
    fe = face_col(geo, p, c, ce, 0);
    fn = face_col(geo, p, c, cn, 1);
    if constexpr (WW) {
      nwc = geo.nw[c];
      fw = face_col(geo, p, cw, c, 0);
      fs = face_col(geo, p, cs, c, 1);
    }
  }
  const Divisor<double> by_dx = uniform_divisor<double>(p.dx), by_dy = uniform_divisor<double>(p.dy);
  struct Level {
    double u, uw, v, vs, de, dw, dn, ds;
    uint8_t m;
  };
  double su = 0.0, sv = 0.0;
  march_down<ZC ? 4 : 3>(
      nz,
      [&](int k) {
        const long long o = k * n2;
        Level L;
        L.u = at_byte(u + o, bc);
        L.v = at_byte(v + o, bc);
        if constexpr (WW) {
          L.uw = at_byte(u + o, bw);
          L.vs = at_byte(v + o, bs);
        }
        if constexpr (!ZC) {
          L.de = at_byte(geo.dz3u + o, bc);
          L.dn = at_byte(geo.dz3v + o, bc);
          if constexpr (WW) {
            L.dw = at_byte(geo.dz3u + o, bw);
            L.ds = at_byte(geo.dz3v + o, bs);
            L.m = at_byte(geo.m3 + o, (unsigned)c);
          }
        }
        return L;
      },
      [&](int k, const Level& L) {
        const double U = (ZC ? fe.dz(k) : L.de) * L.u;
        const double V = (ZC ? fn.dz(k) : L.dn) * L.v;
        if constexpr (TR) {
          su = (k == 0) ? U : su + U;
          sv = (k == 0) ? V : sv + V;
        }
        if constexpr (WW) {
          const double Uw = (ZC ? fw.dz(k) : L.dw) * L.uw;
          const double Vs = (ZC ? fs.dz(k) : L.ds) * L.vs;
          const double wet = (ZC ? k < nwc : L.m != 0) ? 1.0 : 0.0;
          const double dv = wet * (by_dx(U - Uw) + by_dy(V - Vs));
          if constexpr (STAGE) lds[k * COLS] = dv;
          else put_byte(w + k * n2, bc, dv);
        }
      });
  if constexpr (TR) {
    U0[c] = su;
    V0[c] = sv;
  }
  if constexpr (WW) {
    double s = 0.0;
    march_up<8>(
        nz,
        [&](int k) {
          if constexpr (STAGE) return lds[k * COLS];
          else return at_byte(w + k * n2, bc);
        },
        [&](int k, double dv) {
          s = (k == nz - 1) ? dv : s + dv;
          put_byte(w + k * n2, bc, -s);
        });
    w[(long long)nz * n2 + c] = 0.0;
  }
}

template <bool ZC, bool STAGE>
__global__ __launch_bounds__(COLS) void k_w_diag(Dims d, StepParams p, Geo geo,
                                                 const double* __restrict__ u,
                                                 const double* __restrict__ v,
                                                 double* __restrict__ w) {
  extern __shared__ double wd_lds[];
  const long long c = (long long)xcd_linear() * COLS + threadIdx.x;
  if (c < d.n2)
    transports_column<ZC, STAGE, false, true>(d, p, geo, u, v, nullptr, nullptr, w,
                                              wd_lds + threadIdx.x, c);
}

void launch_w_diag(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                   const double* u, const double* v, double* w) {
  const size_t lds = (size_t)d.nz * COLS * sizeof(double);
  with_column_form(p.zcol != 0, lds <= COL_LDS_MAX, [&](auto zc, auto sg) {
    constexpr bool SG = decltype(sg)::value;
    k_w_diag<decltype(zc)::value, SG><<<column_blocks(d), COLS, SG ? lds : 0, s>>>(d, p, geo, u,
                                                                                  v, w);
  });
}

// ------------------------------------------------- the step's prologue
// phi as k_phi forms it and, independently, the transports (U0 set) and w (w
// set): two waves over the same columns (`part`).
// Against one lane marching down for phi and the transports and up again for
// w: 128 x 128 x 30 40 -> 12.5 us, 512 x 512 x 40 117 -> 102, 1000 x 1000 x 30
// 290 -> 250. (The waves in workgroups of their own would each hold the LDS of
// the second: 322 us.)
template <bool ZC, bool STAGE, bool TR, bool WW>
__global__ __launch_bounds__(2 * COLS) void k_prologue(
    Dims d, StepParams p, Geo geo, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ b, double* __restrict__ phi, double* __restrict__ U0,
    double* __restrict__ V0, double* __restrict__ w) {
  extern __shared__ double pro_lds[];
  const int lane = threadIdx.x % COLS;
  const long long c = (long long)xcd_linear() * COLS + lane;
  if (c >= d.n2) return;
  if constexpr (TR || WW) {
    if (__builtin_amdgcn_readfirstlane(threadIdx.x / COLS) == 1) {
      transports_column<ZC, STAGE, TR, WW>(d, p, geo, u, v, U0, V0, w, pro_lds + lane, c);
      return;
    }
  }
  const long long n2 = d.n2;
  const int nz = d.nz;
  const unsigned bc = 8u * (unsigned)c;
  struct Level {
    double x, dz;
  };
  const ColumnGeo cg(geo, p, d, c);
  auto level = [&](const double* f, int k) {
    return Level{at_byte(f + k * n2, bc), ZC ? 0.0 : at_byte(geo.dz3 + k * n2, bc)};
  };
  double above = 0.0;
  march_down<8>(
      nz, [&](int k) { return level(b, k); },
      [&](int k, const Level& L) {
        const double dz = ZC ? cg.dz(k) : L.dz;
        put_byte(phi + k * n2, bc, 0.5 * dz * L.x + above);
        const double t = dz * L.x;
        above = (k == 0) ? t : above + t;
      });
  if (p.pgf_remove) {
    double tot = 0.0, wsum = 0.0;
    march_down<8>(
        nz, [&](int k) { return level(phi, k); },
        [&](int k, const Level& L) {
          const double dz = ZC ? cg.dz(k) : L.dz;
          const double t = dz * L.x;
          tot = (k == 0) ? dz : tot + dz;
          wsum = (k == 0) ? t : wsum + t;
        });
    const double mean = wsum * safe_inv(tot);
    march_down<8>(
        nz, [&](int k) { return at_byte(phi + k * n2, bc); },
        [&](int k, double x) { put_byte(phi + k * n2, bc, x - mean); });
  }
}

void launch_prologue(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                     const double* u, const double* v, const double* b, double* phi, double* U0,
                     double* V0, double* w) {
  const size_t lds = w ? (size_t)d.nz * COLS * sizeof(double) : 0;
  with_column_form(p.zcol != 0, lds <= COL_LDS_MAX, [&](auto zc, auto sg) {
    constexpr bool ZC = decltype(zc)::value, SG = decltype(sg)::value;
    auto go = [&](auto tr, auto ww) {
      constexpr bool TR = decltype(tr)::value, WW = decltype(ww)::value;
      k_prologue<ZC, SG, TR, WW>
          <<<column_blocks(d), TR || WW ? 2 * COLS : COLS, SG ? lds : 0, s>>>(d, p, geo, u, v, b,
                                                                              phi, U0, V0, w);
    };
    using T = std::true_type;
    using F = std::false_type;
    if (U0) {
      if (w) go(T{}, T{});
      else go(T{}, F{});
    } else {
      if (w) go(F{}, T{});
      else go(F{}, F{});
    }
  });
}

// ------------------------------------------------ explicit momentum terms
struct Nb {  // periodic neighbour offsets of a column (a plane has < 2^31 columns)
  int c, e, w, ee, ww, n, s, nn, ss, ne, nw, se, sw;
};
__device__ __forceinline__ Nb neighbours(const Dims& d, int j, int i) {
  Nb q;
  const int ie = wrap(i, 1, d.nx), iw = wrap(i, -1, d.nx);
  const int iee = wrap(i, 2, d.nx), iww = wrap(i, -2, d.nx);
  const int jn = wrap(j, 1, d.ny), js = wrap(j, -1, d.ny);
  const int jnn = wrap(j, 2, d.ny), jss = wrap(j, -2, d.ny);
  q.c = (int)at2(d, j, i);
  q.e = (int)at2(d, j, ie);
  q.w = (int)at2(d, j, iw);
  q.ee = (int)at2(d, j, iee);
  q.ww = (int)at2(d, j, iww);
  q.n = (int)at2(d, jn, i);
  q.s = (int)at2(d, js, i);
  q.nn = (int)at2(d, jnn, i);
  q.ss = (int)at2(d, jss, i);
  q.ne = (int)at2(d, jn, ie);
  q.nw = (int)at2(d, jn, iw);
  q.se = (int)at2(d, js, ie);
  q.sw = (int)at2(d, js, iw);
  return q;
}

// Coriolis partner of u: v averaged over the wet v faces around the u point
// (libs/core/operators_masked.py:45-52).
__device__ __forceinline__ double avg_v_to_u(const double* v, const uint8_t* mv, const uint8_t* mu,
                                             long long o, const Nb& q) {
  const double w0 = mk(mv[o + q.c]), w1 = mk(mv[o + q.s]), w2 = mk(mv[o + q.e]),
               w3 = mk(mv[o + q.se]);
  const double num = 0.0 + w0 * v[o + q.c] + w1 * v[o + q.s] + w2 * v[o + q.e] + w3 * v[o + q.se];
  const double den = 0.0 + w0 + w1 + w2 + w3;
  const double out = den > 0.0 ? num / den : 0.0;
  return out * mk(mu[o + q.c]);
}
// (libs/core/operators_masked.py:55-61)
__device__ __forceinline__ double avg_u_to_v(const double* u, const uint8_t* mu, const uint8_t* mv,
                                             long long o, const Nb& q) {
  const double w0 = mk(mu[o + q.c]), w1 = mk(mu[o + q.w]), w2 = mk(mu[o + q.n]),
               w3 = mk(mu[o + q.nw]);
  const double num = 0.0 + w0 * u[o + q.c] + w1 * u[o + q.w] + w2 * u[o + q.n] + w3 * u[o + q.nw];
  const double den = 0.0 + w0 + w1 + w2 + w3;
  const double out = den > 0.0 ? num / den : 0.0;
  return out * mk(mv[o + q.c]);
}

// Mean over the open ones of four faces (libs/core/operators_masked.py:46-61):
// the weighted sum over the number of open faces, in the reference's order.
// The quotient by 1, 2, 3 or 4 is formed like Divisor's, in the same range, whose
// reciprocals are the constants here.
struct Avg4 {
  double w[4], den, y, own;
  bool any;
  __device__ __forceinline__ Avg4(const bool* f, bool own_) {
    int n = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      w[q] = f[q] ? 1.0 : 0.0;
      n += (int)f[q];
    }
    den = (double)n;
    y = n == 4 ? 0.25 : n == 3 ? 1.0 / 3.0 : n == 2 ? 0.5 : 1.0;
    own = own_ ? 1.0 : 0.0;
    any = n > 0;
  }
  __device__ __forceinline__ double operator()(double a0, double a1, double a2, double a3) const {
    const double num = 0.0 + w[0] * a0 + w[1] * a1 + w[2] * a2 + w[3] * a3;
    const double m = __builtin_amdgcn_div_fixup(scaled_quotient(num, den, y), den, num);
    return (any ? m : 0.0) * own;
  }
};
__device__ __forceinline__ double avg4(const double* a, const bool* f, bool own) {
  return Avg4(f, own)(a[0], a[1], a[2], a[3]);
}

// Explicit vertical diffusion Dz[f] at layer k with surface flux sflux, no
// flux through a column's bottom interface and linear drag on the bottom
// cell (libs/core/vertical_var.py:80-106). dzf is the thickness of f's
// points (dz3u for u, dz3v for v, dz3 for tracers); cell mask3 decides the
// bottom.
__device__ __forceinline__ double explicit_diffusion(const Dims& d, const uint8_t* m3,
                                                     const double* f, const double* nu,
                                                     const double* dzf, double sflux,
                                                     double drag, long long c, int k) {
  const int nz = d.nz;
  const long long n2 = d.n2;
  auto dzi_f = [&](int kk) -> double {  // interface_thickness(dzf)[kk]
    if (kk == 0) return dzf[c];
    if (kk == nz) return dzf[(nz - 1) * n2 + c];
    return 0.5 * (dzf[(kk - 1) * n2 + c] + dzf[kk * n2 + c]);
  };
  auto is_bottom = [&](int kk) -> bool {
    return m3[kk * n2 + c] != 0 && !((kk + 1 < nz) && m3[(kk + 1) * n2 + c] != 0);
  };
  // flux through the top (interface k) and bottom (interface k+1) of cell k
  double ft;
  if (k == 0) {
    ft = sflux;
  } else {
    ft = nu[k * n2 + c] * (f[(k - 1) * n2 + c] - f[k * n2 + c]) * safe_inv(dzi_f(k));
    if (is_bottom(k - 1)) ft = 0.0;
  }
  double fb = 0.0;
  if (k + 1 < nz) {
    fb = nu[(k + 1) * n2 + c] * (f[k * n2 + c] - f[(k + 1) * n2 + c]) * safe_inv(dzi_f(k + 1));
    if (is_bottom(k)) fb = 0.0;
  }
  const double inv = safe_inv(dzf[k * n2 + c]);
  const double out = (ft - fb) * inv;
  const double dr = drag * f[k * n2 + c] * (is_bottom(k) ? 1.0 : 0.0);
  return (out - dr * inv) * (m3[k * n2 + c] != 0 ? 1.0 : 0.0);
}

// u-momentum advection at (k, j, i) (libs/core/advection_v06.py:77-99 for
// up3/up3_tvd, libs/core/advection.py:62-79 for centred2).
__device__ double advect_u(const Dims& d, const StepParams& p, const uint8_t* m3u,
                           const double* u, const double* v, const double* w, long long o,
                           int k, const Nb& q) {
  const long long n2 = d.n2;
  const int nz = d.nz;
  const bool lim = p.advection == ADV_UP3_TVD;
  const double* U = u + o;
  const double* V = v + o;
  double ax, ay, az;
  if (p.advection == ADV_CENTRED2) {
    const double ub = 0.5 * (U[q.w] + U[q.c]);
    const double ube = 0.5 * (U[q.c] + U[q.e]);
    ax = (ube * ube - ub * ub) / p.dx;
    const double vb = 0.5 * (V[q.c] + V[q.e]);
    const double vbs = 0.5 * (V[q.s] + V[q.se]);
    const double fy = vb * (0.5 * (U[q.c] + U[q.n]));
    const double fys = vbs * (0.5 * (U[q.s] + U[q.c]));
    ay = (fy - fys) / p.dy;
  } else {
    const uint8_t* M = m3u + o;
    // x flux at centres i (faces i-1|i) and i+1 (faces i|i+1)
    const double ub = 0.5 * (U[q.w] + U[q.c]);
    const double ube = 0.5 * (U[q.c] + U[q.e]);
    const double uc = kappa_face(U[q.ww], U[q.w], U[q.c], U[q.e], ub, M[q.ww] != 0,
                                 M[q.e] != 0, lim);
    const double uce = kappa_face(U[q.w], U[q.c], U[q.e], U[q.ee], ube, M[q.w] != 0,
                                  M[q.ee] != 0, lim);
    ax = (ube * uce - ub * uc) / p.dx;
    // y flux at corners j (between u[j], u[j+1]) and j-1
    const double vb = 0.5 * (V[q.c] + V[q.e]);
    const double vbs = 0.5 * (V[q.s] + V[q.se]);
    const double uy = kappa_face(U[q.s], U[q.c], U[q.n], U[q.nn], vb, M[q.s] != 0,
                                 M[q.nn] != 0, lim);
    const double uys = kappa_face(U[q.ss], U[q.s], U[q.c], U[q.n], vbs, M[q.ss] != 0,
                                  M[q.n] != 0, lim);
    ay = (vb * uy - vbs * uys) / p.dy;
  }
  // vertical flux on interfaces k (top) and k+1 (bottom)
  auto fz = [&](int kk) -> double {
    if (kk <= 0 || kk >= nz) return 0.0;
    const long long a = (long long)kk * n2;
    const double wb = 0.5 * (w[a + q.c] + w[a + q.e]);
    const double above = u[a - n2 + q.c], below = u[a + q.c];
    if (p.advection == ADV_CENTRED2) return wb * 0.5 * (above + below);
    const double far_up = kk >= 2 ? u[a - 2 * n2 + q.c] : 0.0;
    const double far_dn = kk <= nz - 2 ? u[a + n2 + q.c] : 0.0;
    const bool hu = kk >= 2 && m3u[a - 2 * n2 + q.c] != 0;
    const bool hd = kk <= nz - 2 && m3u[a + n2 + q.c] != 0;
    return wb * kappa_face_z(far_up, above, below, far_dn, wb, hu, hd, lim);
  };
  az = (fz(k) - fz(k + 1)) / p.dz_nom;
  return ax + ay + az;
}

// v-momentum advection (libs/core/advection_v06.py:100-108, advection.py:81-95).
__device__ double advect_v(const Dims& d, const StepParams& p, const uint8_t* m3v,
                           const double* u, const double* v, const double* w, long long o,
                           int k, const Nb& q) {
  const long long n2 = d.n2;
  const int nz = d.nz;
  const bool lim = p.advection == ADV_UP3_TVD;
  const double* U = u + o;
  const double* V = v + o;
  double bx, by, bz;
  if (p.advection == ADV_CENTRED2) {
    const double vb = 0.5 * (V[q.s] + V[q.c]);
    const double vbn = 0.5 * (V[q.c] + V[q.n]);
    by = (vbn * vbn - vb * vb) / p.dy;
    const double ub = 0.5 * (U[q.c] + U[q.n]);
    const double ubw = 0.5 * (U[q.w] + U[q.nw]);
    const double fx = ub * (0.5 * (V[q.c] + V[q.e]));
    const double fxw = ubw * (0.5 * (V[q.w] + V[q.c]));
    bx = (fx - fxw) / p.dx;
  } else {
    const uint8_t* M = m3v + o;
    const double vb = 0.5 * (V[q.s] + V[q.c]);
    const double vbn = 0.5 * (V[q.c] + V[q.n]);
    const double vc = kappa_face(V[q.ss], V[q.s], V[q.c], V[q.n], vb, M[q.ss] != 0,
                                 M[q.n] != 0, lim);
    const double vcn = kappa_face(V[q.s], V[q.c], V[q.n], V[q.nn], vbn, M[q.s] != 0,
                                  M[q.nn] != 0, lim);
    by = (vbn * vcn - vb * vc) / p.dy;
    const double ub = 0.5 * (U[q.c] + U[q.n]);
    const double ubw = 0.5 * (U[q.w] + U[q.nw]);
    const double vx = kappa_face(V[q.w], V[q.c], V[q.e], V[q.ee], ub, M[q.w] != 0,
                                 M[q.ee] != 0, lim);
    const double vxw = kappa_face(V[q.ww], V[q.w], V[q.c], V[q.e], ubw, M[q.ww] != 0,
                                  M[q.e] != 0, lim);
    bx = (ub * vx - ubw * vxw) / p.dx;
  }
  auto fz = [&](int kk) -> double {
    if (kk <= 0 || kk >= nz) return 0.0;
    const long long a = (long long)kk * n2;
    const double wb = 0.5 * (w[a + q.c] + w[a + q.n]);
    const double above = v[a - n2 + q.c], below = v[a + q.c];
    if (p.advection == ADV_CENTRED2) return wb * 0.5 * (above + below);
    const double far_up = kk >= 2 ? v[a - 2 * n2 + q.c] : 0.0;
    const double far_dn = kk <= nz - 2 ? v[a + n2 + q.c] : 0.0;
    const bool hu = kk >= 2 && m3v[a - 2 * n2 + q.c] != 0;
    const bool hd = kk <= nz - 2 && m3v[a + n2 + q.c] != 0;
    return wb * kappa_face_z(far_up, above, below, far_dn, wb, hu, hd, lim);
  };
  bz = (fz(k) - fz(k + 1)) / p.dz_nom;
  return bx + by + bz;
}

// Masked horizontal Laplacian D o G of a at (o + q.c) with gradient masks
// gmu (x faces), gmv (y faces) and divergence mask dm
// (libs/core/operators_masked.py:64-68).
__device__ __forceinline__ double laplacian(const StepParams& p, const double* a,
                                            const uint8_t* gmu, const uint8_t* gmv,
                                            const uint8_t* dm, long long o, const Nb& q) {
  const double* A = a + o;
  const double gx = mk(gmu[o + q.c]) * (A[q.e] - A[q.c]) / p.dx;
  const double gxw = mk(gmu[o + q.w]) * (A[q.c] - A[q.w]) / p.dx;
  const double gy = mk(gmv[o + q.c]) * (A[q.n] - A[q.c]) / p.dy;
  const double gys = mk(gmv[o + q.s]) * (A[q.c] - A[q.s]) / p.dy;
  return mk(dm[o + q.c]) * ((gx - gxw) / p.dx + (gy - gys) / p.dy);
}

// One lane per cell: the step's explicit momentum terms from the state at
// the start of the step (libs/core/model3d_v05.py:352-370):
//   pgx, pgy   baroclinic pressure gradient at the face depth (:195-230)
//   avu, avv   Coriolis partners avg_u_to_v(u), avg_v_to_u(v)
//   dzu, dzv   explicit vertical diffusion with surface stress and drag
//   stu, stv   theta_v dt tau / dz (k = 0) + dt * (-advection + A_h lap)
__global__ void k_momentum_explicit(Dims d, StepParams p, Geo geo, const double* __restrict__ u,
                                    const double* __restrict__ v, const double* __restrict__ b,
                                    const double* __restrict__ phi, const double* __restrict__ w,
                                    const double* __restrict__ Km, double* __restrict__ pgx,
                                    double* __restrict__ pgy, double* __restrict__ avu,
                                    double* __restrict__ avv, double* __restrict__ dzu,
                                    double* __restrict__ dzv, double* __restrict__ stu,
                                    double* __restrict__ stv) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.n3) return;
  const long long c = t % d.n2;
  const int k = (int)(t / d.n2);
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const Nb q = neighbours(d, j, i);
  const long long o = (long long)k * d.n2;

  // pressure gradient
  double gx, gy;
  if (p.pgf_correction) {
    const double zc = geo.zc[o + c];
    {
      const double zr = geo.zc[o + q.e];
      const double zf = 0.5 * (zc + zr);
      const double left = phi[o + c] + b[o + c] * (zf - zc);
      const double right = phi[o + q.e] + b[o + q.e] * (zf - zr);
      gx = mk(geo.m3u[o + c]) * (right - left) / p.dx;
    }
    {
      const double zr = geo.zc[o + q.n];
      const double zf = 0.5 * (zc + zr);
      const double left = phi[o + c] + b[o + c] * (zf - zc);
      const double right = phi[o + q.n] + b[o + q.n] * (zf - zr);
      gy = mk(geo.m3v[o + c]) * (right - left) / p.dy;
    }
  } else {
    gx = mk(geo.m3u[o + c]) * (phi[o + q.e] - phi[o + c]) / p.dx * mk(geo.m3u[o + c]);
    gy = mk(geo.m3v[o + c]) * (phi[o + q.n] - phi[o + c]) / p.dy * mk(geo.m3v[o + c]);
  }
  pgx[t] = gx;
  pgy[t] = gy;

  {  // the Coriolis partners, for callers that ask for them
    if (avv) avv[t] = avg_v_to_u(v, geo.m3v, geo.m3u, o, q);
    if (avu) avu[t] = avg_u_to_v(u, geo.m3u, geo.m3v, o, q);
  }

  dzu[t] = explicit_diffusion(d, geo.m3, u, Km, geo.dz3u, k == 0 ? geo.tau_u[c] : 0.0,
                              p.bottom_drag, c, k);
  dzv[t] = explicit_diffusion(d, geo.m3, v, Km, geo.dz3v, k == 0 ? geo.tau_v[c] : 0.0,
                              p.bottom_drag, c, k);

  double exu = 0.0, exv = 0.0;
  if (p.advection != ADV_NONE) {
    double au, av;
    if (p.advection == ADV_UPWIND1) {
      // upwind1 momentum uses the centred2 form (libs/core/model3d_v05.py:251-254)
      StepParams pc = p;
      pc.advection = ADV_CENTRED2;
      au = advect_u(d, pc, geo.m3u, u, v, w, o, k, q);
      av = advect_v(d, pc, geo.m3v, u, v, w, o, k, q);
    } else {
      au = advect_u(d, p, geo.m3u, u, v, w, o, k, q);
      av = advect_v(d, p, geo.m3v, u, v, w, o, k, q);
    }
    exu = exu - au * mk(geo.m3u[o + c]);
    exv = exv - av * mk(geo.m3v[o + c]);
  }
  if (p.has_A_h) {
    exu = exu + p.A_h * laplacian(p, u, geo.m3u, geo.m3v, geo.m3u, o, q);
    exv = exv + p.A_h * laplacian(p, v, geo.m3u, geo.m3v, geo.m3v, o, q);
  }
  double s0u = 0.0, s0v = 0.0;
  if (k == 0) {
    s0u = p.thv_dt * geo.tau_u[c] * safe_inv(geo.dz3u[c]);
    s0v = p.thv_dt * geo.tau_v[c] * safe_inv(geo.dz3v[c]);
  }
  stu[t] = s0u + p.dt * exu;
  stv[t] = s0v + p.dt * exv;
}

// Depth-integrated transports U = sum_k dz3u u, V = sum_k dz3v v (k order).
__global__ void k_depth_sum(Dims d, StepParams p, Geo geo, const double* __restrict__ u,
                            const double* __restrict__ v, double* __restrict__ U,
                            double* __restrict__ V) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const long long n2 = d.n2;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const FaceGeo fu(geo, p, d, c, at2(d, j, wrap(i, 1, d.nx)), 0);
  const FaceGeo fv(geo, p, d, c, at2(d, wrap(j, 1, d.ny), i), 1);
  double su = 0.0, sv = 0.0;
  for (int k = 0; k < d.nz; ++k) {
    const double tu = fu.dz(k) * u[k * n2 + c];
    const double tv = fv.dz(k) * v[k * n2 + c];
    su = (k == 0) ? tu : su + tu;
    sv = (k == 0) ? tv : sv + tv;
  }
  U[c] = su;
  V[c] = sv;
}

// div = mask ((U - U_w)/dx + (V - V_s)/dy) (libs/core/operators_masked.py:27-32).
__device__ __forceinline__ double div2(const Dims& d, const StepParams& p, const Geo& geo,
                                       const double* U, const double* V, long long c) {
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const long long cw = at2(d, j, wrap(i, -1, d.nx));
  const long long cs = at2(d, wrap(j, -1, d.ny), i);
  return mk(geo.m2[c]) * ((U[c] - U[cw]) / p.dx + (V[c] - V[cs]) / p.dy);
}

// Barotropic divergence with the Flather transports on open edges
// (model3d_v05.py:262-309): on an open edge column the wrapped neighbour
// flux of the masked divergence is swapped for the radiating transport
// u_ext -/+ sqrt(g max(H, 1)) (eta - eta_ext), x edges first, then the
// result is masked again.
__device__ __forceinline__ double div_bt(const Dims& d, const StepParams& p, const Geo& geo,
                                         const double* U, const double* V, const double* eta,
                                         long long c) {
  double dv = div2(d, p, geo, U, V, c);
  if (!p.open_x && !p.open_y) return dv;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  if (p.open_x) {
    const long long cw = at2(d, j, wrap(i, -1, d.nx));
    const double cg = sqrt(p.g * nmax(geo.H[c], 1.0));
    if (i == 0) {
      const double bw = p.u_ext - cg * (eta[c] - p.eta_ext);
      dv = dv + ((U[c] - bw) / p.dx - ((U[c] - U[cw]) / p.dx));
    }
    if (i == d.nx - 1) {
      const double be = p.u_ext + cg * (eta[c] - p.eta_ext);
      dv = dv + ((be - U[cw]) / p.dx - ((U[c] - U[cw]) / p.dx));
    }
  }
  if (p.open_y) {
    const long long cs = at2(d, wrap(j, -1, d.ny), i);
    const double cg = sqrt(p.g * nmax(geo.H[c], 1.0));
    if (j == 0) {
      const double bs = p.u_ext - cg * (eta[c] - p.eta_ext);
      dv = dv + ((V[c] - bs) / p.dy - ((V[c] - V[cs]) / p.dy));
    }
    if (j == d.ny - 1) {
      const double bn = p.u_ext + cg * (eta[c] - p.eta_ext);
      dv = dv + ((bn - V[cs]) / p.dy - ((V[c] - V[cs]) / p.dy));
    }
  }
  return dv * mk(geo.m2[c]);
}

__global__ void k_div2(Dims d, StepParams p, Geo geo, const double* __restrict__ U,
                       const double* __restrict__ V, const double* __restrict__ eta,
                       double* __restrict__ out) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  out[c] = div_bt(d, p, geo, U, V, eta, c);
}

// rhs = eta - dt ((1 - th) div_old + th div(U_g, V_g))  (model3d_v05.py:398-400)
__global__ void k_rhs_eta(Dims d, StepParams p, Geo geo, const double* __restrict__ eta,
                          const double* __restrict__ div_old, const double* __restrict__ Ug,
                          const double* __restrict__ Vg, double* __restrict__ rhs) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const double dg = div_bt(d, p, geo, Ug, Vg, eta, c);
  rhs[c] = eta[c] - p.dt * (p.one_m_th * div_old[c] + p.th * dg);
}

// fb: eta_new = eta - dt div(U, V)  (model3d_v05.py:410-413)
__global__ void k_eta_fb(Dims d, StepParams p, Geo geo, const double* __restrict__ eta,
                         const double* __restrict__ U, const double* __restrict__ V,
                         double* __restrict__ eta_new) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  eta_new[c] = eta[c] - p.dt * div_bt(d, p, geo, U, V, eta, c);
}

// ---------------------------------------------- split-explicit mode
// Barotropic forcing of the split scheme (model3d_v05.py:445-452): the
// Coriolis the barotropic step adds back, formed with the same 2D transport
// averages, removed from the depth-integrated baroclinic tendency.
__global__ void k_split_forcing(Dims d, StepParams p, Geo geo, const double* __restrict__ U0,
                                const double* __restrict__ V0, const double* __restrict__ Um,
                                const double* __restrict__ Vm, double* __restrict__ fx,
                                double* __restrict__ fy) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const Nb q = neighbours(d, j, i);
  const double cor_x = p.f * (p.one_m_tc * avg_v_to_u(V0, geo.mv2, geo.mu2, 0, q) +
                              p.theta_cor * avg_v_to_u(Vm, geo.mv2, geo.mu2, 0, q));
  const double cor_y = p.neg_f * (p.one_m_tc * avg_u_to_v(U0, geo.mu2, geo.mv2, 0, q) +
                                  p.theta_cor * avg_u_to_v(Um, geo.mu2, geo.mv2, 0, q));
  fx[c] = (Um[c] - U0[c]) / p.dt - cor_x;
  fy[c] = (Vm[c] - V0[c]) / p.dt - cor_y;
}

// One Picard pass of a barotropic substep (model3d_v05.py:321-327): from the
// substep's start U, V, e and the current iterate Ui, Vi.
__global__ void k_bt_picard(Dims d, StepParams p, Geo geo, const double* __restrict__ U,
                            const double* __restrict__ V, const double* __restrict__ e,
                            const double* __restrict__ Ui, const double* __restrict__ Vi,
                            const double* __restrict__ fx, const double* __restrict__ fy,
                            const double* __restrict__ Ku, const double* __restrict__ Kv,
                            double* __restrict__ Uo, double* __restrict__ Vo) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const Nb q = neighbours(d, j, i);
  const double mu = mk(geo.mu2[c]), mv = mk(geo.mv2[c]);
  const double gxe = mu * (e[q.e] - e[c]) / p.dx;
  const double gye = mv * (e[q.n] - e[c]) / p.dy;
  const double v_cor = p.one_m_tc * avg_v_to_u(V, geo.mv2, geo.mu2, 0, q) +
                       p.theta_cor * avg_v_to_u(Vi, geo.mv2, geo.mu2, 0, q);
  const double u_cor = p.one_m_tc * avg_u_to_v(U, geo.mu2, geo.mv2, 0, q) +
                       p.theta_cor * avg_u_to_v(Ui, geo.mu2, geo.mv2, 0, q);
  Uo[c] = (U[c] + p.ddt * (p.f * v_cor - p.g * Ku[c] * gxe + fx[c])) * mu;
  Vo[c] = (V[c] + p.ddt * (p.neg_f * u_cor - p.g * Kv[c] * gye + fy[c])) * mv;
}

// e_new = e - ddt div(U, V); the transports summed for the averaged mode
// (model3d_v05.py:329-331).
__global__ void k_bt_eta(Dims d, StepParams p, Geo geo, const double* __restrict__ e,
                         const double* __restrict__ U, const double* __restrict__ V,
                         double* __restrict__ e_new, double* __restrict__ acc_u,
                         double* __restrict__ acc_v) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  e_new[c] = e[c] - p.ddt * div_bt(d, p, geo, U, V, e, c);
  if (acc_u) {
    acc_u[c] = acc_u[c] + U[c];
    acc_v[c] = acc_v[c] + V[c];
  }
}

// Up to S barotropic substeps of P Picard passes each in one launch, the same
// operations per cell as k_bt_picard and k_bt_eta: a tile of BT_W x BT_H cells
// with the halo that S substeps need (one cell per pass and one for the
// level), one thread per cell of the region, its coefficients and own values in
// registers and the fields that neighbours read in LDS. A cell beyond the halo
// reads itself; no cell of the tile sees its value. From U, V, e into Uo, Vo,
// eo; acc_u, acc_v: the transports summed for the averaged mode (from substep
// 0 on; n0 is this launch's first), or null.
//
// Bound: latency (launch, loads, P + 1 barriers per substep). Two substeps of
// two passes on 197 x 131 take 7.2 us against 24 in six launches; a step on 64 x
// 64 x 12 188 us against 271, on 400 x 400 x 12 796 against 871, on 1000 x 1000
// x 12 4429 against 4477. Tiles of 16 x 8 gain 1 to 3% on the small grids and
// lose as much on the 400 x 400 one; three substeps per launch likewise.
constexpr int BT_W = 16, BT_H = 16;
template <int S, int P>
struct BtRegion {
  static constexpr int H = S * (P + 1), RW = BT_W + 2 * H, RH = BT_H + 2 * H, RN = RW * RH;
  static constexpr int NT = (RN + 63) / 64 * 64;
};
template <int S, int P>
__global__ __launch_bounds__((BtRegion<S, P>::NT)) void k_bt_substeps(
    Dims d, StepParams p, Geo geo, int n0, int ns, const double* __restrict__ U,
    const double* __restrict__ V, const double* __restrict__ e, const double* __restrict__ fx,
    const double* __restrict__ fy, const double* __restrict__ Ku,
    const double* __restrict__ Kv, double* __restrict__ Uo, double* __restrict__ Vo,
    double* __restrict__ eo, double* __restrict__ acc_u, double* __restrict__ acc_v) {
  using Rg = BtRegion<S, P>;
  constexpr int RW = Rg::RW, RH = Rg::RH, H = Rg::H;
  __shared__ double lu[3][Rg::RN], lv[3][Rg::RN], le[Rg::RN];
  const bool on = (int)threadIdx.x < Rg::RN;
  const int t = on ? (int)threadIdx.x : 0;
  const int li = t % RW, lj = t / RW;
  const int nx = d.nx, ny = d.ny;
  auto wrapped = [](int x, int n) {
    x %= n;
    return x < 0 ? x + n : x;
  };
  const int ui = (int)blockIdx.x * BT_W + li - H, uj = (int)blockIdx.y * BT_H + lj - H;
  const int i = wrapped(ui, nx), j = wrapped(uj, ny);
  const Nb q = neighbours(d, j, i);
  const int c = q.c;
  // the region's neighbours
  const int te = li + 1 < RW ? t + 1 : t, tw = li > 0 ? t - 1 : t;
  const int tn = lj + 1 < RH ? t + RW : t, ts = lj > 0 ? t - RW : t;
  const int tse = lj > 0 && li + 1 < RW ? t - RW + 1 : t;
  const int tnw = lj + 1 < RH && li > 0 ? t + RW - 1 : t;
  const bool ov = geo.mv2[c] != 0, ou = geo.mu2[c] != 0;
  const bool fv[4] = {ov, geo.mv2[q.s] != 0, geo.mv2[q.e] != 0, geo.mv2[q.se] != 0};
  const bool fu[4] = {ou, geo.mu2[q.w] != 0, geo.mu2[q.n] != 0, geo.mu2[q.nw] != 0};
  const double mu = ou ? 1.0 : 0.0, mv = ov ? 1.0 : 0.0, m = mk(geo.m2[c]);
  const double fxc = fx[c], fyc = fy[c], gKu = p.g * Ku[c], gKv = p.g * Kv[c];
  const double cg = p.open_x || p.open_y ? sqrt(p.g * nmax(geo.H[c], 1.0)) : 0.0;
  const Divisor<double> by_dx = uniform_divisor<double>(p.dx), by_dy = uniform_divisor<double>(p.dy);
  const Avg4 to_u(fv, ou), to_v(fu, ov);
  double u0 = U[c], v0 = V[c], ec = e[c];
  const bool own = on && li >= H && li < H + BT_W && lj >= H && lj < H + BT_H && ui < nx && uj < ny;
  double au = 0.0, av = 0.0;
  if (acc_u && own && n0 > 0) {
    au = acc_u[c];
    av = acc_v[c];
  }
  int start = 0;  // the buffers of the substep's start and of the last iterate
  if (on) {
    lu[0][t] = u0;
    lv[0][t] = v0;
    le[t] = ec;
  }
  __syncthreads();
  for (int n = 0; n < ns; ++n) {
    const double gxe = by_dx(mu * (le[te] - ec)), gye = by_dy(mv * (le[tn] - ec));
    auto avg_v = [&](const double* f, double own_v) { return to_u(own_v, f[ts], f[te], f[tse]); };
    auto avg_u = [&](const double* f, double own_u) { return to_v(own_u, f[tw], f[tn], f[tnw]); };
    const double av0 = avg_v(lv[start], v0), au0 = avg_u(lu[start], u0);
    double un = u0, vn = v0;
    int it = start;
#pragma unroll
    for (int m_ = 0; m_ < P; ++m_) {
      const double v_cor = p.one_m_tc * av0 + p.theta_cor * (m_ == 0 ? av0 : avg_v(lv[it], vn));
      const double u_cor = p.one_m_tc * au0 + p.theta_cor * (m_ == 0 ? au0 : avg_u(lu[it], un));
      un = (u0 + p.ddt * (p.f * v_cor - gKu * gxe + fxc)) * mu;
      vn = (v0 + p.ddt * (p.neg_f * u_cor - gKv * gye + fyc)) * mv;
      int nxt = 0;  // the buffer that is neither the start's nor the last iterate's
      while (nxt == start || nxt == it) ++nxt;
      if (on) {
        lu[nxt][t] = un;
        lv[nxt][t] = vn;
      }
      it = nxt;
      __syncthreads();
    }
    // e - ddt div(U, V) as div_bt forms it
    const double uw = lu[it][tw], vs = lv[it][ts];
    double dv = m * (by_dx(un - uw) + by_dy(vn - vs));
    if (p.open_x || p.open_y) {
      if (p.open_x && i == 0) {
        const double bw = p.u_ext - cg * (ec - p.eta_ext);
        dv = dv + (by_dx(un - bw) - by_dx(un - uw));
      }
      if (p.open_x && i == nx - 1) {
        const double be = p.u_ext + cg * (ec - p.eta_ext);
        dv = dv + (by_dx(be - uw) - by_dx(un - uw));
      }
      if (p.open_y && j == 0) {
        const double bs = p.u_ext - cg * (ec - p.eta_ext);
        dv = dv + (by_dy(vn - bs) - by_dy(vn - vs));
      }
      if (p.open_y && j == ny - 1) {
        const double bn = p.u_ext + cg * (ec - p.eta_ext);
        dv = dv + (by_dy(bn - vs) - by_dy(vn - vs));
      }
      dv = dv * m;
    }
    ec = ec - p.ddt * dv;
    if (on) le[t] = ec;
    u0 = un;
    v0 = vn;
    start = it;
    au = au + un;
    av = av + vn;
    if (n + 1 < ns) __syncthreads();
  }
  if (!own) return;
  Uo[c] = u0;
  Vo[c] = v0;
  eo[c] = ec;
  if (acc_u) {
    acc_u[c] = au;
    acc_v[c] = av;
  }
}

bool launch_bt_substeps(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo, int n0,
                        int ns, const double* U, const double* V, const double* e, const double* fx,
                        const double* fy, const double* Ku, const double* Kv, double* Uo,
                        double* Vo, double* eo, double* acc_u, double* acc_v) {
  const dim3 grid((unsigned)((d.nx + BT_W - 1) / BT_W), (unsigned)((d.ny + BT_H - 1) / BT_H));
  auto go = [&](auto pp) {
    constexpr int P = decltype(pp)::value;
    k_bt_substeps<BT_SUBSTEPS, P><<<grid, BtRegion<BT_SUBSTEPS, P>::NT, 0, s>>>(
        d, p, geo, n0, ns, U, V, e, fx, fy, Ku, Kv, Uo, Vo, eo, acc_u, acc_v);
  };
  // a region of up to 1024 cells: three passes at most
  if (p.n_picard == 1) go(std::integral_constant<int, 1>{});
  else if (p.n_picard == 2) go(std::integral_constant<int, 2>{});
  else if (p.n_picard == 3) go(std::integral_constant<int, 3>{});
  else return false;
  return true;
}

__global__ void k_bt_mean(Dims d, StepParams p, const double* __restrict__ acc_u,
                          const double* __restrict__ acc_v, double* __restrict__ U,
                          double* __restrict__ V) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  U[c] = acc_u[c] / (double)p.n_split;
  V[c] = acc_v[c] / (double)p.n_split;
}

// Depth-mean replacement (model3d_v05.py:454-462): u = (gh_u - Um/Hu + U/Hu)
// on the wet u faces, with Hu = sum_k dz3u.
__global__ void k_split_final(Dims d, Geo geo, const double* __restrict__ gh_u,
                              const double* __restrict__ gh_v, const double* __restrict__ Um,
                              const double* __restrict__ Vm, const double* __restrict__ U,
                              const double* __restrict__ V, const double* __restrict__ Hu,
                              const double* __restrict__ Hv, double* __restrict__ u,
                              double* __restrict__ v) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.n3) return;
  const long long c = t % d.n2;
  const double ihu = safe_inv(Hu[c]), ihv = safe_inv(Hv[c]);
  u[t] = (gh_u[t] - Um[c] * ihu + U[c] * ihu) * mk(geo.m3u[t]);
  v[t] = (gh_v[t] - Vm[c] * ihv + V[c] * ihv) * mk(geo.m3v[t]);
}

// Hu = sum_k dz3u, Hv = sum_k dz3v, summed from the surface.
__global__ void k_face_depth(Dims d, Geo geo, double* __restrict__ Hu, double* __restrict__ Hv) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  double su = 0.0, sv = 0.0;
  for (int k = 0; k < d.nz; ++k) {
    su = (k == 0) ? geo.dz3u[c] : su + geo.dz3u[k * d.n2 + c];
    sv = (k == 0) ? geo.dz3v[c] : sv + geo.dz3v[k * d.n2 + c];
  }
  Hu[c] = su;
  Hv[c] = sv;
}

// ------------------------------------------- predictor and column solves
// One Picard pass (model3d_v05.py:387-396), one wave per 64 columns and
// velocity component:
//   v_cor = (1-tc) avg_v_to_u(v) + tc avg_v_to_u(v_it),  u_cor likewise
// (both partners formed here, from the state and from the iterate; FIRST: the
// iterate is the state)
//   gu = u + dt (f v_cor + pgx) - g dt (1-th) Gx(eta) + (1-thv) dt dzu
//   gh_u = A_m^-1 (gu + stu) * mask3, and the same for v,
// then the depth sums Ug = sum dz3u gh_u, Vg = sum dz3v gh_v for the
// Helmholtz right-hand side. ZC: masks and thicknesses from the columns' wet
// levels (a face mask at level k is k < its threshold: the 2D face mask and
// the shallower of the face's two cells) instead of the arrays, the same bits.
// STAGE: d* and the solution stay in LDS between the three sweeps instead of
// in gh_u / gh_v.
//
// Bound: memory on large grids (16 fields of the grid in a first pass, 20 in
// a later one, and the neighbour rows of two), latency of the
// march on small ones. One wave per component, operands two levels ahead and
// d* in LDS, against one lane for both components, no loads ahead and d*, x in
// memory, per launch (mean of both passes): 128 x 4 x 20 47 -> 17 us, 128 x
// 128 x 30 84 -> 25, 512 x 512 x 40 322 -> 305, 640 x 512 x 48 584 -> 449,
// 1000 x 1000 x 30 930 -> 795. Four levels ahead cost more in registers than
// they hide (1000 x 1000 x 30: 891).
constexpr int PRED_AHEAD = 2;
template <bool ZC, bool FIRST, bool STAGE>
__global__ __launch_bounds__(2 * COLS) void k_predictor(
    Dims d, StepParams p, Geo geo, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ eta, const double* __restrict__ u_it,
    const double* __restrict__ v_it, const double* __restrict__ pgx,
    const double* __restrict__ pgy, const double* __restrict__ dzu,
    const double* __restrict__ dzv, const double* __restrict__ stu,
    const double* __restrict__ stv, const double* __restrict__ sub,
    const double* __restrict__ den, const double* __restrict__ cst, double* __restrict__ gh_u,
    double* __restrict__ gh_v, double* __restrict__ Ug, double* __restrict__ Vg) {
  extern __shared__ double pred_lds[];  // STAGE: [2][nz][COLS], a thread's own column
  const int comp = __builtin_amdgcn_readfirstlane(threadIdx.x / COLS);
  const int lane = threadIdx.x % COLS;
  const long long c = (long long)xcd_linear() * COLS + lane;
  if (c >= d.n2) return;
  const int j = (int)((unsigned)c / (unsigned)d.nx), i = (int)((unsigned)c - (unsigned)j * d.nx);
  const Nb q = neighbours(d, j, i);
  const long long n2 = d.n2;
  const int nz = d.nz;
  const bool split = p.scheme == SCHEME_SPLIT;
  // this component's field and, of the other one's, the four faces round it
  const double* f = comp ? v : u;
  const double* g = comp ? u : v;
  const double* gi = comp ? u_it : v_it;
  const double* pg = comp ? pgy : pgx;
  const double* dzf = comp ? dzv : dzu;
  const double* st = comp ? stv : stu;
  double* gh = comp ? gh_v : gh_u;
  const uint8_t* mo = comp ? geo.m3v : geo.m3u;
  const uint8_t* mg = comp ? geo.m3u : geo.m3v;
  const int o4[4] = {q.c, comp ? q.w : q.s, comp ? q.n : q.e, comp ? q.nw : q.se};
  const double fc = comp ? p.neg_f : p.f;
  const int far = comp ? q.n : q.e;
  const uint8_t* m2o = comp ? geo.mv2 : geo.mu2;
  const double ge = mk(m2o[c]) * (eta[far] - eta[c]) / (comp ? p.dy : p.dx);
  int th[4] = {}, tho = 0, nwc = 0;
  if constexpr (ZC) {
    nwc = geo.nw[c];
    const uint8_t* m2g = comp ? geo.mu2 : geo.mv2;
    const int far4[4] = {comp ? q.e : q.n, q.c, q.ne, comp ? q.n : q.e};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int a = geo.nw[o4[t]], b = geo.nw[far4[t]];
      th[t] = m2g[o4[t]] ? (a < b ? a : b) : 0;
    }
    const int b = geo.nw[far];
    tho = m2o[c] ? (nwc < b ? nwc : b) : 0;
  }
  struct Level {
    double f, g[4], gi[FIRST ? 1 : 4], pg, dz, st, sub, den;
    uint8_t m[ZC ? 1 : 5];
  };
  double* lds = STAGE ? pred_lds + (size_t)comp * nz * COLS + lane : nullptr;
  const unsigned bc = 8u * (unsigned)c;
  double prev = 0.0;
  march_down<PRED_AHEAD>(
      nz,
      [&](int k) {
        const long long o = k * n2;
        Level L;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          L.g[s] = at_byte(g + o, 8u * (unsigned)o4[s]);
          if constexpr (!FIRST) L.gi[s] = at_byte(gi + o, 8u * (unsigned)o4[s]);
          if constexpr (!ZC) L.m[s] = at_byte(mg + o, (unsigned)o4[s]);
        }
        if constexpr (!ZC) L.m[4] = at_byte(mo + o, (unsigned)c);
        L.f = at_byte(f + o, bc);
        L.pg = at_byte(pg + o, bc);
        L.dz = at_byte(dzf + o, bc);
        L.st = at_byte(st + o, bc);
        L.sub = at_byte(sub + o, bc);
        L.den = at_byte(den + o, bc);
        return L;
      },
      [&](int k, const Level& L) {
        bool open[4], own;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if constexpr (ZC) open[s] = k < th[s];
          else open[s] = L.m[s] != 0;
        }
        if constexpr (ZC) own = k < tho;
        else own = L.m[4] != 0;
        const double av = avg4(L.g, open, own);
        const double av_it = FIRST ? av : avg4(L.gi, open, own);
        const double cor = p.one_m_tc * av + p.theta_cor * av_it;
        const double gxe = ge * (own ? 1.0 : 0.0);
        // split_explicit leaves the surface gradient to the barotropic substeps
        // (model3d_v05.py:431-432)
        const double r0 = L.f + p.dt * (fc * cor + L.pg);
        const double r1 = split ? r0 : r0 - p.c_gx * gxe;
        const double rhs = (r1 + p.c_dzd * L.dz) + L.st;
        const Divisor<double> by_den(L.den);
        prev = k == 0 ? by_den(rhs) : by_den(rhs - L.sub * prev);
        if constexpr (STAGE) lds[k * COLS] = prev;
        else put_byte(gh + k * n2, bc, prev);
      });
  struct Back {
    double cst, d;
    uint8_t m;
  };
  double x = 0.0;
  march_up<8>(
      nz,
      [&](int k) {
        const long long o = k * n2;
        Back B;
        B.cst = at_byte(cst + o, bc);
        if constexpr (STAGE) B.d = lds[k * COLS];
        else B.d = at_byte(gh + o, bc);
        if constexpr (ZC) B.m = k < nwc;
        else B.m = at_byte(geo.m3 + o, (unsigned)c);
        return B;
      },
      [&](int k, const Back& B) {
        x = k == nz - 1 ? B.d : B.d - B.cst * x;
        const double xm = x * mk(B.m);
        if constexpr (STAGE) lds[k * COLS] = xm;
        put_byte(gh + k * n2, bc, xm);
      });
  FaceCol face{};
  if constexpr (ZC) face = face_col(geo, p, c, far, comp);
  const double* dzface = comp ? geo.dz3v : geo.dz3u;
  struct Sum {
    double dz, x;
  };
  double s = 0.0;
  march_down<8>(
      nz,
      [&](int k) {
        Sum S;
        S.dz = ZC ? 0.0 : at_byte(dzface + k * n2, bc);
        if constexpr (STAGE) S.x = lds[k * COLS];
        else S.x = at_byte(gh + k * n2, bc);
        return S;
      },
      [&](int k, const Sum& S) {
        const double t = (ZC ? face.dz(k) : S.dz) * S.x;
        s = k == 0 ? t : s + t;
      });
  (comp ? Vg : Ug)[c] = s;
}

void launch_predictor(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                      const double* u, const double* v, const double* eta, const double* u_it,
                      const double* v_it, const double* pgx, const double* pgy,
                      const double* dzu, const double* dzv, const double* stu,
                      const double* stv, const double* sub, const double* den,
                      const double* cst, double* gh_u, double* gh_v, double* Ug, double* Vg) {
  const size_t lds = (size_t)2 * d.nz * COLS * sizeof(double);
  with_column_form(p.zcol != 0, lds <= COL_LDS_MAX, [&](auto zc, auto sg) {
    constexpr bool ZC = decltype(zc)::value, SG = decltype(sg)::value;
    auto go = [&](auto fi) {
      k_predictor<ZC, decltype(fi)::value, SG><<<column_blocks(d), 2 * COLS, SG ? lds : 0, s>>>(
          d, p, geo, u, v, eta, u_it, v_it, pgx, pgy, dzu, dzv, stu, stv, sub, den, cst, gh_u,
          gh_v, Ug, Vg);
    };
    if (u_it == u && v_it == v) go(std::true_type{});
    else go(std::false_type{});
  });
}

// u_it = (gh_u - g dt th q Gx(eta_new) mask3u) mask3 (model3d_v05.py:404-406)
__global__ void k_backsub(Dims d, StepParams p, Geo geo, const double* __restrict__ gh_u,
                          const double* __restrict__ gh_v, const double* __restrict__ q,
                          const double* __restrict__ eta_n, double* __restrict__ u_it,
                          double* __restrict__ v_it) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.n3) return;
  const long long c = t % d.n2;
  const int i = (int)(c % d.nx), j = (int)(c / d.nx);
  const long long ce = at2(d, j, wrap(i, 1, d.nx));
  const long long cn = at2(d, wrap(j, 1, d.ny), i);
  const double gx = mk(geo.mu2[c]) * (eta_n[ce] - eta_n[c]) / p.dx;
  const double gy = mk(geo.mv2[c]) * (eta_n[cn] - eta_n[c]) / p.dy;
  bool m3, m3u, m3v;
  if (p.zcol) {
    const int k = (int)(t / d.n2);
    const int nwc = geo.nw[c];
    m3 = k < nwc;
    m3u = geo.mu2[c] && m3 && k < geo.nw[ce];
    m3v = geo.mv2[c] && m3 && k < geo.nw[cn];
  } else {
    m3 = geo.m3[t] != 0;
    m3u = geo.m3u[t] != 0;
    m3v = geo.m3v[t] != 0;
  }
  const double mm = m3 ? 1.0 : 0.0;
  u_it[t] = (gh_u[t] - p.c_bs * q[t] * gx * (m3u ? 1.0 : 0.0)) * mm;
  v_it[t] = (gh_v[t] - p.c_bs * q[t] * gy * (m3v ? 1.0 : 0.0)) * mm;
}

// The last Picard pass's back-substitution fused with w of the new
// velocity (model3d_v05.py:404-406 then 232-235), one lane per column
// marching up from the bottom: u and v of the column are formed and stored
// as k_backsub forms them; the west u and the south v that the transport
// divergence needs are formed again from the same operands (the same bits),
// so w is k_w_diag's of the stored fields without reading them back.
// Two levels ahead, spacings divided by a reciprocal: 128 x 128 x 30 45 -> 20
// us, 512 x 512 x 40 112 -> 103, 640 x 512 x 48 198 -> 160.
template <bool ZC>
__global__ __launch_bounds__(COLS) void k_backsub_w(
    Dims d, StepParams p, Geo geo, const double* __restrict__ gh_u,
    const double* __restrict__ gh_v, const double* __restrict__ q,
    const double* __restrict__ eta_n, double* __restrict__ u, double* __restrict__ v,
    double* __restrict__ w) {
  const long long c = (long long)xcd_linear() * COLS + threadIdx.x;
  if (c >= d.n2) return;
  const int j = (int)((unsigned)c / (unsigned)d.nx), i = (int)((unsigned)c - (unsigned)j * d.nx);
  const long long ce = at2(d, j, wrap(i, 1, d.nx)), cw = at2(d, j, wrap(i, -1, d.nx));
  const long long cn = at2(d, wrap(j, 1, d.ny), i), cs = at2(d, wrap(j, -1, d.ny), i);
  const long long n2 = d.n2;
  const int nz = d.nz;
  // surface-gradient factors of the column and of its west (u) and south (v)
  // neighbours, as k_backsub forms them
  const double gx_c = mk(geo.mu2[c]) * (eta_n[ce] - eta_n[c]) / p.dx;
  const double gx_w = mk(geo.mu2[cw]) * (eta_n[c] - eta_n[cw]) / p.dx;
  const double gy_c = mk(geo.mv2[c]) * (eta_n[cn] - eta_n[c]) / p.dy;
  const double gy_s = mk(geo.mv2[cs]) * (eta_n[c] - eta_n[cs]) / p.dy;
  const unsigned bc = 8u * (unsigned)c, bw = 8u * (unsigned)cw, bs = 8u * (unsigned)cs;
  FaceCol fe{}, fw{}, fn{}, fs{};
  int nwc = 0, nww = 0, nws = 0;
  if constexpr (ZC) {
    fe = face_col(geo, p, c, ce, 0);
    fw = face_col(geo, p, cw, c, 0);
    fn = face_col(geo, p, c, cn, 1);
    fs = face_col(geo, p, cs, c, 1);
    nwc = geo.nw[c];
    nww = geo.nw[cw];
    nws = geo.nw[cs];
  }
  const Divisor<double> by_dx = uniform_divisor<double>(p.dx), by_dy = uniform_divisor<double>(p.dy);
  struct Level {
    double u, v, uw, vs, q, qw, qs, de, dw, dn, ds;
    uint8_t m, mw, ms, me, mfw, mn, mfs;
  };
  double sum = 0.0;
  march_up<2>(
      nz,
      [&](int k) {
        const long long o = k * n2;
        Level L;
        L.u = at_byte(gh_u + o, bc);
        L.v = at_byte(gh_v + o, bc);
        L.uw = at_byte(gh_u + o, bw);
        L.vs = at_byte(gh_v + o, bs);
        L.q = at_byte(q + o, bc);
        L.qw = at_byte(q + o, bw);
        L.qs = at_byte(q + o, bs);
        if constexpr (!ZC) {
          L.de = geo.dz3u[o + c];
          L.dw = geo.dz3u[o + cw];
          L.dn = geo.dz3v[o + c];
          L.ds = geo.dz3v[o + cs];
          L.m = geo.m3[o + c];
          L.mw = geo.m3[o + cw];
          L.ms = geo.m3[o + cs];
          L.me = geo.m3u[o + c];
          L.mfw = geo.m3u[o + cw];
          L.mn = geo.m3v[o + c];
          L.mfs = geo.m3v[o + cs];
        }
        return L;
      },
      [&](int k, const Level& L) {
        const double mc = (ZC ? k < nwc : L.m != 0) ? 1.0 : 0.0;
        const double mw = (ZC ? k < nww : L.mw != 0) ? 1.0 : 0.0;
        const double ms = (ZC ? k < nws : L.ms != 0) ? 1.0 : 0.0;
        const double me = (ZC ? fe.wet(k) : L.me != 0) ? 1.0 : 0.0;
        const double mfw = (ZC ? fw.wet(k) : L.mfw != 0) ? 1.0 : 0.0;
        const double mn = (ZC ? fn.wet(k) : L.mn != 0) ? 1.0 : 0.0;
        const double mfs = (ZC ? fs.wet(k) : L.mfs != 0) ? 1.0 : 0.0;
        const double uc = (L.u - p.c_bs * L.q * gx_c * me) * mc;
        const double vc = (L.v - p.c_bs * L.q * gy_c * mn) * mc;
        const double uw = (L.uw - p.c_bs * L.qw * gx_w * mfw) * mw;
        const double vs = (L.vs - p.c_bs * L.qs * gy_s * mfs) * ms;
        put_byte(u + k * n2, bc, uc);
        put_byte(v + k * n2, bc, vc);
        const double U = (ZC ? fe.dz(k) : L.de) * uc;
        const double Uw = (ZC ? fw.dz(k) : L.dw) * uw;
        const double V = (ZC ? fn.dz(k) : L.dn) * vc;
        const double Vs = (ZC ? fs.dz(k) : L.ds) * vs;
        const double dv = mc * (by_dx(U - Uw) + by_dy(V - Vs));
        sum = (k == nz - 1) ? dv : sum + dv;
        put_byte(w + k * n2, bc, -sum);
      });
  w[(long long)nz * n2 + c] = 0.0;
}

void launch_backsub_w(hipStream_t s, const Dims& d, const StepParams& p, const Geo& geo,
                      const double* gh_u, const double* gh_v, const double* q,
                      const double* eta_n, double* u, double* v, double* w) {
  const unsigned nb = column_blocks(d);
  if (p.zcol) k_backsub_w<true><<<nb, COLS, 0, s>>>(d, p, geo, gh_u, gh_v, q, eta_n, u, v, w);
  else k_backsub_w<false><<<nb, COLS, 0, s>>>(d, p, geo, gh_u, gh_v, q, eta_n, u, v, w);
}

// ------------------------------------------------------------- tracers
// Flux-form tracer advection divergence at (k, j, i) with face thickness
// (libs/core/model3d_v05.py:482-512).
__device__ double tracer_advection(const Dims& d, const StepParams& p, const Geo& geo,
                                   const double* cc, const double* u, const double* v,
                                   const double* w, long long c, int k, const Nb& q) {
  const long long n2 = d.n2;
  const int nz = d.nz;
  const long long o = (long long)k * n2;
  const double* C = cc + o;
  const uint8_t* M = geo.m3 + o;
  const bool up3 = p.advection == ADV_UP3 || p.advection == ADV_UP3_TVD;
  const bool lim = p.advection == ADV_UP3_TVD;
  auto face = [&](double cm, double c0, double c1, double c2, double vel, bool wm,
                  bool w2) -> double {
    if (up3) return kappa_face(cm, c0, c1, c2, vel, wm, w2, lim);
    if (p.advection == ADV_CENTRED2) return 0.5 * (c0 + c1);
    return vel > 0.0 ? c0 : c1;
  };
  const double ue = u[o + q.c], uw = u[o + q.w];
  const double vn = v[o + q.c], vs = v[o + q.s];
  const double cx = face(C[q.w], C[q.c], C[q.e], C[q.ee], ue, M[q.w] != 0, M[q.ee] != 0);
  const double cxw = face(C[q.ww], C[q.w], C[q.c], C[q.e], uw, M[q.ww] != 0, M[q.e] != 0);
  const double cy = face(C[q.s], C[q.c], C[q.n], C[q.nn], vn, M[q.s] != 0, M[q.nn] != 0);
  const double cys = face(C[q.ss], C[q.s], C[q.c], C[q.n], vs, M[q.ss] != 0, M[q.n] != 0);
  const double fx = geo.dz3u[o + q.c] * ue * cx;
  const double fxw = geo.dz3u[o + q.w] * uw * cxw;
  const double fy = geo.dz3v[o + q.c] * vn * cy;
  const double fys = geo.dz3v[o + q.s] * vs * cys;
  const double inv = safe_inv(geo.dz3[o + c]);
  const double hdiv = ((fx - fxw) / p.dx + (fy - fys) / p.dy) * inv;
  auto cf = [&](int kk) -> double {  // interface value, kk in 0..nz
    if (kk == 0) return cc[c];
    if (kk == nz) return 0.0;
    const long long a = (long long)kk * n2;
    const double above = cc[a - n2 + c], below = cc[a + c];
    if (!up3) return 0.5 * (above + below);
    const double far_up = kk >= 2 ? cc[a - 2 * n2 + c] : 0.0;
    const double far_dn = kk <= nz - 2 ? cc[a + n2 + c] : 0.0;
    const bool hu = kk >= 2 && geo.m3[a - 2 * n2 + c] != 0;
    const bool hd = kk <= nz - 2 && geo.m3[a + n2 + c] != 0;
    return kappa_face_z(far_up, above, below, far_dn, w[a + c], hu, hd, lim);
  };
  const double vdiv = (w[o + c] * cf(k) - w[o + n2 + c] * cf(k + 1)) * inv;
  return (hdiv + vdiv) * mk(M[q.c]);
}

// ---------------------------------------------- standalone operator kernels
// Batched tridiagonal solve, one lane per column (libs/core/vertical.py:17-44);
// x holds d* between the sweeps, cs holds c*.
__global__ void k_thomas(long long ncol, int n, const double* __restrict__ sub,
                         const double* __restrict__ diag, const double* __restrict__ sup,
                         const double* __restrict__ rhs, double* __restrict__ x,
                         double* __restrict__ cs) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncol) return;
  double cp = 0.0, dp = 0.0;
  for (int k = 0; k < n; ++k) {
    const long long t = k * ncol + c;
    double cc, dd;
    if (k == 0) {
      cc = sup[t] / diag[t];
      dd = rhs[t] / diag[t];
    } else {
      const double den = diag[t] - sub[t] * cp;
      cc = sup[t] / den;
      dd = (rhs[t] - sub[t] * dp) / den;
    }
    cs[t] = cc;
    x[t] = dd;
    cp = cc;
    dp = dd;
  }
  double xn = x[(long long)(n - 1) * ncol + c];
  for (int k = n - 2; k >= 0; --k) {
    const long long t = k * ncol + c;
    xn = x[t] - cs[t] * xn;
    x[t] = xn;
  }
}

// Buoyancy from T, S at depth z for n points (libs/core/eos.py:130-133).
__global__ void k_eos(long long n, StepParams p, const double* __restrict__ T,
                      const double* __restrict__ S, const double* __restrict__ z,
                      double* __restrict__ b) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  b[t] = buoyancy(p, T[t], S[t], z[t]);
}

// Tracer advection divergence over the whole 3D field (the operator alone).
__global__ void k_tracer_advection(Dims d, StepParams p, Geo geo, const double* __restrict__ cc,
                                   const double* __restrict__ u, const double* __restrict__ v,
                                   const double* __restrict__ w, double* __restrict__ out) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.n3) return;
  const long long c = t % d.n2;
  const int k = (int)(t / d.n2);
  const Nb q = neighbours(d, (int)(c / d.nx), (int)(c % d.nx));
  out[t] = tracer_advection(d, p, geo, cc, u, v, w, c, k, q);
}

// Momentum advection (u, v) over the whole field (the operator alone).
__global__ void k_momentum_advection(Dims d, StepParams p, Geo geo, const double* __restrict__ u,
                                     const double* __restrict__ v, const double* __restrict__ w,
                                     double* __restrict__ au, double* __restrict__ av) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= d.n3) return;
  const long long c = t % d.n2;
  const int k = (int)(t / d.n2);
  const Nb q = neighbours(d, (int)(c / d.nx), (int)(c % d.nx));
  const long long o = (long long)k * d.n2;
  au[t] = advect_u(d, p, geo.m3u, u, v, w, o, k, q);
  av[t] = advect_v(d, p, geo.m3v, u, v, w, o, k, q);
}

}  // namespace hoc
