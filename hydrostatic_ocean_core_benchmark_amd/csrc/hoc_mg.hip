// Multigrid hierarchy and smoothers of the Helmholtz solvers
// (libs/core/solvers_var.py:63-160, plus the pcg_mg preconditioner):
//   coarse operators by face agglomeration, red-black Gauss-Seidel and
//   damped Jacobi sweeps, residual + full-weighting restriction, masked
//   piecewise-constant prolongation. Elementwise only -- every kernel is one
//   pass over a level -- and in the reference's operand order, so the
//   iterates are bitwise those of the oracle.
#include <type_traits>

#include "hoc_device.h"
#include "hoc_kernels.h"
#include "hoc_reduce.h"

namespace hoc {

template <class R>
__device__ __forceinline__ void lvl_ij(const MgLevelT<R>& L, long long c, int& i, int& j) {
  j = (int)((unsigned)c / (unsigned)L.nx);  // a level has fewer than 2^31 cells
  i = (int)((unsigned)c - (unsigned)j * (unsigned)L.nx);
}

template <class R>
__device__ __forceinline__ R mkr(uint8_t m) {
  return m ? R(1) : R(0);
}

// A x at c from the values at c and its four neighbours, x masked first
// (solvers_var.py:47-53); ce/cw/cn/cs are the neighbours' indices. In the
// level's type R throughout (for R = double the reference's arithmetic).
// The same from the operands themselves: the faces' Ku[c], Ku[cw], Kv[c],
// Kv[cs] and the five cells' masks (as 0/1 values of R).
template <class R>
__device__ __forceinline__ R apply_from(R coef, R dx2, R dy2, R ku_c, R ku_w, R kv_c, R kv_s,
                                        R mc, R me, R mw, R mn, R ms, R x0, R x_e, R x_w, R x_n,
                                        R x_s) {
  const R xc = x0 * mc;
  const R xe = x_e * me;
  const R xw = x_w * mw;
  const R xn = x_n * mn;
  const R xs = x_s * ms;
  const R fx = ku_c * (xe - xc);
  const R fxw = ku_w * (xc - xw);
  const R fy = kv_c * (xn - xc);
  const R fys = kv_s * (xc - xs);
  const R lap = (fx - fxw) / dx2 + (fy - fys) / dy2;
  return (xc - coef * lap) * mc + xc * (R(1) - mc);
}

template <class R>
__device__ __forceinline__ R apply_vals(const MgLevelT<R>& L, long long c, long long ce,
                                        long long cw, long long cn, long long cs, R x0, R x_e,
                                        R x_w, R x_n, R x_s) {
  return apply_from<R>(L.coef, L.dx2, L.dy2, L.Ku[c], L.Ku[cw], L.Kv[c], L.Kv[cs],
                       mkr<R>(L.mask[c]), mkr<R>(L.mask[ce]), mkr<R>(L.mask[cw]),
                       mkr<R>(L.mask[cn]), mkr<R>(L.mask[cs]), x0, x_e, x_w, x_n, x_s);
}

// Red-black Gauss-Seidel update at c: inv_diag (b + neighbour_sum(x)), the
// neighbours' values unmasked (solvers_var.py:55-69), in the operand order
// of mg_neighbour_sum.
template <class R>
__device__ __forceinline__ R rbgs_from(R inv, R b, R cx, R cy, R ku_c, R ku_w, R kv_c, R kv_s,
                                       R x_e, R x_w, R x_n, R x_s) {
  return inv * (b + (cx * (ku_c * x_e + ku_w * x_w) + cy * (kv_c * x_n + kv_s * x_s)));
}

struct Nbr {
  long long c, ce, cw, cn, cs;
};

template <class R>
__device__ __forceinline__ Nbr nbr_of(const MgLevelT<R>& L, int i, int j) {
  const long long row = (long long)j * L.nx;
  return Nbr{row + i, row + wrap(i, 1, L.nx), row + wrap(i, -1, L.nx),
             (long long)wrap(j, 1, L.ny) * L.nx + i, (long long)wrap(j, -1, L.ny) * L.nx + i};
}

__device__ __forceinline__ double mg_apply(const MgLevel& L, const double* x, long long c) {
  int i, j;
  lvl_ij(L, c, i, j);
  const Nbr n = nbr_of(L, i, j);
  return apply_vals(L, c, n.ce, n.cw, n.cn, n.cs, x[c], x[n.ce], x[n.cw], x[n.cn], x[n.cs]);
}

// -(A - diag) x, unmasked x (solvers_var.py:55-60).
__device__ __forceinline__ double mg_neighbour_sum(const MgLevel& L, const double* x, long long c) {
  int i, j;
  lvl_ij(L, c, i, j);
  const long long ce = (long long)j * L.nx + wrap(i, 1, L.nx);
  const long long cw = (long long)j * L.nx + wrap(i, -1, L.nx);
  const long long cn = (long long)wrap(j, 1, L.ny) * L.nx + i;
  const long long cs = (long long)wrap(j, -1, L.ny) * L.nx + i;
  return L.cx * (L.Ku[c] * x[ce] + L.Ku[cw] * x[cw]) +
         L.cy * (L.Kv[c] * x[cn] + L.Kv[cs] * x[cs]);
}

__device__ __forceinline__ int mg_pmod(int a, int n) {
  const int r = a % n;
  return r < 0 ? r + n : r;
}

__device__ __forceinline__ bool finished(const PcgScalars* sc) { return sc && sc->done; }

// Coarse faces: mean of the two fine faces on the coarse cell's east
// (north) edge; coarse cell wet if any child is (solvers_var.py:118-127).
__global__ void k_mg_coarsen(MgLevel f, MgLevel c, double* __restrict__ cKu,
                             double* __restrict__ cKv, uint8_t* __restrict__ cm) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= c.n) return;
  const int I = (int)(t % c.nx), J = (int)(t / c.nx);
  const long long f00 = (long long)(2 * J) * f.nx + 2 * I;
  const long long f01 = f00 + 1, f10 = f00 + f.nx, f11 = f10 + 1;
  cKu[t] = 0.5 * (f.Ku[f01] + f.Ku[f11]);
  cKv[t] = 0.5 * (f.Kv[f10] + f.Kv[f11]);
  uint8_t m = f.mask[f00];
  m = f.mask[f01] > m ? f.mask[f01] : m;
  m = f.mask[f10] > m ? f.mask[f10] : m;
  m = f.mask[f11] > m ? f.mask[f11] : m;
  cm[t] = m;
}

__global__ void k_mg_diag(MgLevel L, double* __restrict__ inv_diag) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= L.n) return;
  int i, j;
  lvl_ij(L, c, i, j);
  const long long cw = (long long)j * L.nx + wrap(i, -1, L.nx);
  const long long cs = (long long)wrap(j, -1, L.ny) * L.nx + i;
  double dg = 1.0 + L.cx * (L.Ku[c] + L.Ku[cw]) + L.cy * (L.Kv[c] + L.Kv[cs]);
  dg = L.mask[c] ? dg : 1.0;
  inv_diag[c] = 1.0 / dg;
}

// The face coefficient of a level `depth` levels below the fine one: the
// fine faces v[0], v[stride], ..., v[(2^depth - 1) stride] along the coarse
// cell's edge, averaged pairwise as k_mg_coarsen's recursion does, level by
// level (0.5 (left + right) at each node of the balanced tree).
__device__ __forceinline__ double mean_tree(const double* __restrict__ v, long long stride,
                                            int depth) {
  double st[MG_BUILD_LEVELS];
  const int len = 1 << depth;
  for (int q = 0; q < len; ++q) {
    double x = v[(long long)q * stride];
    int lv = 0;
    for (int qq = q; qq & 1; qq >>= 1) x = 0.5 * (st[lv++] + x);
    st[lv] = x;
  }
  return st[depth];
}

// The same tree for a depth known at compile time: every load issued at
// once, then the combine levels.
template <int D>
__device__ __forceinline__ double mean_tree_d(const double* __restrict__ v, long long stride) {
  constexpr int N = 1 << D;
  double x[N];
#pragma unroll
  for (int q = 0; q < N; ++q) x[q] = v[(long long)q * stride];
#pragma unroll
  for (int w = N; w > 1; w >>= 1)
#pragma unroll
    for (int q = 0; q < w / 2; ++q) x[q] = 0.5 * (x[2 * q] + x[2 * q + 1]);
  return x[0];
}

__device__ __forceinline__ double mean_tree_any(const double* __restrict__ v, long long stride,
                                                int depth) {
  switch (depth) {
    case 1: return mean_tree_d<1>(v, stride);
    case 2: return mean_tree_d<2>(v, stride);
    case 3: return mean_tree_d<3>(v, stride);
    case 4: return mean_tree_d<4>(v, stride);
    case 5: return mean_tree_d<5>(v, stride);
    default: return mean_tree(v, stride, depth);
  }
}

// Level l's Ku at (J, I) is the tree over the level-0 Ku of column
// (I + 1) 2^l - 1, rows J 2^l .. (J + 1) 2^l - 1; its Kv the tree over the
// level-0 Kv of row (J + 1) 2^l - 1, columns I 2^l .. (I + 1) 2^l - 1. Every
// level halves even sides, so level 0 is exactly 2^l times as wide.
__global__ void k_mg_levels(MgBuildArgs A) {
  const int l = (int)blockIdx.y + A.l_first;
  if (l >= A.nlev) return;
  const MgLevel& L = A.lev[l];
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= L.n) return;
  if (l == 0) {
    A.fKu[0][t] = (float)L.Ku[t];
    A.fKv[0][t] = (float)L.Kv[t];
    A.finv[0][t] = (float)L.inv_diag[t];
    return;
  }
  const MgLevel& F = A.lev[0];
  const int I = (int)(t % L.nx), J = (int)(t / L.nx);
  const long long span = 1ll << l;
  auto ku_at = [&](int jj, int ii) {
    return mean_tree_any(F.Ku + jj * span * F.nx + (ii + 1) * span - 1, F.nx, l);
  };
  auto kv_at = [&](int jj, int ii) {
    return mean_tree_any(F.Kv + ((jj + 1) * span - 1) * F.nx + ii * span, 1, l);
  };
  const double ku = ku_at(J, I), kv = kv_at(J, I);
  const double kuw = ku_at(J, wrap(I, -1, L.nx)), kvs = kv_at(wrap(J, -1, L.ny), I);
  double dg = 1.0 + L.cx * (ku + kuw) + L.cy * (kv + kvs);
  dg = L.mask[t] ? dg : 1.0;
  const double inv = 1.0 / dg;
  A.Ku[l][t] = ku;
  A.Kv[l][t] = kv;
  A.inv[l][t] = inv;
  if (A.fKu[l]) {
    A.fKu[l][t] = (float)ku;
    A.fKv[l][t] = (float)kv;
    A.finv[l][t] = (float)inv;
  }
}

__global__ void k_mg_zero(long long n, double* __restrict__ x, const PcgScalars* sc) {
  if (finished(sc)) return;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) x[c] = 0.0;
}

// One colour of a red-black Gauss-Seidel sweep, out of place: the colour's
// cells take inv_diag (b + neighbour_sum(xin)), the others keep xin. The
// second colour of a sweep (last = 1) masks the whole field, as the
// reference does after both colours (solvers_var.py:63-69). Out of place
// because a periodic level with an odd side has same-colour neighbours
// across the wrap, whose old values the reference reads.
__global__ void k_mg_rbgs(MgLevel L, int colour, int last, const double* __restrict__ b,
                          const double* __restrict__ xin, double* __restrict__ xout,
                          const PcgScalars* sc) {
  if (finished(sc)) return;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= L.n) return;
  int i, j;
  lvl_ij(L, c, i, j);
  const double v = (((i + j) & 1) == colour) ? L.inv_diag[c] * (b[c] + mg_neighbour_sum(L, xin, c))
                                             : xin[c];
  xout[c] = last ? v * mk(L.mask[c]) : v;
}

// One whole red-black sweep (first colour c0, then the other) in one launch,
// xout = sweep(xin) masked, exactly as the two launches of k_mg_rbgs compute
// it: a RB_TW x RB_TH tile stages the old field with a two-cell halo in LDS,
// computes the first colour on the tile and a one-cell halo from it (the
// other colour keeps its old value there), then the second colour on the
// tile from those values.
// Every first-colour update reads the old field only and every second-colour
// update reads first-colour values and old second-colour values, so odd
// periodic sides (where same-coloured cells meet) keep the whole-array
// semantics. Halo positions wrap; on sides shorter than the tile they alias
// cells of the tile and hold the same values.
__global__ __launch_bounds__(RB_TW * RB_TH) void k_mg_rbgs2(MgLevel L, int c0,
                                                            const double* __restrict__ b,
                                                            const double* __restrict__ xin,
                                                            double* __restrict__ xout,
                                                            const PcgScalars* sc) {
  if (finished(sc)) return;
  constexpr int SW = RB_TW + 2, SH = RB_TH + 2;   // first-colour region: tile + 1
  constexpr int XW = RB_TW + 4, XH = RB_TH + 4;   // old field: tile + 2
  __shared__ double xs[XH][XW];
  __shared__ double v1[SH][SW];
  const int tid = threadIdx.x;
  const int i0 = blockIdx.x * RB_TW, j0 = blockIdx.y * RB_TH;
  for (int q = tid; q < XW * XH; q += RB_TW * RB_TH) {
    const int ly = q / XW, lx = q % XW;
    xs[ly][lx] = xin[(long long)mg_pmod(j0 + ly - 2, L.ny) * L.nx + mg_pmod(i0 + lx - 2, L.nx)];
  }
  __syncthreads();
  for (int q = tid; q < SW * SH; q += RB_TW * RB_TH) {
    const int ly = q / SW, lx = q % SW;
    const int i = mg_pmod(i0 + lx - 1, L.nx), j = mg_pmod(j0 + ly - 1, L.ny);
    const long long g = (long long)j * L.nx + i;
    if (((i + j) & 1) == c0) {
      const long long cw = (long long)j * L.nx + wrap(i, -1, L.nx);
      const long long cs = (long long)wrap(j, -1, L.ny) * L.nx + i;
      const double nb = L.cx * (L.Ku[g] * xs[ly + 1][lx + 2] + L.Ku[cw] * xs[ly + 1][lx]) +
                        L.cy * (L.Kv[g] * xs[ly + 2][lx + 1] + L.Kv[cs] * xs[ly][lx + 1]);
      v1[ly][lx] = L.inv_diag[g] * (b[g] + nb);
    } else {
      v1[ly][lx] = xs[ly + 1][lx + 1];
    }
  }
  __syncthreads();
  const int tx = tid % RB_TW, ty = tid / RB_TW;
  const int i = i0 + tx, j = j0 + ty;
  if (i >= L.nx || j >= L.ny) return;
  const long long c = (long long)j * L.nx + i;
  double v;
  if (((i + j) & 1) != c0) {
    const long long cw = (long long)j * L.nx + wrap(i, -1, L.nx);
    const long long cs = (long long)wrap(j, -1, L.ny) * L.nx + i;
    const double nb = L.cx * (L.Ku[c] * v1[ty + 1][tx + 2] + L.Ku[cw] * v1[ty + 1][tx]) +
                      L.cy * (L.Kv[c] * v1[ty + 2][tx + 1] + L.Kv[cs] * v1[ty][tx + 1]);
    v = L.inv_diag[c] * (b[c] + nb);
  } else {
    v = v1[ty + 1][tx + 1];
  }
  xout[c] = v * mk(L.mask[c]);
}

// Damped Jacobi: xo = x + omega (inv_diag (b - A x)) mask.
__global__ void k_mg_jacobi(MgLevel L, double omega, const double* __restrict__ x,
                            const double* __restrict__ b, double* __restrict__ xo,
                            const PcgScalars* sc) {
  if (finished(sc)) return;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= L.n) return;
  xo[c] = x[c] + omega * (L.inv_diag[c] * (b[c] - mg_apply(L, x, c))) * mk(L.mask[c]);
}

// bc = restrict((b - A x) mask), 1/4 of the 2 x 2 children in the order
// [0::2,0::2] + [0::2,1::2] + [1::2,0::2] + [1::2,1::2].
__global__ void k_mg_residual_restrict(MgLevel f, MgLevel c, const double* __restrict__ x,
                                       const double* __restrict__ b, double* __restrict__ bc,
                                       double* __restrict__ xc_zero, const PcgScalars* sc) {
  if (finished(sc)) return;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= c.n) return;
  const int I = (int)(t % c.nx), J = (int)(t / c.nx);
  const long long f00 = (long long)(2 * J) * f.nx + 2 * I;
  const long long ch[4] = {f00, f00 + 1, f00 + f.nx, f00 + f.nx + 1};
  double r[4];
  for (int q = 0; q < 4; ++q) r[q] = (b[ch[q]] - mg_apply(f, x, ch[q])) * mk(f.mask[ch[q]]);
  bc[t] = 0.25 * (r[0] + r[1] + r[2] + r[3]);
  if (xc_zero) xc_zero[t] = 0.0;  // the coarse correction's zero start, when asked
}

// x += prolong(xc) * mask (piecewise constant).
__global__ void k_mg_prolong(MgLevel f, const double* __restrict__ xc, int cnx,
                             double* __restrict__ x, const PcgScalars* sc) {
  if (finished(sc)) return;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= f.n) return;
  int i, j;
  lvl_ij(f, t, i, j);
  x[t] = x[t] + xc[(long long)(j / 2) * cnx + i / 2] * mk(f.mask[t]);
}

// Partial sums of (rhs - A x)^2 per part (residual norm of the stationary
// solvers, solvers_var.py:176).
__global__ __launch_bounds__(PCG_WG) void k_mg_res_parts(PcgArgs a, MgLevel L,
                                                         const double* __restrict__ x) {
  const int done = a.sc->done;
  __shared__ double lds[PCG_STAGE];
  const int part = blockIdx.x;
  const double s = part_sum(a, part, [&](long long e) -> double {
    const double r = a.rhs[e] - mg_apply(L, x, e);
    return r * r;
  }, lds);
  if (threadIdx.x == 0 && !done) a.part_b[part] = s;
}

// Stationary-solver bookkeeping after iteration `it`: ||rhs - A x|| <= tol.
__global__ __launch_bounds__(PCG_WG) void k_mg_check(PcgArgs a, int it) {
  const int done = a.sc->done;
  __shared__ double cs[PCG_CS];
  const double res = sqrt(total_from_parts(a, a.part_b, cs));
  if (threadIdx.x != 0 || done) return;
  PcgScalars* sc = a.sc;
  sc->res = res;
  if (res <= sc->tol) {
    sc->done = 1;
    sc->converged = 1;
    sc->iters = it;
    a.counters[0] += it;
  } else if (it >= a.max_iter) {
    sc->done = 1;
    sc->converged = 0;
    sc->iters = a.max_iter;
    a.counters[0] += a.max_iter;
    a.counters[1] += 1;
  }
}

// ||rhs|| and the zero-rhs shortcut for the stationary solvers; x = 0.
__global__ __launch_bounds__(PCG_WG) void k_mg_start(PcgArgs a) {
  __shared__ double cs[PCG_CS];
  const double nb = sqrt(total_from_parts(a, a.part_a, cs));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.sc->norm_b = nb;
    a.sc->tol = a.rtol * nb;
    a.sc->iters = 0;
    a.sc->converged = 1;
    a.sc->done = (nb == 0.0) ? 1 : 0;
    a.sc->res = 0.0;
  }
}

// x wrapped into [0, n) for x in [-H, n + TW + H).
template <int H, int TW>
__device__ __forceinline__ int tile_wrap(int x, int n) {
  if (n >= TW + H) {  // one period either way (the same for every thread)
    if (x < 0) x += n;
    return x >= n ? x - n : x;
  }
  return mg_pmod(x, n);
}

// ------------------------------ fused pcg_mg V-cycle legs, damped Jacobi
// The pcg_mg preconditioner with S damped-Jacobi sweeps per side, as LDS
// tiles of TW x TH fine cells plus the halo the later steps still need
// (radius 1 per remaining step, neighbours wrapping like the operator), so one
// launch replaces the zero / S sweeps / residual-restrict launches of the way
// down and the prolong / S sweeps launches of the way up, with the same
// arithmetic per cell. A thread owns its cells (one; two for the largest tile)
// for the whole leg, coefficients, right-hand side and value in registers, and
// a sweep reads only the four neighbours' values from LDS; from zero the first
// sweep reads none, so the way down needs no halo for it. R is the arithmetic
// and storage type of the level's vectors; RB the type of the right-hand side
// read (double on level 0 of the fp32 cycle, where it is the fp64 PCG
// residual), RO the type of the way-up result (double on level 0 of the fp32
// cycle).
// Bound: latency, that of the loads before the first sweep and of one barrier,
// four LDS reads and five dependent operations per sweep; with the region
// walked in several rounds by 256 threads, coefficients re-read and divisions
// by the spacings, a leg down and up took 5.5 and 4.5 us on average under
// 128 x 128 and 6.0 and 5.6 us in fp32 under 640 x 512; so it is 3.7 and 3.7,
// 3.7 and 3.6 us. A level can be smaller than a tile and its halo: positions
// wrap round it as often as needed.
// The cells of a TW x TH tile with a halo of H: Q per thread.
template <int H, int TW, int TH>
struct JacRegion {
  static constexpr int RW = TW + 2 * H, RH = TH + 2 * H, RN = RW * RH;
  static constexpr int Q = (RN + 1023) / 1024;
  static constexpr int NT = ((RN + Q - 1) / Q + 63) / 64 * 64;
};

// One cell of a thread: its coefficients, right-hand side, 1/diag and mask,
// the LDS positions of its neighbours and of itself, its index on the level
// and its place in the tile. A cell's neighbours beyond the region are itself
// (a value that no valid cell uses).
template <class R>
struct JacCell {
  R inv, b, ke, kw, kn, ks, m;
  int q, e, w, n, s, g, up, ti, tj;
};

template <class R, class RB, int H, int TW, int TH>
__device__ __forceinline__ JacCell<R> jac_cell(const MgLevelT<R>& L, const RB* __restrict__ b,
                                               int i0, int j0, int t) {
  using Rg = JacRegion<H, TW, TH>;
  const int lj = t / Rg::RW, li = t % Rg::RW;
  const int ui = i0 - H + li, uj = j0 - H + lj;
  const int i = tile_wrap<H, TW>(ui, L.nx), iw = tile_wrap<H + 1, TW>(ui - 1, L.nx);
  const int j = tile_wrap<H, TH>(uj, L.ny), js = tile_wrap<H + 1, TH>(uj - 1, L.ny);
  JacCell<R> K;
  K.g = j * L.nx + i;
  K.inv = L.inv_diag[K.g];
  K.b = (R)b[K.g];
  K.ke = L.Ku[K.g];
  K.kw = L.Ku[j * L.nx + iw];
  K.kn = L.Kv[K.g];
  K.ks = L.Kv[js * L.nx + i];
  K.m = mkr<R>(L.mask[K.g]);
  K.q = t;
  K.e = li + 1 < Rg::RW ? t + 1 : t;
  K.w = li > 0 ? t - 1 : t;
  K.n = lj + 1 < Rg::RH ? t + Rg::RW : t;
  K.s = lj > 0 ? t - Rg::RW : t;
  K.up = (j / 2) * (L.nx / 2) + i / 2;
  K.ti = li - H;
  K.tj = lj - H;
  return K;
}

// A x at a cell in apply_from's order; the values are masked already, so its
// multiplications by the masks are exact no-ops.
template <class R>
__device__ __forceinline__ R jac_apply(const JacCell<R>& K, R coef, const Divisor<R>& by_dx2,
                                       const Divisor<R>& by_dy2, R xc, R xe, R xw, R xn, R xs) {
  const R lap = by_dx2(K.ke * (xe - xc) - K.kw * (xc - xw)) +
                by_dy2(K.kn * (xn - xc) - K.ks * (xc - xs));
  return (xc - coef * lap) * K.m + xc * (R(1) - K.m);
}

// Way down on one level: x_S = S sweeps from zero (written out for the way
// up) and bc = restrict((b - A x_S) mask).
template <int S, class R, class RB, int TW, int TH>
__global__ __launch_bounds__((JacRegion<S, TW, TH>::NT)) void k_mg_down(
    MgLevelT<R> L, MgLevelT<R> C, R omega, const RB* __restrict__ b, R* __restrict__ xs_out,
    R* __restrict__ bc, const PcgScalars* sc) {
  const bool done = finished(sc);  // tested once the loads are on their way
  constexpr int H = S;
  using Rg = JacRegion<H, TW, TH>;
  constexpr int Q = Rg::Q;
  __shared__ R buf[2][Rg::RN];
  const int i0 = blockIdx.x * TW, j0 = blockIdx.y * TH;
  const Divisor<R> by_dx2 = uniform_divisor<R>(L.dx2), by_dy2 = uniform_divisor<R>(L.dy2);
  JacCell<R> K[Q];
  R v[Q];
  bool on[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int t = threadIdx.x + q * Rg::NT;
    on[q] = t < Rg::RN;
    K[q] = jac_cell<R, RB, H, TW, TH>(L, b, i0, j0, on[q] ? t : 0);
    v[q] = R(0);
  }
#pragma unroll
  for (int k = 1; k <= S; ++k) {
    const R* src = buf[k & 1];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const R z = R(0);
      const R ax = k == 1 ? jac_apply(K[q], L.coef, by_dx2, by_dy2, z, z, z, z, z)
                          : jac_apply(K[q], L.coef, by_dx2, by_dy2, v[q], src[K[q].e],
                                      src[K[q].w], src[K[q].n], src[K[q].s]);
      v[q] = v[q] + omega * (K[q].inv * (K[q].b - ax)) * K[q].m;
      if (on[q]) buf[(k - 1) & 1][K[q].q] = v[q];
    }
    __syncthreads();
    if (k == 1 && done) return;
  }
  const R* xs = buf[(S - 1) & 1];
  R* res = buf[S & 1];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (!on[q] || K[q].ti < 0 || K[q].ti >= TW || K[q].tj < 0 || K[q].tj >= TH) continue;
    if (i0 + K[q].ti < L.nx && j0 + K[q].tj < L.ny) xs_out[K[q].g] = v[q];
    const R ax = jac_apply(K[q], L.coef, by_dx2, by_dy2, v[q], xs[K[q].e], xs[K[q].w],
                           xs[K[q].n], xs[K[q].s]);
    res[K[q].q] = (K[q].b - ax) * K[q].m;
  }
  __syncthreads();
  constexpr int CW = TW / 2, CH = TH / 2;
  for (int u = threadIdx.x; u < CW * CH; u += Rg::NT) {
    const int I = i0 / 2 + u % CW, J = j0 / 2 + u / CW;
    if (I >= C.nx || J >= C.ny) continue;
    const int q = (H + 2 * (u / CW)) * Rg::RW + H + 2 * (u % CW);
    bc[(long long)J * C.nx + I] =
        R(0.25) * (res[q] + res[q + 1] + res[q + Rg::RW] + res[q + Rg::RW + 1]);
  }
}

// Way up on one level: x = x_S + prolong(ec) mask, then S sweeps; out = x.
template <int S, class R, class RB, class RO, int TW, int TH>
__global__ __launch_bounds__((JacRegion<S, TW, TH>::NT)) void k_mg_up(
    MgLevelT<R> L, R omega, const R* __restrict__ xs_in, const R* __restrict__ ec,
    const RB* __restrict__ b, RO* __restrict__ out, const PcgScalars* sc) {
  const bool done = finished(sc);  // tested once the loads are on their way
  constexpr int H = S;
  using Rg = JacRegion<H, TW, TH>;
  constexpr int Q = Rg::Q;
  __shared__ R buf[2][Rg::RN];
  const int i0 = blockIdx.x * TW, j0 = blockIdx.y * TH;
  const Divisor<R> by_dx2 = uniform_divisor<R>(L.dx2), by_dy2 = uniform_divisor<R>(L.dy2);
  JacCell<R> K[Q];
  R v[Q];
  bool on[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int t = threadIdx.x + q * Rg::NT;
    on[q] = t < Rg::RN;
    K[q] = jac_cell<R, RB, H, TW, TH>(L, b, i0, j0, on[q] ? t : 0);
    v[q] = xs_in[K[q].g] + ec[K[q].up] * K[q].m;
    if (on[q]) buf[0][K[q].q] = v[q];
  }
  __syncthreads();
  if (done) return;
#pragma unroll
  for (int k = 1; k <= S; ++k) {
    const R* src = buf[(k - 1) & 1];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const R ax = jac_apply(K[q], L.coef, by_dx2, by_dy2, v[q], src[K[q].e], src[K[q].w],
                             src[K[q].n], src[K[q].s]);
      v[q] = v[q] + omega * (K[q].inv * (K[q].b - ax)) * K[q].m;
      if (k < S && on[q]) buf[k & 1][K[q].q] = v[q];
    }
    if (k < S) __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (!on[q] || K[q].ti < 0 || K[q].ti >= TW || K[q].tj < 0 || K[q].tj >= TH) continue;
    if (i0 + K[q].ti < L.nx && j0 + K[q].tj < L.ny) out[K[q].g] = (RO)v[q];
  }
}

// ---------------------------------- fused V-cycle legs, red-black smoother
// The legs of a V-cycle whose smoother is red-black Gauss-Seidel: S sweeps
// red-black on the way down and S sweeps black-red on the way up, each
// half-sweep evaluated on the tile plus the halo that the later ones still
// need, so a leg is one launch with the arithmetic of k_mg_rbgs per cell.
// These legs run on the levels above the coarse cycle, which are all
// coarsened and so have even sides: a cell's colour is then the parity of its
// unwrapped coordinates.
//
// Bound by the latency of one chain (launch, loads, 2S half-sweeps with a
// barrier each, residual, stores), not by work. So one thread owns one pair
// of neighbouring cells along x, one of each colour, for the whole leg: both
// cells' coefficients, right-hand sides and values stay in its registers, and
// a half-sweep reads only the updated cell's three other neighbours from LDS.
// Against both colours walked in rounds by 256 threads, a leg down and up fell
// from 5.1 and 4.9 us to 4.3 and 4.2 on average under 128 x 128 (16 x 16
// tiles) and from 6.1 and 5.7 to 5.2 and 5.1 under 512 x 512. The stationary
// multigrid's level-0 sweeps start from x_in with one more cell of halo; in
// legs its cycle on 400 x 400 takes 4 launches fewer per level, and a solve
// 0.49 instead of 1.28 ms.
// One cell of a thread's pair: its coefficients towards the horizontal
// neighbour outside the pair and to the north and south, its right-hand
// side, 1/diag and mask, the LDS positions of those neighbours and of itself.
struct RbCell {
  double inv, b, kh, kn, ks, m;
  int h, n, s, q;
};

// The pairs of a TW x TH tile with a halo of H cells: one thread each.
template <int H, int TW, int TH>
struct RbRegion {
  static constexpr int RW = TW + 2 * H, RH = TH + 2 * H, RN = RW * RH, PW = RW / 2;
  static constexpr int PAIRS = PW * RH, NT = (PAIRS + 63) / 64 * 64;
  static_assert(NT <= 1024, "one thread per pair");
};

// This thread's pair: [0] the red cell, [1] the black one; kp is the face
// between them, g the cells' indices on the level, (gi, gj) the first cell's
// unwrapped position.
struct RbPair {
  RbCell c[2];
  double kp, x[2];
  int g[2], up[2];  // indices on the level and, of the cell holding it, on the coarser one
  int ti[2], tj;    // columns and row in the tile
};

template <int H, int TW, int TH>
__device__ __forceinline__ RbPair rb_pair(const MgLevel& L, const double* __restrict__ b, int i0,
                                          int j0, int t) {
  using Rg = RbRegion<H, TW, TH>;
  const int lj = t / Rg::PW, li = 2 * (t % Rg::PW);
  const int ui = i0 - H + li, uj = j0 - H + lj;
  const int ia = tile_wrap<H, TW>(ui, L.nx), ib = tile_wrap<H, TW>(ui + 1, L.nx);
  const int iw = tile_wrap<H + 1, TW>(ui - 1, L.nx);
  const int jj = tile_wrap<H, TH>(uj, L.ny), js = tile_wrap<H + 1, TH>(uj - 1, L.ny);
  const int row = jj * L.nx, rs = js * L.nx;
  const int ga = row + ia, gb = row + ib;
  const int q = lj * Rg::RW + li;
  const int qn = lj + 1 < Rg::RH ? Rg::RW : 0, qs = lj > 0 ? Rg::RW : 0;
  RbCell A, B;
  A.inv = L.inv_diag[ga];
  B.inv = L.inv_diag[gb];
  A.b = b[ga];
  B.b = b[gb];
  A.kh = L.Ku[row + iw];
  B.kh = L.Ku[gb];
  A.kn = L.Kv[ga];
  B.kn = L.Kv[gb];
  A.ks = L.Kv[rs + ia];
  B.ks = L.Kv[rs + ib];
  A.m = mkr<double>(L.mask[ga]);
  B.m = mkr<double>(L.mask[gb]);
  RbPair P;
  P.kp = L.Ku[ga];
  A.q = q;
  A.h = li > 0 ? q - 1 : q;  // beyond the region: a value that no valid cell uses
  A.n = q + qn;
  A.s = q - qs;
  B.q = q + 1;
  B.h = li + 2 < Rg::RW ? q + 2 : q + 1;
  B.n = q + 1 + qn;
  B.s = q + 1 - qs;
  const bool black_first = ((ui + uj) & 1) != 0;
  P.c[0] = black_first ? B : A;
  P.c[1] = black_first ? A : B;
  P.g[0] = black_first ? gb : ga;
  P.g[1] = black_first ? ga : gb;
  const int ur = (jj / 2) * (L.nx / 2);
  P.up[0] = ur + (black_first ? ib : ia) / 2;
  P.up[1] = ur + (black_first ? ia : ib) / 2;
  P.ti[0] = li - H + (black_first ? 1 : 0);
  P.ti[1] = li - H + (black_first ? 0 : 1);
  P.tj = lj - H;
  P.x[0] = P.x[1] = 0.0;
  return P;
}

// One half-sweep of colour `col` from the neighbours in src; the wet mask
// over both cells after the sweep's second colour (mask_all).
__device__ __forceinline__ void rb_update(RbPair& P, double cx, double cy, int col, bool mask_all,
                                          const double* src) {
  const RbCell& c = P.c[col];
  P.x[col] = rbgs_from<double>(c.inv, c.b, cx, cy, P.kp, c.kh, c.kn, c.ks, P.x[1 - col],
                               src[c.h], src[c.n], src[c.s]);
  if (mask_all) {
    P.x[0] = P.x[0] * P.c[0].m;
    P.x[1] = P.x[1] * P.c[1].m;
  }
}

__device__ __forceinline__ void rb_put(const RbPair& P, double* dst) {
  dst[P.c[0].q] = P.x[0];
  dst[P.c[1].q] = P.x[1];
}

// Way down: x_S = S sweeps (from zero, or from x_in with FROM_X: level 0 of
// the stationary multigrid) written out for the way up, and
// bc = restrict((b - A x_S) mask). From zero the first half-sweep reads no
// neighbour, so the halo is one cell narrower.
template <int S, bool FROM_X, int TW, int TH>
__global__ __launch_bounds__((RbRegion<2 * S + (FROM_X ? 1 : 0), TW, TH>::NT)) void k_mg_down_rb(
    MgLevel L, MgLevel C, const double* __restrict__ x_in, const double* __restrict__ b,
    double* __restrict__ xs_out, double* __restrict__ bc, const PcgScalars* sc) {
  const bool done = finished(sc);  // tested once the loads are on their way
  constexpr int H = 2 * S + (FROM_X ? 1 : 0);
  using Rg = RbRegion<H, TW, TH>;
  __shared__ double buf[2][Rg::RN];
  const int i0 = blockIdx.x * TW, j0 = blockIdx.y * TH;
  const int t = threadIdx.x;
  const bool on = t < Rg::PAIRS;
  RbPair P = rb_pair<H, TW, TH>(L, b, i0, j0, on ? t : 0);
  if (FROM_X) {
    P.x[0] = x_in[P.g[0]];
    P.x[1] = x_in[P.g[1]];
    if (on) rb_put(P, buf[0]);
    __syncthreads();
    rb_update(P, L.cx, L.cy, 0, false, buf[0]);
  } else {
    const RbCell& c = P.c[0];
    P.x[0] = rbgs_from<double>(c.inv, c.b, L.cx, L.cy, P.kp, c.kh, c.kn, c.ks, 0.0, 0.0, 0.0,
                               0.0);
  }
  if (on) rb_put(P, buf[1]);
  __syncthreads();
  if (done) return;
#pragma unroll
  for (int ph = 2; ph <= 2 * S; ++ph) {  // red first
    rb_update(P, L.cx, L.cy, (ph - 1) & 1, (ph & 1) == 0, buf[(ph - 1) & 1]);
    if (on) rb_put(P, buf[ph & 1]);
    __syncthreads();
  }
  const double* xs = buf[0];  // 2S half-sweeps end in buf[0]
  double* res = buf[1];
  const Divisor<double> by_dx2 = uniform_divisor<double>(L.dx2),
                        by_dy2 = uniform_divisor<double>(L.dy2);
  if (on) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const RbCell& c = P.c[k];
      if (P.ti[k] < 0 || P.ti[k] >= TW || P.tj < 0 || P.tj >= TH) continue;
      if (i0 + P.ti[k] < L.nx && j0 + P.tj < L.ny) xs_out[P.g[k]] = P.x[k];
      // the residual in apply_from's order; the values are masked already
      // (x m m = x m for a 0/1 mask). The pair's cell to the east is the
      // other one for the western cell, and the sums of two commute.
      const double xc = P.x[k], xp = P.x[1 - k], xh = xs[c.h], xn = xs[c.n], xsv = xs[c.s];
      const bool west = P.ti[k] < P.ti[1 - k];
      const double fe = west ? P.kp * (xp - xc) : c.kh * (xh - xc);
      const double fw = west ? c.kh * (xc - xh) : P.kp * (xc - xp);
      const double fn = c.kn * (xn - xc), fs = c.ks * (xc - xsv);
      const double lap = by_dx2(fe - fw) + by_dy2(fn - fs);
      const double ax = (xc - L.coef * lap) * c.m + xc * (1.0 - c.m);
      res[c.q] = (c.b - ax) * c.m;
    }
  }
  __syncthreads();
  constexpr int CW = TW / 2, CH = TH / 2;
  for (int u = t; u < CW * CH; u += Rg::NT) {
    const int I = i0 / 2 + u % CW, J = j0 / 2 + u / CW;
    if (I >= C.nx || J >= C.ny) continue;
    const int q = (H + 2 * (u / CW)) * Rg::RW + H + 2 * (u % CW);
    bc[(long long)J * C.nx + I] =
        0.25 * (res[q] + res[q + 1] + res[q + Rg::RW] + res[q + Rg::RW + 1]);
  }
}

// Way up: x = x_S + prolong(ec) mask, then S reversed sweeps; out = x.
template <int S, int TW, int TH>
__global__ __launch_bounds__((RbRegion<2 * S, TW, TH>::NT)) void k_mg_up_rb(
    MgLevel L, const double* __restrict__ xs_in, const double* __restrict__ ec,
    const double* __restrict__ b, double* __restrict__ out, const PcgScalars* sc) {
  const bool done = finished(sc);  // tested once the loads are on their way
  constexpr int H = 2 * S;
  using Rg = RbRegion<H, TW, TH>;
  __shared__ double buf[2][Rg::RN];
  const int i0 = blockIdx.x * TW, j0 = blockIdx.y * TH;
  const int t = threadIdx.x;
  const bool on = t < Rg::PAIRS;
  RbPair P = rb_pair<H, TW, TH>(L, b, i0, j0, on ? t : 0);
#pragma unroll
  for (int k = 0; k < 2; ++k) P.x[k] = xs_in[P.g[k]] + ec[P.up[k]] * P.c[k].m;
  if (on) rb_put(P, buf[0]);
  __syncthreads();
  if (done) return;
#pragma unroll
  for (int ph = 1; ph <= 2 * S; ++ph) {  // black first
    rb_update(P, L.cx, L.cy, ph & 1, (ph & 1) == 0, buf[(ph - 1) & 1]);
    if (ph == 2 * S) break;
    if (on) rb_put(P, buf[ph & 1]);
    __syncthreads();
  }
  if (!on) return;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (P.ti[k] < 0 || P.ti[k] >= TW || P.tj < 0 || P.tj >= TH) continue;
    if (i0 + P.ti[k] < L.nx && j0 + P.tj < L.ny) out[P.g[k]] = P.x[k];
  }
}

// The coarse end of the pcg_mg V-cycle (and of the stationary multigrid's) in
// one workgroup: levels C.lev[0..nl) (the first with at most MG_COARSE_MAX
// cells, or the last level alone), S sweeps from zero + residual restriction
// down, 2S sweeps from zero on the last level (the second S reversed),
// prolongation + S sweeps up; the same arithmetic per cell as the tiled legs.
// With C.rb the sweeps are red-black Gauss-Seidel, reversed (black first) on
// the way up and in the last level's second S. b0 is level 0's right-hand
// side, out receives its result; x0, when given, is level 0's starting field
// (the stationary multigrid on a grid small enough to need no legs).
//
// Bound by latency: a chain of about 10 half-sweeps per level, each a round of
// LDS reads, five dependent fp64 operations and a barrier. So a thread owns
// its cells for a whole visit of a level, their coefficients, right-hand sides
// and values in registers (level 0's for the whole cycle), and a half-sweep
// reads only the four neighbours' values from LDS; the levels below the first
// have at most one cell per thread. Sweeps are out of place between two
// buffers, because a level with an odd periodic side has same-colour
// neighbours across the wrap, whose old values the reference reads.
// The three levels from 32 x 32 down: 11.2 us against 14.9 with every field
// in LDS and 1024 threads (rbgs), 10.4 against 14.7 (Jacobi). A last level of
// more than 1024 cells is k_mg_last_level's.
template <class R>
struct CycCell {
  R inv, b, ke, kw, kn, ks, m;
  int c, ce, cw, cn, cs;
  int up;  // the coarser level's cell that holds this one
  int par;
  bool on;
};

// Neighbours and colour of cell c of level L (n cells; off when c >= n).
template <class R>
__device__ __forceinline__ CycCell<R> cyc_index(const MgLevelT<R>& L, int c) {
  CycCell<R> K;
  K.on = c < (int)L.n;
  K.c = K.on ? c : 0;
  const int j = K.c / L.nx, i = K.c - j * L.nx;
  K.ce = j * L.nx + wrap(i, 1, L.nx);
  K.cw = j * L.nx + wrap(i, -1, L.nx);
  K.cn = wrap(j, 1, L.ny) * L.nx + i;
  K.cs = wrap(j, -1, L.ny) * L.nx + i;
  K.up = (j / 2) * (L.nx / 2) + i / 2;
  K.par = (i + j) & 1;
  return K;
}
template <class R>
__device__ __forceinline__ void cyc_coefficients(CycCell<R>& K, const R* ku, const R* kv,
                                                 const R* inv, const uint8_t* m) {
  K.inv = inv[K.c];
  K.ke = ku[K.c];
  K.kw = ku[K.cw];
  K.kn = kv[K.c];
  K.ks = kv[K.cs];
  K.m = mkr<R>(m[K.c]);
}

// A x at a cell from its own value and its neighbours' (all masked already,
// so apply_from's multiplications by the masks are exact no-ops).
template <class R>
__device__ __forceinline__ R cyc_apply(const CycCell<R>& K, R coef, const Divisor<R>& by_dx2,
                                       const Divisor<R>& by_dy2, R xc, R xe, R xw, R xn, R xs) {
  const R lap = by_dx2(K.ke * (xe - xc) - K.kw * (xc - xw)) +
                by_dy2(K.kn * (xn - xc) - K.ks * (xc - xs));
  return (xc - coef * lap) * K.m + xc * (R(1) - K.m);
}

// The two field buffers of the cycle; `cur` holds the last field written.
template <class R>
struct CycField {
  R *cur, *next;
  __device__ __forceinline__ void swap() {
    R* t = cur;
    cur = next;
    next = t;
  }
};

// S sweeps on the cells of one level, from f.cur (or from zero), the own
// values in v; the result in v and in f.cur.
template <class R, int Q>
__device__ __forceinline__ void cyc_sweeps(const MgLevelT<R>& L, CycCell<R>* K, R* v,
                                           CycField<R>& f, R omega, bool rb, int S, bool zero,
                                           bool reverse) {
  // all cells' loads, then all updates, then all stores: a thread's cells
  // overlap, and a cell that is off or of the other colour computes a value
  // that is not kept
  R xe[Q], xw[Q], xn[Q], xs[Q];
  auto neighbours = [&](bool z) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      xe[q] = z ? R(0) : f.cur[K[q].ce];
      xw[q] = z ? R(0) : f.cur[K[q].cw];
      xn[q] = z ? R(0) : f.cur[K[q].cn];
      xs[q] = z ? R(0) : f.cur[K[q].cs];
    }
  };
  auto put = [&] {
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (K[q].on) f.next[K[q].c] = v[q];
    __syncthreads();
    f.swap();
  };
  if (rb) {
    auto half = [&](int col, bool last, bool z) {
      neighbours(z);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const R u = rbgs_from<R>(K[q].inv, K[q].b, L.cx, L.cy, K[q].ke, K[q].kw, K[q].kn,
                                 K[q].ks, xe[q], xw[q], xn[q], xs[q]);
        v[q] = K[q].par == col ? u : v[q];
        if (last) v[q] = v[q] * K[q].m;
      }
      put();
    };
    const int first = reverse ? 1 : 0;
    for (int s = 0; s < S; ++s) {
      half(first, false, zero && s == 0);
      half(1 - first, true, false);
    }
  } else {
    const Divisor<R> by_dx2 = uniform_divisor<R>(L.dx2), by_dy2 = uniform_divisor<R>(L.dy2);
    for (int s = 0; s < S; ++s) {
      neighbours(zero && s == 0);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const R ax = cyc_apply(K[q], L.coef, by_dx2, by_dy2, v[q], xe[q], xw[q], xn[q], xs[q]);
        v[q] = v[q] + omega * (K[q].inv * (K[q].b - ax)) * K[q].m;
      }
      put();
    }
  }
}

// The masked residual of the level's field (f.cur, own values v) into res.
template <class R, int Q>
__device__ __forceinline__ void cyc_residual(const MgLevelT<R>& L, const CycCell<R>* K,
                                             const R* v, const CycField<R>& f, R* res) {
  const Divisor<R> by_dx2 = uniform_divisor<R>(L.dx2), by_dy2 = uniform_divisor<R>(L.dy2);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (!K[q].on) continue;
    const R ax = cyc_apply(K[q], L.coef, by_dx2, by_dy2, v[q], f.cur[K[q].ce], f.cur[K[q].cw],
                           f.cur[K[q].cn], f.cur[K[q].cs]);
    res[K[q].c] = (K[q].b - ax) * K[q].m;
  }
  __syncthreads();
}

constexpr int CYC_THREADS = 256, CYC_CELLS = MG_COARSE_MAX / CYC_THREADS;
template <class R, class RB, class RO>
__global__ __launch_bounds__(CYC_THREADS) void k_mg_coarse_cycle(MgCycleT<R> C, R omega, int S,
                                                                 const RB* __restrict__ b0,
                                                                 const R* x0, RO* out,
                                                                 const PcgScalars* sc) {
  constexpr int NT = CYC_THREADS, Q = CYC_CELLS;
  const bool done = finished(sc);  // tested once the loads are on their way
  extern __shared__ __align__(16) unsigned char cyc_raw[];
  R* cyc = reinterpret_cast<R*>(cyc_raw);
  const int tid = threadIdx.x;
  const int n0 = (int)C.lev[0].n;
  const bool rb = C.rb != 0;
  CycField<R> f{cyc, cyc + n0};
  R* res = cyc + 2 * n0;
  // level 0's cells, for the whole cycle; the levels below copied into LDS
  // when they fit
  CycCell<R> K0[Q];
  R v0[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    K0[q] = cyc_index(C.lev[0], tid + q * NT);
    cyc_coefficients(K0[q], C.lev[0].Ku, C.lev[0].Kv, C.lev[0].inv_diag, C.lev[0].mask);
    K0[q].b = (R)b0[K0[q].c];
    v0[q] = x0 ? x0[K0[q].c] : R(0);
  }
  if (C.stage)
    for (int l = 1; l < C.nl; ++l) {
      const MgLevelT<R>& G = C.lev[l];
      const int n = (int)G.n;
      if (tid < n) {
        R* k = cyc + C.coff[l];
        k[tid] = G.Ku[tid];
        k[n + tid] = G.Kv[tid];
        k[2 * n + tid] = G.inv_diag[tid];
        cyc_raw[C.moff[l] + tid] = G.mask[tid];
      }
    }
  if (x0) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (K0[q].on) f.cur[K0[q].c] = v0[q];
  }
  __syncthreads();
  if (done) return;
  auto level = [&](int l) {  // this thread's cell of a level below the first
    const MgLevelT<R>& G = C.lev[l];
    CycCell<R> K = cyc_index(G, tid);
    if (C.stage) {
      const R* k = cyc + C.coff[l];
      cyc_coefficients(K, k, k + (int)G.n, k + 2 * (int)G.n, cyc_raw + C.moff[l]);
    } else {
      cyc_coefficients(K, G.Ku, G.Kv, G.inv_diag, G.mask);
    }
    return K;
  };
  const int last = C.nl - 1;
  cyc_sweeps<R, Q>(C.lev[0], K0, v0, f, omega, rb, S, x0 == nullptr, false);
  if (last == 0) {
    cyc_sweeps<R, Q>(C.lev[0], K0, v0, f, omega, rb, S, false, true);
  } else {
    cyc_residual<R, Q>(C.lev[0], K0, v0, f, res);
    for (int l = 1; l <= last; ++l) {
      CycCell<R> K = level(l);
      // the restricted residual of the level above (its cells by rows)
      const int fnx = C.lev[l - 1].nx;
      const int j = K.c / C.lev[l].nx, i = K.c - j * C.lev[l].nx;
      const int q = 2 * j * fnx + 2 * i;
      K.b = R(0.25) * (res[q] + res[q + 1] + res[q + fnx] + res[q + fnx + 1]);
      R v = R(0);
      cyc_sweeps<R, 1>(C.lev[l], &K, &v, f, omega, rb, S, true, false);
      if (l == last) {
        cyc_sweeps<R, 1>(C.lev[l], &K, &v, f, omega, rb, S, false, true);
      } else {
        if (K.on) {
          cyc[C.boff[l] + K.c] = K.b;
          cyc[C.xoff[l] + K.c] = v;
        }
        cyc_residual<R, 1>(C.lev[l], &K, &v, f, res);
      }
    }
    for (int l = last - 1; l >= 1; --l) {
      CycCell<R> K = level(l);
      K.b = cyc[C.boff[l] + K.c];
      R v = cyc[C.xoff[l] + K.c] + f.cur[K.up] * K.m;
      if (K.on) f.next[K.c] = v;
      __syncthreads();
      f.swap();
      cyc_sweeps<R, 1>(C.lev[l], &K, &v, f, omega, rb, S, false, true);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (!K0[q].on) continue;
      v0[q] = v0[q] + f.cur[K0[q].up] * K0[q].m;
      f.next[K0[q].c] = v0[q];
    }
    __syncthreads();
    f.swap();
    cyc_sweeps<R, Q>(C.lev[0], K0, v0, f, omega, rb, S, false, true);
  }
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (K0[q].on) out[K0[q].c] = (RO)v0[q];
}

// A last level alone of 1025 to MG_COARSE_LAST_MAX cells in one workgroup: S
// sweeps and S reversed ones from x0 (null: zero), the same arithmetic per cell
// as k_mg_coarse_cycle's. RBS: red-black Gauss-Seidel, else damped Jacobi. A
// thread owns P pairs of consecutive cells, which are one red and one black on
// any width, so a half-sweep updates one cell of each pair; coefficients,
// right-hand sides and values are in registers, the fields neighbours read in
// LDS (two buffers of n0 values).
// Bound by latency, and with 16 waves by LDS reads. A solve on one level of
// 64 x 64, rbgs and Jacobi: 1207 and 1655 us; with every field in LDS and the
// coefficients from memory 2187 and 2587; in the form above, where cells of both
// colours compute in every half-sweep and four cells per thread spill 78
// registers, 2885 and 3070. On 50 x 50 1155 and 1634, 1506 and 1983, 2788 and 2988.
template <class R>
struct LastCell {
  R inv, b, ke, kw, kn, ks, m;
  int c, ce, cw, cn, cs;
  bool on;
};
template <class R, class RB, class RO, int P, bool RBS>
__global__ __launch_bounds__(1024) void k_mg_last_level(MgLevelT<R> L, R omega, int S,
                                                        const RB* __restrict__ b0, const R* x0,
                                                        RO* out, const PcgScalars* sc) {
  const bool done = finished(sc);  // tested once the loads are on their way
  extern __shared__ __align__(16) unsigned char last_raw[];
  const int n = (int)L.n;
  R* cur = reinterpret_cast<R*>(last_raw);
  R* next = cur + n;
  LastCell<R> K[P][2];  // a pair's red and black cell
  R v[P][2];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int c0 = 2 * ((int)threadIdx.x + p * 1024);
    const int j0 = c0 / L.nx, black = (c0 - j0 * L.nx + j0) & 1;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      LastCell<R>& k = K[p][q];
      const int c = c0 + (q ^ black);
      k.on = c < n;
      k.c = k.on ? c : 0;
      const int j = k.c / L.nx, i = k.c - j * L.nx;
      k.ce = j * L.nx + wrap(i, 1, L.nx);
      k.cw = j * L.nx + wrap(i, -1, L.nx);
      k.cn = wrap(j, 1, L.ny) * L.nx + i;
      k.cs = wrap(j, -1, L.ny) * L.nx + i;
      k.inv = L.inv_diag[k.c];
      k.b = (R)b0[k.c];
      k.ke = L.Ku[k.c];
      k.kw = L.Ku[k.cw];
      k.kn = L.Kv[k.c];
      k.ks = L.Kv[k.cs];
      k.m = mkr<R>(L.mask[k.c]);
      v[p][q] = x0 ? x0[k.c] : R(0);
    }
  }
  auto put = [&] {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (K[p][q].on) next[K[p][q].c] = v[p][q];
    __syncthreads();
    R* t = cur;
    cur = next;
    next = t;
  };
  put();  // the starting field
  if (done) return;
  const Divisor<R> by_dx2 = uniform_divisor<R>(L.dx2), by_dy2 = uniform_divisor<R>(L.dy2);
  for (int s = 0; s < 2 * S; ++s) {
    if constexpr (RBS) {
      const bool reverse = s >= S;
      auto half = [&](auto colour, bool last) {
        constexpr int q = decltype(colour)::value;
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const LastCell<R>& k = K[p][q];
          v[p][q] = rbgs_from<R>(k.inv, k.b, L.cx, L.cy, k.ke, k.kw, k.kn, k.ks, cur[k.ce],
                                 cur[k.cw], cur[k.cn], cur[k.cs]);
          if (last) {
            v[p][0] = v[p][0] * K[p][0].m;
            v[p][1] = v[p][1] * K[p][1].m;
          }
        }
        put();
      };
      using Red = std::integral_constant<int, 0>;
      using Black = std::integral_constant<int, 1>;
      if (reverse) {
        half(Black{}, false);
        half(Red{}, true);
      } else {
        half(Red{}, false);
        half(Black{}, true);
      }
    } else {
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const LastCell<R>& k = K[p][q];
          const R xc = v[p][q];
          const R lap = by_dx2(k.ke * (cur[k.ce] - xc) - k.kw * (xc - cur[k.cw])) +
                        by_dy2(k.kn * (cur[k.cn] - xc) - k.ks * (xc - cur[k.cs]));
          const R ax = (xc - L.coef * lap) * k.m + xc * (R(1) - k.m);
          v[p][q] = xc + omega * (k.inv * (k.b - ax)) * k.m;
        }
      put();
    }
  }
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (K[p][q].on) out[K[p][q].c] = (RO)v[p][q];
}

// LDS of a cycle: two field buffers and the residual, the lower levels'
// right-hand sides and x_S, and their coefficients when they fit.
template <class R>
size_t mg_cycle_layout(MgCycleT<R>& C) {
  int off = 3 * (int)C.lev[0].n;
  for (int l = 1; l < C.nl; ++l) {
    C.boff[l] = off;
    off += (int)C.lev[l].n;
    C.xoff[l] = off;
    off += (int)C.lev[l].n;
  }
  const size_t vectors = (size_t)off * sizeof(R);
  for (int l = 1; l < C.nl; ++l) {
    C.coff[l] = off;
    off += 3 * (int)C.lev[l].n;
  }
  size_t bytes = (size_t)off * sizeof(R);
  for (int l = 1; l < C.nl; ++l) {
    C.moff[l] = (int)bytes;
    bytes += (size_t)C.lev[l].n;
  }
  bytes = (bytes + 15) / 16 * 16;
  C.stage = bytes <= MG_CYCLE_LDS ? 1 : 0;
  return C.stage ? bytes : vectors;
}
template size_t mg_cycle_layout<double>(MgCycle&);
template size_t mg_cycle_layout<float>(MgCycleF&);

namespace {
// go(kernel, threads) for the cycle's first level of n0 cells: the cycle up to
// MG_COARSE_MAX, beyond that (a last level alone) one or two pairs of cells for
// each of 1024 threads.
template <class R, class RB, class RO, class Cycle, class Last>
auto with_cycle(long long n0, bool rb, const Cycle& cycle, const Last& last) {
  if (n0 <= MG_COARSE_MAX) return cycle(k_mg_coarse_cycle<R, RB, RO>);
  if constexpr (std::is_same_v<R, double>) {
    if (rb)
      return n0 <= 2048 ? last(k_mg_last_level<R, RB, RO, 1, true>)
                        : last(k_mg_last_level<R, RB, RO, 2, true>);
  }
  return n0 <= 2048 ? last(k_mg_last_level<R, RB, RO, 1, false>)
                    : last(k_mg_last_level<R, RB, RO, 2, false>);
}
template <class R, class RB, class RO>
int cycle_lds(const MgCycleT<R>& C, size_t lds) {
  const long long n0 = C.lev[0].n;
  if (lds > MG_CYCLE_LDS || n0 > MG_COARSE_LAST_MAX || (n0 > MG_COARSE_MAX && C.nl != 1))
    return -1;
  auto set = [&](auto kernel) {
    return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds) == hipSuccess
               ? 0
               : -2;
  };
  return with_cycle<R, RB, RO>(n0, C.rb != 0, set, set);
}
template <class R, class RB, class RO>
void launch_cycle(const MgCycleT<R>& C, size_t lds, R omega, int S, const RB* b0, const R* x0,
                  RO* out, const PcgScalars* sc, hipStream_t s) {
  with_cycle<R, RB, RO>(
      C.lev[0].n, C.rb != 0,
      [&](auto kernel) { kernel<<<1, CYC_THREADS, lds, s>>>(C, omega, S, b0, x0, out, sc); },
      [&](auto kernel) { kernel<<<1, 1024, lds, s>>>(C.lev[0], omega, S, b0, x0, out, sc); });
}
}  // namespace

int mg_cycle_prepare(const MgCycle& C, size_t lds) {
  return cycle_lds<double, double, double>(C, lds);
}

int mg_cycle_prepare_f32(const MgCycleF& C, size_t lds) {
  const int rc = cycle_lds<float, double, double>(C, lds);
  return rc ? rc : cycle_lds<float, float, float>(C, lds);
}

void launch_mg_coarse_cycle(const MgCycle& C, size_t lds, double omega, int S, const double* b0,
                            const double* x0, double* out, const PcgScalars* sc, hipStream_t s) {
  launch_cycle<double, double, double>(C, lds, omega, S, b0, x0, out, sc, s);
}

void launch_mg_coarse_cycle_f32(const MgCycleF& C, size_t lds, float omega, int S,
                                const double* b0_d, const float* b0_f, double* out_d,
                                float* out_f, const PcgScalars* sc, hipStream_t s) {
  if (b0_d)
    launch_cycle<float, double, double>(C, lds, omega, S, b0_d, nullptr, out_d, sc, s);
  else
    launch_cycle<float, float, float>(C, lds, omega, S, b0_f, nullptr, out_f, sc, s);
}

// Fused-leg tile shapes (cells per workgroup tile; every shape gives the
// same values, they differ only in halo recomputation and occupancy):
// 0: 32 x 16, 1: 64 x 8, 2: 16 x 16, 3: 64 x 16. Shapes 1-3 are built for
// 2 sweeps per side (the default), other sweep counts use shape 0.
constexpr int SHAPE_W[MG_TILE_SHAPES] = {32, 64, 16, 64}, SHAPE_H[MG_TILE_SHAPES] = {16, 8, 16, 16};
template <class R>
dim3 mg_tile_grid_shape(const MgLevelT<R>& L, int shape) {
  return dim3((unsigned)((L.nx + SHAPE_W[shape] - 1) / SHAPE_W[shape]),
              (unsigned)((L.ny + SHAPE_H[shape] - 1) / SHAPE_H[shape]));
}

namespace {
// One leg kernel per sweep count and tile shape.
template <class Go>
void leg_dispatch(int S, int shape, const Go& go) {
  if (S == 1) go(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
  else if (S == 3) go(std::integral_constant<int, 3>{}, std::integral_constant<int, 0>{});
  else if (shape == 1) go(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
  else if (shape == 2) go(std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
  else if (shape == 3) go(std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 2>{}, std::integral_constant<int, 0>{});
}
int leg_shape(int S, int shape) { return S == 2 && shape >= 0 && shape < MG_TILE_SHAPES ? shape : 0; }

template <class R, class RB>
void leg_down(int S, int shape, hipStream_t s, const MgLevelT<R>& L, const MgLevelT<R>& C, R omega,
              const RB* b, R* xs_out, R* bc, const PcgScalars* sc) {
  shape = leg_shape(S, shape);
  const dim3 grid = mg_tile_grid_shape(L, shape);
  leg_dispatch(S, shape, [&](auto sv, auto qv) {
    constexpr int SS = decltype(sv)::value, W = SHAPE_W[decltype(qv)::value],
                  T = SHAPE_H[decltype(qv)::value];
    k_mg_down<SS, R, RB, W, T><<<grid, JacRegion<SS, W, T>::NT, 0, s>>>(L, C, omega, b, xs_out, bc,
                                                                       sc);
  });
}
template <class R, class RB, class RO>
void leg_up(int S, int shape, hipStream_t s, const MgLevelT<R>& L, R omega, const R* xs_in,
            const R* ec, const RB* b, RO* out, const PcgScalars* sc) {
  shape = leg_shape(S, shape);
  const dim3 grid = mg_tile_grid_shape(L, shape);
  leg_dispatch(S, shape, [&](auto sv, auto qv) {
    constexpr int SS = decltype(sv)::value, W = SHAPE_W[decltype(qv)::value],
                  T = SHAPE_H[decltype(qv)::value];
    k_mg_up<SS, R, RB, RO, W, T><<<grid, JacRegion<SS, W, T>::NT, 0, s>>>(L, omega, xs_in, ec, b,
                                                                         out, sc);
  });
}
}  // namespace

void launch_mg_down(int S, int shape, hipStream_t s, const MgLevel& L, const MgLevel& C,
                    double omega, const double* b, double* xs_out, double* bc,
                    const PcgScalars* sc) {
  leg_down<double, double>(S, shape, s, L, C, omega, b, xs_out, bc, sc);
}
void launch_mg_up(int S, int shape, hipStream_t s, const MgLevel& L, double omega,
                  const double* xs_in, const double* ec, const double* b, double* out,
                  const PcgScalars* sc) {
  leg_up<double, double, double>(S, shape, s, L, omega, xs_in, ec, b, out, sc);
}
void launch_mg_down_f32(int S, int shape, hipStream_t s, const MgLevelF& L, const MgLevelF& C,
                        float omega, const double* b_d, const float* b_f, float* xs_out,
                        float* bc, const PcgScalars* sc) {
  if (b_d) leg_down<float, double>(S, shape, s, L, C, omega, b_d, xs_out, bc, sc);
  else leg_down<float, float>(S, shape, s, L, C, omega, b_f, xs_out, bc, sc);
}
void launch_mg_up_f32(int S, int shape, hipStream_t s, const MgLevelF& L, float omega,
                      const float* xs_in, const float* ec, const double* b_d, const float* b_f,
                      double* out_d, float* out_f, const PcgScalars* sc) {
  if (b_d) leg_up<float, double, double>(S, shape, s, L, omega, xs_in, ec, b_d, out_d, sc);
  else leg_up<float, float, float>(S, shape, s, L, omega, xs_in, ec, b_f, out_f, sc);
}

// x_in: the level's starting field (null: zero; 2 sweeps only otherwise).
void launch_mg_down_rb(int S, int shape, hipStream_t s, const MgLevel& L, const MgLevel& C,
                       const double* x_in, const double* b, double* xs_out, double* bc,
                       const PcgScalars* sc) {
  shape = leg_shape(S, shape);
  const dim3 grid = mg_tile_grid_shape(L, shape);
  leg_dispatch(S, shape, [&](auto sv, auto qv) {
    constexpr int SS = decltype(sv)::value, W = SHAPE_W[decltype(qv)::value],
                  T = SHAPE_H[decltype(qv)::value];
    if constexpr (SS == 2) {
      if (x_in) {
        k_mg_down_rb<SS, true, W, T><<<grid, RbRegion<2 * SS + 1, W, T>::NT, 0, s>>>(
            L, C, x_in, b, xs_out, bc, sc);
        return;
      }
    }
    k_mg_down_rb<SS, false, W, T><<<grid, RbRegion<2 * SS, W, T>::NT, 0, s>>>(
        L, C, nullptr, b, xs_out, bc, sc);
  });
}

void launch_mg_up_rb(int S, int shape, hipStream_t s, const MgLevel& L, const double* xs_in,
                     const double* ec, const double* b, double* out, const PcgScalars* sc) {
  shape = leg_shape(S, shape);
  const dim3 grid = mg_tile_grid_shape(L, shape);
  leg_dispatch(S, shape, [&](auto sv, auto qv) {
    constexpr int SS = decltype(sv)::value, W = SHAPE_W[decltype(qv)::value],
                  T = SHAPE_H[decltype(qv)::value];
    k_mg_up_rb<SS, W, T><<<grid, RbRegion<2 * SS, W, T>::NT, 0, s>>>(L, xs_in, ec, b, out, sc);
  });
}

// fp32 copies of one level's face coefficients and inverse diagonal
// (round to nearest).
__global__ void k_mg_to_f32(long long n, const double* __restrict__ Ku,
                            const double* __restrict__ Kv, const double* __restrict__ inv,
                            float* __restrict__ fKu, float* __restrict__ fKv,
                            float* __restrict__ finv) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  fKu[c] = (float)Ku[c];
  fKv[c] = (float)Kv[c];
  finv[c] = (float)inv[c];
}

}  // namespace hoc
