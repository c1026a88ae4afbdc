// LDS-tiled column kernels ("2.5D"): a workgroup owns a TX x TY tile of
// columns and marches down a range of levels. At each level the fields that enter
// horizontal stencils are staged once in LDS with a 2-cell periodic halo,
// so every value is read from HBM about once instead of once per stencil
// point; the column's own vertical neighbours stay in a register window.
// Arithmetic and operand order are those of the untiled kernels (and of the
// reference's NumPy expressions), so the results are bitwise the same (in the
// range stated at Divisor).
#include <type_traits>

#include "hoc_device.h"
#include "hoc_kernels.h"

namespace hoc {

// Tile shape: 32 x 8 (HOC_TILE_TX, HOC_TILE_TY override it at build time;
// every shape with TX * TY = 256 gives the same bits).
#ifndef HOC_TILE_TX
#define HOC_TILE_TX 32
#endif
#ifndef HOC_TILE_TY
#define HOC_TILE_TY 8
#endif
constexpr int TX = HOC_TILE_TX, TY = HOC_TILE_TY, HALO = 2;
static_assert(TX * TY == 256 && TX + TY <= 256, "tile of 256 threads");
constexpr int SX = TX + 2 * HALO, SY = TY + 2 * HALO;
constexpr int TILE_THREADS = TX * TY;

__device__ __forceinline__ int pmod(int a, int n) {
  int r = a % n;
  return r < 0 ? r + n : r;
}

// Tracer face value for the configured scheme (model3d_v05.py:486-494), in
// the flux type R (double: the reference's arithmetic; float: the mixed step).
template <class R>
__device__ __forceinline__ R tracer_face(int adv, R cm, R c0, R c1, R c2, R vel, bool wm,
                                         bool w2) {
  if (adv == ADV_UP3 || adv == ADV_UP3_TVD)
    return kappa_face<R>(cm, c0, c1, c2, vel, wm, w2, adv == ADV_UP3_TVD);
  if (adv == ADV_CENTRED2) return R(0.5) * (c0 + c1);
  return vel > R(0) ? c0 : c1;
}

// Vertical interface value at interface kk of a column whose window holds
// c[kk-2], c[kk-1], c[kk], c[kk+1] and the wet flags of c[kk-2], c[kk+1].
template <class R>
__device__ __forceinline__ R tracer_face_z(int adv, int kk, int nz, R far_up, R above, R below,
                                           R far_dn, bool mup, bool mdn, R w) {
  if (kk == nz) return R(0);
  if (!(adv == ADV_UP3 || adv == ADV_UP3_TVD)) return R(0.5) * (above + below);
  const bool hu = kk >= 2 && mup;
  const bool hd = kk <= nz - 2 && mdn;
  return kappa_face_z<R>(kk >= 2 ? far_up : R(0), above, below, kk <= nz - 2 ? far_dn : R(0), w,
                         hu, hd, adv == ADV_UP3_TVD);
}

struct NoTile {};

// First threads that form the tile's west column of faces (TY of them) and
// its south row (TX): two different waves.
constexpr int EDGE_X = TX > 64 ? TX : 64, EDGE_Y = 0;
static_assert(EDGE_X + TY <= TILE_THREADS && EDGE_Y + TX <= EDGE_X, "edge threads");

// Levels at which the east (axis 0) or north (axis 1) face of column (j, i)
// is wet, for a static z-level geometry, and the face's thickness at the last
// of them (its other levels are the face rule of two full cells).
__device__ __forceinline__ int face_levels(const Geo& geo, int axis, int j, int i, int ny,
                                           int nx) {
  const int c0 = j * nx + i;
  const int c1 = axis == 0 ? j * nx + pmod(i + 1, nx) : pmod(j + 1, ny) * nx + i;
  const int a = geo.nw[c0], b = geo.nw[c1];
  return (axis == 0 ? geo.mu2[c0] : geo.mv2[c0]) ? (a < b ? a : b) : 0;
}
__device__ __forceinline__ double face_last(const StepParams& p, const Geo& geo, int axis, int n,
                                            int j, int i, int ny, int nx) {
  if (n <= 0) return 0.0;
  const int c0 = j * nx + i;
  const int c1 = axis == 0 ? j * nx + pmod(i + 1, nx) : pmod(j + 1, ny) * nx + i;
  return face_value(p.face_rule, cg_dz(p.dzr, geo.nw[c0], geo.hb[c0], n - 1),
                    cg_dz(p.dzr, geo.nw[c1], geo.hb[c1], n - 1));
}

// ------------------------------------------------------------- tracers
// Staged tile of one tracer on one level (two buffers: level k + 1 lands
// while level k is read), with the cell masks for geometry read from the
// arrays.
template <class R>
struct TracerLds {
  R c[SY][SX];
};
struct TracerMaskLds {
  uint8_t m[SY][SX];
};

// Face fluxes of one field on one level, each computed once: the advective
// flux and the horizontal-diffusion gradient, on the x-faces (index q:
// between tile columns q-1 and q) and the y-faces (between rows q-1 and q).
template <class R>
struct FaceLds {
  R fx[TY][TX + 1], gx[TY][TX + 1];
  R fy[TY + 1][TX], gy[TY + 1][TX];
};

constexpr int ST_H = (SX * SY + TILE_THREADS - 1) / TILE_THREADS;  // halo slots per thread

// Plane indexes of this thread's slots of the tile with its halo (slots
// beyond the tile read its first ones again; the value is not stored).
struct HaloOffs {
  unsigned h[ST_H];
};
__device__ __forceinline__ HaloOffs halo_offsets(int tid, int i0, int j0, int nx, int ny) {
  HaloOffs F;
#pragma unroll
  for (int q = 0; q < ST_H; ++q) {
    const int t = tid + q * TILE_THREADS;
    const int tt = t < SX * SY ? t : tid;
    F.h[q] = (unsigned)(pmod(j0 + tt / SX - HALO, ny) * nx + pmod(i0 + tt % SX - HALO, nx));
  }
  return F;
}

// Operands of the own east face, the own north face and, for the edge
// threads, the edge face at one level: velocity and, for geometry read from
// the arrays, thickness and mask.
struct TracerFaceRegs {
  double vel[3];
  double dz[3];
  uint8_t m[3];
};

// Right-hand sides of the tracers' implicit vertical diffusion: one tracer of
// one tile on the levels [k0, k0 + nk) per workgroup: advection + K_h
// Laplacian + explicit part of the vertical diffusion + surface flux
// (libs/core/model3d_v05.py:466-512), which k_tracer_solve then solves in
// place. R is the type of the advective fluxes and the K_h gradients: double
// for the plain step (bitwise the reference), float for the mixed step. ZC:
// the static z-level geometry in column form (thicknesses, their inverses and
// masks from the columns' wet-level counts and deepest thicknesses, in
// registers; the same bits).
// Bound by the latency of its fp64 chains, like the momentum kernel: one
// tracer per workgroup (128 registers, 4 waves per SIMD), the column solve in
// a kernel of its own so that the levels can be cut into ranges, and the own
// faces' velocities straight from their arrays. Two more fields pass through
// memory than with the solve in the same march (67 us of traffic at 512 x 512
// x 40), which marched 64 tiles at 128 x 128 with the recurrence in every
// level. Both kernels per step, before -> now: 128 x 4 x 20 135 -> 24 us,
// 128 x 128 x 30 224 -> 64, 512 x 512 x 40 689 -> 430, 1000 x 1000 x 30 1690 ->
// 1179; fp32 fluxes at 640 x 512 x 48 1244 -> 626.
template <class R, bool ZC, bool TVD>
__global__ __launch_bounds__(TILE_THREADS) void k_tracer_rhs(
    Dims d, StepParams p, Geo geo, int nk, const double* __restrict__ T,
    const double* __restrict__ S, const double* __restrict__ b, const double* __restrict__ u,
    const double* __restrict__ v, const double* __restrict__ w, const double* __restrict__ Kh,
    double* __restrict__ T_out, double* __restrict__ S_out, double* __restrict__ b_out) {
  __shared__ TracerLds<R> LB[2];
  __shared__ FaceLds<R> F;
  __shared__ std::conditional_t<ZC, NoTile, TracerMaskLds> MB[2];
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  const long long n2 = d.n2;
  const bool ts = p.tracers_ts != 0;
  const BlockTile B = xcd_block((nx + TX - 1) / TX, (ny + TY - 1) / TY, ts ? 2 : 1);
  const double* C = B.part == 1 ? S : (ts ? T : b);
  double* out = B.part == 1 ? S_out : (ts ? T_out : b_out);
  const double flux = B.part == 1 ? p.flux_S : (ts ? p.flux_T : 0.0);
  const int tid = threadIdx.x;
  const int tx = tid % TX, ty = tid / TX;
  const int i0 = B.x * TX, j0 = B.y * TY;
  const int i = i0 + tx, j = j0 + ty;
  const bool active = i < nx && j < ny;
  const int k0 = B.z * nk;
  const int k1 = k0 + nk < nz ? k0 + nk : nz;
  const int adv = TVD ? (int)ADV_UP3_TVD : p.advection;
  const bool has_adv = adv != ADV_NONE;
  const Divisor<R> by_dx = uniform_divisor<R>(p.dx), by_dy = uniform_divisor<R>(p.dy);
  // plane indexes of the own point (clamped into the grid for the lanes
  // beyond it) and of the point before this thread's edge face
  const int jc = pmod(j, ny), ic = pmod(i, nx);
  const int cc = jc * nx + ic;
  const int xe = tid - EDGE_X, ye = tid - EDGE_Y;
  const bool is_x = xe >= 0 && xe < TY, is_y = ye >= 0 && ye < TX;
  const int je = is_x ? pmod(j0 + xe, ny) : (is_y ? pmod(j0 - 1, ny) : jc);
  const int ie = is_x ? pmod(i0 - 1, nx) : (is_y ? pmod(i0 + ye, nx) : ic);
  const int ce = je * nx + ie;
  const unsigned b0 = 8u * (unsigned)cc, be = 8u * (unsigned)ce;
  const double* ve = is_x ? u : v;  // the edge face's velocity, thickness and mask arrays
  const double* dze = is_x ? geo.dz3u : geo.dz3v;
  const uint8_t* me = is_x ? geo.m3u : geo.m3v;

  R rc[ST_H];
  uint8_t rm[ST_H];
  TracerFaceRegs rf;
  const HaloOffs HO = halo_offsets(tid, i0, j0, nx, ny);
  auto load = [&](long long o) {
#pragma unroll
    for (int q = 0; q < ST_H; ++q) {
      rc[q] = (R)at_byte(C + o, 8u * HO.h[q]);
      if constexpr (!ZC) rm[q] = at_byte(geo.m3 + o, HO.h[q]);
    }
    rf.vel[0] = at_byte(u + o, b0);
    rf.vel[1] = at_byte(v + o, b0);
    rf.vel[2] = ve[o + ce];
    if constexpr (!ZC) {
      rf.dz[0] = at_byte(geo.dz3u + o, b0);
      rf.dz[1] = at_byte(geo.dz3v + o, b0);
      rf.dz[2] = dze[o + ce];
      rf.m[0] = at_byte(geo.m3u + o, (unsigned)cc);
      rf.m[1] = at_byte(geo.m3v + o, (unsigned)cc);
      rf.m[2] = me[o + ce];
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < ST_H; ++q) {
      const int t = tid + q * TILE_THREADS;
      if (t < SX * SY) {
        LB[buf].c[t / SX][t % SX] = rc[q];
        if constexpr (!ZC) MB[buf].m[t / SX][t % SX] = rm[q];
      }
    }
  };
  load((long long)k0 * n2);

  // the column form: wet levels of the far cells and of the face itself
  // (bytes: before, beyond, own; a count is at most 255) and the thickness at
  // the last one, for the east, north and edge face; the own column
  unsigned fw[3] = {0, 0, 0};
  double fl[3] = {0.0, 0.0, 0.0};
  double full = 0.0;
  InvCol ca{};
  int nwc = 0;
  if constexpr (ZC) {
    auto face = [&](int axis, int jj, int ii, unsigned& wet, double& last) {
      const int jm = axis ? pmod(jj - 1, ny) : jj, j2 = axis ? pmod(jj + 2, ny) : jj;
      const int im = axis ? ii : pmod(ii - 1, nx), i2 = axis ? ii : pmod(ii + 2, nx);
      const int n = face_levels(geo, axis, jj, ii, ny, nx);
      wet = (unsigned)geo.nw[jm * nx + im] | (unsigned)geo.nw[j2 * nx + i2] << 8 |
            (unsigned)n << 16;
      last = face_last(p, geo, axis, n, jj, ii, ny, nx);
    };
    face(0, jc, ic, fw[0], fl[0]);
    face(1, jc, ic, fw[1], fl[1]);
    if (is_x || is_y) face(is_x ? 0 : 1, je, ie, fw[2], fl[2]);
    full = uniform_value(face_value(p.face_rule, p.dzr, p.dzr));
    nwc = geo.nw[cc];
    ca = inv_col(nwc, uniform_value(p.dzr), nwc > 0 ? geo.hb[cc] : 0.0);
  }
  auto cell_wet = [&](int kk) -> bool {  // the own column, 0 <= kk < nz
    if constexpr (ZC) return kk < nwc;
    else return at_byte(geo.m3 + kk * n2, (unsigned)cc) != 0;
  };
  auto idz = [&](int kk) -> double {  // 1 / spacing on interface kk, 1 <= kk < nz
    if constexpr (ZC) return ca.idzi(kk);
    else return safe_inv(at_byte(geo.dzi + kk * n2, b0));
  };
  auto inv = [&](int kk) -> double {
    if constexpr (ZC) return ca.inv(kk);
    else return safe_inv(at_byte(geo.dz3 + kk * n2, b0));
  };

  store(0);
  // own-column window of the tracer at k-2..k+2, with its wet flags (bits of
  // one register, or from the level count)
  double c5[5];
  unsigned m5 = 0;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const int kk = k0 + q - 2;
    const bool in = kk >= 0 && kk < nz;
    c5[q] = in ? at_byte(C + kk * n2, b0) : 0.0;
    if constexpr (!ZC)
      if (in && cell_wet(kk)) m5 |= 1u << q;
  }
  auto wet_at = [&](int k, int q) -> bool {  // cell k-2+q
    if constexpr (ZC) return k + q - 2 >= 0 && k + q - 2 < nwc;
    else return (m5 >> q & 1u) != 0;
  };
  double w_k = at_byte(w + k0 * n2, b0);
  double kh_k = at_byte(Kh + k0 * n2, b0);  // K_h and 1 / spacing on interface k
  double idz_k = k0 > 0 ? idz(k0) : 0.0;
  // interface value at the top of level k: of the first level the surface
  // cell's, else what the range above forms as its bottom one
  R cf_top = k0 == 0 ? R(c5[2])
                     : tracer_face_z<R>(adv, k0, nz, R(c5[0]), R(c5[1]), R(c5[2]), R(c5[3]),
                                        wet_at(k0, 0), wet_at(k0, 3), R(w_k));
  __syncthreads();
  for (int k = k0; k < k1; ++k) {
    const long long o = (long long)k * n2;
    const TracerLds<R>& L = LB[(k - k0) & 1];
    const TracerFaceRegs f = rf;
    if (k + 1 < k1) load(o + n2);
    // the own column's operands below level k, issued before the face pass
    const double w_k1 = at_byte(w + o + n2, b0);
    const double kh_k1 = at_byte(Kh + o + n2, b0);
    const double c_k3 = k + 3 < nz ? at_byte(C + o + 3 * n2, b0) : 0.0;
    // ---- faces: the own east and north ones, and the tile's west and south
    // edge ones by the edge threads
    {
      // thickness, far wet flags and own mask of face q whose point before it
      // is (yy, xx) of the tile
      auto geometry = [&](int q, int axis, int yy, int xx, R& dz, bool* m) {
        if constexpr (ZC) {
          const int n = (int)(fw[q] >> 16);
          dz = R(k < n - 1 ? full : (k == n - 1 ? fl[q] : 0.0));
          m[0] = k < (int)(fw[q] & 255u);
          m[1] = k < (int)(fw[q] >> 8 & 255u);
          m[2] = k < n;
        } else {
          const TracerMaskLds& M = MB[(k - k0) & 1];
          dz = R(f.dz[q]);
          m[0] = (axis ? M.m[yy - 1][xx] : M.m[yy][xx - 1]) != 0;
          m[1] = (axis ? M.m[yy + 2][xx] : M.m[yy][xx + 2]) != 0;
          m[2] = f.m[q] != 0;
        }
      };
      // x-face q of row r (between columns q-1 and q), operands s
      auto xface = [&](int r, int q, int s) {
        const int yy = r + HALO, x0 = q - 1 + HALO;
        R dz;
        bool m[3];
        geometry(s, 0, yy, x0, dz, m);
        const R a0 = L.c[yy][x0], a1 = L.c[yy][x0 + 1], vel = R(f.vel[s]);
        if (TVD || has_adv)
          F.fx[r][q] = dz * vel * tracer_face<R>(adv, L.c[yy][x0 - 1], a0, a1, L.c[yy][x0 + 2],
                                                 vel, m[0], m[1]);
        F.gx[r][q] = by_dx((m[2] ? R(1) : R(0)) * (a1 - a0));
      };
      // y-face q of column r (between rows q-1 and q)
      auto yface = [&](int q, int r, int s) {
        const int xx = r + HALO, y0 = q - 1 + HALO;
        R dz;
        bool m[3];
        geometry(s, 1, y0, xx, dz, m);
        const R a0 = L.c[y0][xx], a1 = L.c[y0 + 1][xx], vel = R(f.vel[s]);
        if (TVD || has_adv)
          F.fy[q][r] = dz * vel * tracer_face<R>(adv, L.c[y0 - 1][xx], a0, a1, L.c[y0 + 2][xx],
                                                 vel, m[0], m[1]);
        F.gy[q][r] = by_dy((m[2] ? R(1) : R(0)) * (a1 - a0));
      };
      xface(ty, tx + 1, 0);
      yface(ty + 1, tx, 1);
      if (is_x) xface(xe, 0, 2);
      if (is_y) yface(0, ye, 2);
    }
    __syncthreads();
    // ---- the own cell
    {
      const bool m_k = wet_at(k, 2);
      const double iv = inv(k);
      const bool lower = k + 1 < nz;
      const double idz_k1 = lower ? idz(k + 1) : 0.0;
      double tend = 0.0;
      if (!ts) tend = p.neg_N2 * (0.5 * (w_k + w_k1));
      if (TVD || has_adv) {
        const R hdiv = (by_dx(F.fx[ty][tx + 1] - F.fx[ty][tx]) +
                        by_dy(F.fy[ty + 1][tx] - F.fy[ty][tx])) * R(iv);
        const R cfb = tracer_face_z<R>(adv, k + 1, nz, R(c5[1]), R(c5[2]), R(c5[3]), R(c5[4]),
                                       wet_at(k, 1), wet_at(k, 4), R(w_k1));
        const R vdiv = (R(w_k) * cf_top - R(w_k1) * cfb) * R(iv);
        cf_top = cfb;
        tend = tend - (double)((hdiv + vdiv) * (m_k ? R(1) : R(0)));
      }
      if (p.has_K_h)
        tend = tend + p.K_h * (double)((m_k ? R(1) : R(0)) *
                                       (by_dx(F.gx[ty][tx + 1] - F.gx[ty][tx]) +
                                        by_dy(F.gy[ty + 1][tx] - F.gy[ty][tx])));
      // explicit vertical diffusion with the surface flux (vertical_var.py:80-106)
      const double dzd = explicit_diffusion_inv(k, nz, c5[1], c5[2], c5[3], idz_k, idz_k1, iv,
                                                wet_at(k, 1), m_k, lower && wet_at(k, 3), kh_k,
                                                kh_k1, flux, 0.0);
      double rhs = c5[2] + p.dt * tend + p.c_dzd * dzd;
      if (k == 0) rhs = rhs + p.thv_dt * flux * iv;
      if (active) put_byte(out + o, b0, rhs);
      // advance the windows
#pragma unroll
      for (int q = 0; q < 4; ++q) c5[q] = c5[q + 1];
      c5[4] = c_k3;
      if constexpr (!ZC) m5 = m5 >> 1 | (k + 3 < nz && cell_wet(k + 3) ? 16u : 0u);
      w_k = w_k1;
      kh_k = kh_k1;
      idz_k = idz_k1;
    }
    if (k + 1 < k1) store((k + 1 - k0) & 1);
    __syncthreads();
  }
}

// The tracers' implicit vertical diffusion, in place on the right-hand sides
// k_tracer_rhs left in the outputs: tri_b (K_h, no drag) factored and the
// forward sweep in one march down the column (c* parked in `cst`, d* in the
// outputs), then the back-substitution, the mask and the EOS
// (libs/core/model3d_v05.py:476-533). One pivot serves c* and both tracers:
// its reciprocal is formed once. Bound by HBM where the columns fill the chip
// (12 fields of 8 bytes per cell: 165 us at 512 x 512 x 40, 6.1 TB/s) and by the
// recurrence's latency below that, so operands are loaded SOLVE_AHEAD levels
// at a time ahead of it (2 / 4 / 8 levels: 436 / 425 / 454 us for both tracer
// kernels at 512 x 512 x 40, equal at 128 x 128 x 30) and a workgroup is one
// wave, which spreads few columns over the most compute units.
constexpr int SOLVE_AHEAD = 4, SOLVE_THREADS = 64;
template <bool ZC>
__global__ __launch_bounds__(SOLVE_THREADS) void k_tracer_solve(
    Dims d, StepParams p, Geo geo, const double* __restrict__ zs, const double* __restrict__ Kh,
    double* __restrict__ cst, double* __restrict__ T_out, double* __restrict__ S_out,
    double* __restrict__ b_out) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= d.n2) return;
  const int nz = d.nz;
  const long long n2 = d.n2;
  const bool ts = p.tracers_ts != 0;
  double* A = ts ? T_out : b_out;
  constexpr int W = SOLVE_AHEAD;
  InvCol ca{};
  int nwc = 0;
  double hbc = 0.0, bot = 0.0;
  if constexpr (ZC) {
    nwc = geo.nw[c];
    hbc = geo.hb[c];
    ca = inv_col(nwc, p.dzr, nwc > 0 ? hbc : 0.0);
    bot = nwc > 0 ? zs[nwc - 1] + hbc : 0.0;
  }
  // operands of W levels: right-hand sides, K_h below, and the geometry read
  // from the arrays
  struct Ahead {
    double a[W], s[W], kh[W], dz[W], dzi[W];
    bool wet[W];
  };
  auto load = [&](int kb, Ahead& g) {
#pragma unroll
    for (int q = 0; q < W; ++q) {
      const long long k = kb + q < nz ? kb + q : nz - 1;
      g.a[q] = A[k * n2 + c];
      g.s[q] = ts ? S_out[k * n2 + c] : 0.0;
      g.kh[q] = Kh[(k + 1) * n2 + c];
      if constexpr (!ZC) {
        g.dz[q] = geo.dz3[k * n2 + c];
        g.dzi[q] = geo.dzi[(k + 1) * n2 + c];
        g.wet[q] = kb + q + 1 < nz && geo.m3[(k + 1 < nz ? k + 1 : k) * n2 + c] != 0;
      }
    }
  };
  Ahead cur, nxt;
  load(0, cur);
  double kh_t = Kh[c], c_prev = 0.0, da = 0.0, ds = 0.0;
  double idzi_t;
  bool wet;
  if constexpr (ZC) {
    idzi_t = ca.inv(0);
    wet = nwc > 0;
  } else {
    idzi_t = safe_inv(geo.dzi[c]);
    wet = geo.m3[c] != 0;
  }
  for (int kb = 0; kb < nz; kb += W) {
    if (kb + W < nz) load(kb + W, nxt);
#pragma unroll
    for (int q = 0; q < W; ++q) {
      const int k = kb + q;
      if (k >= nz) break;
      double inv, idzi_b;
      bool below;
      if constexpr (ZC) {
        inv = ca.inv(k);
        idzi_b = k + 1 == nz ? inv : ca.idzi(k + 1);
        below = k + 1 < nwc;
      } else {
        inv = safe_inv(cur.dz[q]);
        idzi_b = safe_inv(cur.dzi[q]);
        below = cur.wet[q];
      }
      double sub, sup, den;
      matrix_row(p, k, inv, kh_t, cur.kh[q], idzi_t, idzi_b, wet, below, p.thv_dt * 0.0, c_prev,
                 sub, sup, den);
      const Divisor<double> by_den(den);
      const double cs = by_den(sup);
      da = k == 0 ? by_den(cur.a[q]) : by_den(cur.a[q] - sub * da);
      ds = k == 0 ? by_den(cur.s[q]) : by_den(cur.s[q] - sub * ds);
      const long long t = k * n2 + c;
      cst[t] = cs;
      A[t] = da;
      if (ts) S_out[t] = ds;
      c_prev = cs;
      kh_t = cur.kh[q];
      idzi_t = idzi_b;
      wet = below;
    }
    cur = nxt;
  }
  // back-substitution, W levels loaded ahead
  struct Back {
    double a[W], s[W], cs[W], z[W];
    bool wet[W];
  };
  auto load_back = [&](int kt, Back& g) {  // levels kt, kt - 1, ...
#pragma unroll
    for (int q = 0; q < W; ++q) {
      const long long k = kt - q > 0 ? kt - q : 0;
      g.a[q] = A[k * n2 + c];
      g.s[q] = ts ? S_out[k * n2 + c] : 0.0;
      g.cs[q] = cst[k * n2 + c];
      if constexpr (ZC) {
        g.z[q] = cg_zc_at(zs[k], p.dzr, nwc, hbc, bot, (int)k);
        g.wet[q] = k < nwc;
      } else {
        g.z[q] = ts ? geo.zc[k * n2 + c] : 0.0;
        g.wet[q] = geo.m3[k * n2 + c] != 0;
      }
    }
  };
  Back bc, bn;
  load_back(nz - 1, bc);
  double xa = 0.0, xs = 0.0;
  for (int kt = nz - 1; kt >= 0; kt -= W) {
    if (kt - W >= 0) load_back(kt - W, bn);
#pragma unroll
    for (int q = 0; q < W; ++q) {
      const int k = kt - q;
      if (k < 0) break;
      const long long t = k * n2 + c;
      const double mm = bc.wet[q] ? 1.0 : 0.0;
      xa = k == nz - 1 ? bc.a[q] : bc.a[q] - bc.cs[q] * xa;
      A[t] = xa * mm;
      if (ts) {
        xs = k == nz - 1 ? bc.s[q] : bc.s[q] - bc.cs[q] * xs;
        S_out[t] = xs * mm;
        const double bb = p.eos_mixed ? buoyancy_mixed(p, xa * mm, xs * mm, bc.z[q])
                                      : buoyancy(p, xa * mm, xs * mm, bc.z[q]);
        b_out[t] = bb * mm;
      }
    }
    bc = bn;
  }
}

// ------------------------------------------------- explicit momentum terms
// Staged tile of one level for one velocity component A (u or v): A with a
// 2-cell halo and the other component on the face points around the tile
// (two buffers: level k + 1 lands while level k is read). Row and column 0 of
// the other component are the tile's own first row and column for v's faces
// (A = v) shifted one column west, for u's (A = u) one row south.
template <class R>
struct MomLds {
  R a[SY][SX];
  R o[TY + 1][TX + 1];
};

// The level's face masks, for geometry read from the arrays: A's with the
// halo, the other component's on the own points and one row / column before.
struct MomMaskLds {
  uint8_t ma[SY][SX];
  uint8_t mo[TY + 1][TX + 1];
};

constexpr int MS_O = ((TY + 1) * (TX + 1) + TILE_THREADS - 1) / TILE_THREADS;  // +1 slots

// Level-k staging held in registers between its global loads and its LDS
// stores or its use, and this thread's plane offsets.
template <class R>
struct MomRegs {
  R a[ST_H], o[MS_O];
  double phi[2], b[2];  // at the own point and the next one along the component's direction
  R w[2];               // on interface k + 1
};
struct MomGeoRegs {  // geometry read from the arrays
  uint8_t ma[ST_H], mo[MS_O];
  double zc[2];
};

// Plane indexes of this thread's slots of the other component's points.
struct MomOffs {
  unsigned o[MS_O];
};
template <int COMP>
__device__ __forceinline__ MomOffs mom_offsets(int tid, int i0, int j0, int nx, int ny) {
  MomOffs F;
#pragma unroll
  for (int q = 0; q < MS_O; ++q) {
    const int t = tid + q * TILE_THREADS;
    const int tt = t < (TY + 1) * (TX + 1) ? t : tid;
    const int lx = tt % (TX + 1), ly = tt / (TX + 1);
    F.o[q] = (unsigned)(pmod(j0 + ly - (COMP == 0 ? 1 : 0), ny) * nx +
                        pmod(i0 + lx - (COMP == 0 ? 0 : 1), nx));
  }
  return F;
}

// Vertical momentum flux on interface kk of the column: wb times the
// interface value of the advected velocity (advection_v06.py:95-99,
// advection.py:75-79); f* hold the velocity at kk-2..kk+1, m* the wet flags
// of kk-2 and kk+1.
template <class R, bool TVD>
__device__ __forceinline__ R mom_flux_z(int adv, int kk, int nz, R wb, R far_up, R above, R below,
                                        R far_dn, bool mup, bool mdn) {
  R f;
  if (!TVD && adv == ADV_CENTRED2) {
    f = wb * R(0.5) * (above + below);
  } else {
    const bool hu = kk >= 2 && mup;
    const bool hd = kk <= nz - 2 && mdn;
    f = wb * kappa_face_z<R>(kk >= 2 ? far_up : R(0), above, below,
                             kk <= nz - 2 ? far_dn : R(0), wb, hu, hd,
                             TVD || adv == ADV_UP3_TVD);
  }
  return kk <= 0 || kk >= nz ? R(0) : f;
}

// Wet flags that the values of component COMP on the x-face (axis 0) or
// y-face (axis 1) after column (j, i) need: A's points before and beyond the
// face's two, and the face's own gradient mask. Each is k < a number of
// levels, kept in a register for the whole march (bytes: before, beyond, own;
// a count is at most 255).
template <int COMP>
__device__ __forceinline__ unsigned mom_face_wet(const Geo& geo, int axis, int j, int i, int ny,
                                                 int nx) {
  const int j0 = pmod(j, ny), i0 = pmod(i, nx);
  const int jm = axis ? pmod(j - 1, ny) : j0, j2 = axis ? pmod(j + 2, ny) : j0;
  const int im = axis ? i0 : pmod(i - 1, nx), i2 = axis ? i0 : pmod(i + 2, nx);
  return (unsigned)face_levels(geo, COMP, jm, im, ny, nx) |
         (unsigned)face_levels(geo, COMP, j2, i2, ny, nx) << 8 |
         (unsigned)face_levels(geo, axis, j0, i0, ny, nx) << 16;
}

// The explicit terms of one velocity component (COMP 0: u, 1: v) of the tile
// with origin (i0, j0) on the levels [k0, k1).
template <class R, bool ZC, bool TVD, int COMP, class Mask>
__device__ __forceinline__ void momentum_component(
    const Dims& d, const StepParams& p, const Geo& geo, int i0, int j0, int k0, int k1,
    MomLds<R>* LB, Mask* MB, FaceLds<R>& F, const double* __restrict__ A,
    const double* __restrict__ O, const double* __restrict__ b, const double* __restrict__ phi,
    const double* __restrict__ w, const double* __restrict__ Km, const double* __restrict__ zs,
    double* __restrict__ pg, double* __restrict__ dzo, double* __restrict__ st) {
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  const long long n2 = d.n2;
  const int tid = threadIdx.x;
  const int tx = tid % TX, ty = tid / TX;
  const int i = i0 + tx, j = j0 + ty;
  const bool active = i < nx && j < ny;
  // momentum keeps the centred form for upwind1; TVD: the scheme is known at
  // compile time, so that a level's face values are one straight line
  const int adv = TVD ? (int)ADV_UP3_TVD
                      : (p.advection == ADV_UPWIND1 ? (int)ADV_CENTRED2 : p.advection);
  const bool lim = adv == ADV_UP3_TVD;
  // the tile's west faces and south faces are formed by two different waves
  const int xe = tid - EDGE_X, ye = tid - EDGE_Y;
  const Divisor<R> by_dx = uniform_divisor<R>(p.dx), by_dy = uniform_divisor<R>(p.dy),
                   by_dz = uniform_divisor<R>(p.dz_nom);
  const Divisor<double> by_ds = uniform_divisor<double>(COMP == 0 ? p.dx : p.dy);
  const uint8_t* mA = COMP == 0 ? geo.m3u : geo.m3v;
  const uint8_t* mO = COMP == 0 ? geo.m3v : geo.m3u;
  const double* dzf = COMP == 0 ? geo.dz3u : geo.dz3v;
  const double* tau = COMP == 0 ? geo.tau_u : geo.tau_v;

  // plane indexes of the own point and of the next one along the component's
  // direction (clamped into the grid for the lanes beyond it)
  const int jc = pmod(j, ny), ic = pmod(i, nx);
  const int cc = jc * nx + ic;
  const int c1 = COMP == 0 ? jc * nx + pmod(i + 1, nx) : pmod(j + 1, ny) * nx + ic;
  const unsigned b0 = 8u * (unsigned)cc, b1 = 8u * (unsigned)c1;

  MomRegs<R> RG;
  MomGeoRegs GG;
  const HaloOffs HO = halo_offsets(tid, i0, j0, nx, ny);
  const MomOffs MO = mom_offsets<COMP>(tid, i0, j0, nx, ny);
  auto load = [&](long long o) {
#pragma unroll
    for (int q = 0; q < ST_H; ++q) {
      RG.a[q] = (R)at_byte(A + o, 8u * HO.h[q]);
      if constexpr (!ZC) GG.ma[q] = at_byte(mA + o, HO.h[q]);
    }
#pragma unroll
    for (int q = 0; q < MS_O; ++q) {
      RG.o[q] = (R)at_byte(O + o, 8u * MO.o[q]);
      if constexpr (!ZC) GG.mo[q] = at_byte(mO + o, MO.o[q]);
    }
    RG.phi[0] = at_byte(phi + o, b0);
    RG.phi[1] = at_byte(phi + o, b1);
    RG.b[0] = at_byte(b + o, b0);
    RG.b[1] = at_byte(b + o, b1);
    RG.w[0] = (R)at_byte(w + o + n2, b0);
    RG.w[1] = (R)at_byte(w + o + n2, b1);
    if constexpr (!ZC) {
      GG.zc[0] = at_byte(geo.zc + o, b0);
      GG.zc[1] = at_byte(geo.zc + o, b1);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < ST_H; ++q) {
      const int t = tid + q * TILE_THREADS;
      if (t < SX * SY) {
        LB[buf].a[t / SX][t % SX] = RG.a[q];
        if constexpr (!ZC) MB[buf].ma[t / SX][t % SX] = GG.ma[q];
      }
    }
#pragma unroll
    for (int q = 0; q < MS_O; ++q) {
      const int t = tid + q * TILE_THREADS;
      if (t < (TY + 1) * (TX + 1)) {
        LB[buf].o[t / (TX + 1)][t % (TX + 1)] = RG.o[q];
        if constexpr (!ZC) MB[buf].mo[t / (TX + 1)][t % (TX + 1)] = GG.mo[q];
      }
    }
  };
  load((long long)k0 * n2);

  // the column form, in registers: wet levels of the east, north and edge
  // faces' points, the own A point's column, and the cell's and its neighbour's
  unsigned xw = 0, yw = 0, exw = 0, eyw = 0;
  InvCol ca{};
  int nw0 = 0, nw1 = 0, na = 0;
  double hb0 = 0.0, hb1 = 0.0, bot0 = 0.0, bot1 = 0.0;
  if constexpr (ZC) {
    xw = mom_face_wet<COMP>(geo, 0, j, i, ny, nx);
    yw = mom_face_wet<COMP>(geo, 1, j, i, ny, nx);
    if (xe >= 0 && xe < TY) exw = mom_face_wet<COMP>(geo, 0, j0 + xe, i0 - 1, ny, nx);
    if (ye >= 0 && ye < TX) eyw = mom_face_wet<COMP>(geo, 1, j0 - 1, i0 + ye, ny, nx);
    na = (int)((COMP == 0 ? xw : yw) >> 16);
    nw0 = geo.nw[cc];
    nw1 = geo.nw[c1];
    hb0 = geo.hb[cc];
    hb1 = geo.hb[c1];
    bot0 = nw0 > 0 ? zs[nw0 - 1] + hb0 : 0.0;
    bot1 = nw1 > 0 ? zs[nw1 - 1] + hb1 : 0.0;
    const double full = uniform_value(face_value(p.face_rule, p.dzr, p.dzr));
    const double last = na > 0 ? face_value(p.face_rule, cg_dz(p.dzr, nw0, hb0, na - 1),
                                            cg_dz(p.dzr, nw1, hb1, na - 1))
                               : 0.0;
    ca = inv_col(na, full, last);
  }
  auto own_wet = [&](int kk) -> bool {  // the own A point
    if constexpr (ZC) return kk < na;
    else return at_byte(mA + kk * n2, (unsigned)cc) != 0;
  };
  auto cell_wet = [&](int kk) -> bool {
    if constexpr (ZC) return kk < nw0;
    else return at_byte(geo.m3 + kk * n2, (unsigned)cc) != 0;
  };
  auto idz = [&](int kk) -> double {  // 1 / A's spacing on interface kk, 1 <= kk < nz
    if constexpr (ZC) return ca.idzi(kk);
    else return safe_inv(0.5 * (at_byte(dzf + (kk - 1) * n2, b0) + at_byte(dzf + kk * n2, b0)));
  };
  auto inv = [&](int kk) -> double {  // 1 / A's thickness
    if constexpr (ZC) return ca.inv(kk);
    else return safe_inv(at_byte(dzf + kk * n2, b0));
  };

  store(0);
  // own-column window of A at k-2..k+2; its wet flags follow from the level
  // count, or are bits of one register (bit q: level k-2+q)
  double a5[5];
  unsigned m5 = 0;
  bool cw0 = k0 >= 1 && cell_wet(k0 - 1), cw1 = cell_wet(k0);  // cells k-1, k
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const int kk = k0 + q - 2;
    const bool in = kk >= 0 && kk < nz;
    a5[q] = in ? at_byte(A + kk * n2, b0) : 0.0;
    if constexpr (!ZC)
      if (in && own_wet(kk)) m5 |= 1u << q;
  }
  auto wet_at = [&](int k, int q) -> bool {  // A's point at level k-2+q
    if constexpr (ZC) return k + q - 2 >= 0 && k + q - 2 < na;
    else return (m5 >> q & 1u) != 0;
  };
  double km_k = at_byte(Km + k0 * n2, b0);  // K_m and 1 / spacing on interface k
  double idz_k = k0 > 0 ? idz(k0) : 0.0;
  R fz_top = R(0);
  if (k0 > 0 && adv != ADV_NONE) {
    // the flux through this range's top interface, which the range above
    // forms as its bottom one: the same operands, the same bits
    const double* wk = w + (long long)k0 * n2;
    fz_top = mom_flux_z<R, TVD>(adv, k0, nz, R(0.5) * ((R)at_byte(wk, b0) + (R)at_byte(wk, b1)),
                           R(a5[0]), R(a5[1]), R(a5[2]), R(a5[3]), wet_at(k0, 0),
                           wet_at(k0, 3));
  }
  __syncthreads();
  for (int k = k0; k < k1; ++k) {
    const long long o = (long long)k * n2;
    const MomLds<R>& L = LB[(k - k0) & 1];
    // level k's cell-pass inputs, loaded during level k - 1, before the loads
    // of level k + 1 reuse the registers
    const double phi0 = RG.phi[0], phi1 = RG.phi[1], bb0 = RG.b[0], bb1 = RG.b[1];
    const R wb = R(0.5) * (RG.w[0] + RG.w[1]);
    double zc0, zc1;
    if constexpr (ZC) {
      zc0 = cg_zc_at(zs[k], p.dzr, nw0, hb0, bot0, k);
      zc1 = cg_zc_at(zs[k], p.dzr, nw1, hb1, bot1, k);
    } else {
      zc0 = GG.zc[0];
      zc1 = GG.zc[1];
    }
    // the own column's viscosity below level k, issued before the face pass
    const double km_k1 = at_byte(Km + o + n2, b0);
    if (k + 1 < k1) load(o + n2);
    const double a_k3 = k + 3 < nz ? at_byte(A + o + 3 * n2, b0) : 0.0;  // the window's next
    // ---- faces
    {
      // the face's wet flags from its packed level counts or the mask tile:
      // (ym, xm), (y2, x2) the far points, (yy, xx) the point before the face
      auto flags = [&](unsigned f, int axis, int yy, int xx, bool* m) {
        if constexpr (ZC) {
          m[0] = k < (int)(f & 255u);
          m[1] = k < (int)(f >> 8 & 255u);
          m[2] = k < (int)(f >> 16);
        } else {
          const MomMaskLds& M = MB[(k - k0) & 1];
          m[0] = (axis ? M.ma[yy - 1][xx] : M.ma[yy][xx - 1]) != 0;
          m[1] = (axis ? M.ma[yy + 2][xx] : M.ma[yy][xx + 2]) != 0;
          // the gradient mask: A's own for the face along A, the other's across
          m[2] = axis == COMP ? M.ma[yy][xx] != 0
                 : COMP == 0  ? M.mo[yy - HALO + 1][xx - HALO] != 0
                              : M.mo[yy - HALO][xx - HALO + 1] != 0;
        }
      };
      // x-face q of row r (between columns q-1 and q)
      auto xface = [&](int r, int q, unsigned f) {
        const int yy = r + HALO, x0 = q - 1 + HALO;  // x0: the column west of the face
        bool m[3];
        flags(f, 0, yy, x0, m);
        const R a0 = L.a[yy][x0], a1 = L.a[yy][x0 + 1];
        if (adv != ADV_NONE) {
          const R vel = COMP == 0 ? R(0.5) * (a0 + a1) : R(0.5) * (L.o[r][q] + L.o[r + 1][q]);
          if (adv == ADV_CENTRED2)
            F.fx[r][q] = COMP == 0 ? vel * vel : vel * (R(0.5) * (a0 + a1));
          else
            F.fx[r][q] = vel * kappa_face<R>(L.a[yy][x0 - 1], a0, a1, L.a[yy][x0 + 2], vel, m[0],
                                             m[1], lim);
        }
        F.gx[r][q] = by_dx((m[2] ? R(1) : R(0)) * (a1 - a0));
      };
      // y-face q of column r (between rows q-1 and q)
      auto yface = [&](int q, int r, unsigned f) {
        const int xx = r + HALO, y0 = q - 1 + HALO;  // y0: the row south of the face
        bool m[3];
        flags(f, 1, y0, xx, m);
        const R a0 = L.a[y0][xx], a1 = L.a[y0 + 1][xx];
        if (adv != ADV_NONE) {
          const R vel = COMP == 0 ? R(0.5) * (L.o[q][r] + L.o[q][r + 1]) : R(0.5) * (a0 + a1);
          if (adv == ADV_CENTRED2)
            F.fy[q][r] = COMP == 0 ? vel * (R(0.5) * (a0 + a1)) : vel * vel;
          else
            F.fy[q][r] = vel * kappa_face<R>(L.a[y0 - 1][xx], a0, a1, L.a[y0 + 2][xx], vel, m[0],
                                             m[1], lim);
        }
        F.gy[q][r] = by_dy((m[2] ? R(1) : R(0)) * (a1 - a0));
      };
      xface(ty, tx + 1, xw);
      yface(ty + 1, tx, yw);
      if (xe >= 0 && xe < TY) xface(xe, 0, exw);
      if (ye >= 0 && ye < TX) yface(0, ye, eyw);
    }
    __syncthreads();
    {
      const double m_c = wet_at(k, 2) ? 1.0 : 0.0;
      // pressure gradient at the face depth (model3d_v05.py:195-230)
      double pg_k;
      if (p.pgf_correction) {
        const double zf = 0.5 * (zc0 + zc1);
        const double left = phi0 + bb0 * (zf - zc0);
        const double right = phi1 + bb1 * (zf - zc1);
        pg_k = by_ds(m_c * (right - left));
      } else {
        pg_k = by_ds(m_c * (phi1 - phi0)) * m_c;
      }
      // explicit vertical diffusion with surface stress and bottom drag
      const bool lower = k + 1 < nz;
      const bool cw2 = lower && cell_wet(k + 1);
      const double idz_k1 = lower ? idz(k + 1) : 0.0;
      const double iv = inv(k);
      const double tau_k = k == 0 ? at_byte(tau, b0) : 0.0;
      const double dz_k = explicit_diffusion_inv(k, nz, a5[1], a5[2], a5[3], idz_k, idz_k1, iv,
                                                 cw0, cw1, cw2, km_k, km_k1, tau_k,
                                                 p.bottom_drag);
      // advection and horizontal viscosity
      double ex = 0.0;
      if (adv != ADV_NONE) {
        const R ax = by_dx(F.fx[ty][tx + 1] - F.fx[ty][tx]);
        const R ay = by_dy(F.fy[ty + 1][tx] - F.fy[ty][tx]);
        // vertical fluxes: the top one is the bottom one of the level above
        const R fz_bot = mom_flux_z<R, TVD>(adv, k + 1, nz, wb, R(a5[1]), R(a5[2]), R(a5[3]),
                                       R(a5[4]), wet_at(k, 1), wet_at(k, 4));
        const R az = by_dz(fz_top - fz_bot);
        fz_top = fz_bot;
        ex = ex - (double)((ax + ay + az) * R(m_c));
      }
      if (p.has_A_h)
        ex = ex + p.A_h * (double)(R(m_c) * (by_dx(F.gx[ty][tx + 1] - F.gx[ty][tx]) +
                                             by_dy(F.gy[ty + 1][tx] - F.gy[ty][tx])));
      double s0 = 0.0;
      if (k == 0) s0 = p.thv_dt * tau_k * iv;
      if (active) {
        put_byte(pg + o, b0, pg_k);
        put_byte(dzo + o, b0, dz_k);
        put_byte(st + o, b0, s0 + p.dt * ex);
      }
      // advance the windows
      km_k = km_k1;
      idz_k = idz_k1;
      cw0 = cw1;
      cw1 = cw2;
#pragma unroll
      for (int q = 0; q < 4; ++q) a5[q] = a5[q + 1];
      a5[4] = a_k3;
      if constexpr (!ZC) m5 = m5 >> 1 | (k + 3 < nz && own_wet(k + 3) ? 16u : 0u);
    }
    if (k + 1 < k1) store((k + 1 - k0) & 1);
    __syncthreads();
  }
}

// The step's explicit momentum terms (libs/core/model3d_v05.py:352-370): the
// pressure gradient, the explicit vertical diffusion, and the stress,
// advection and viscosity of u and v; same outputs as k_momentum_explicit.
// One workgroup marches one component of one tile down the levels [k0, k0 +
// nk). Staging is double-buffered (level k + 1 loads in flight while level k
// is computed) and every horizontal face flux is formed once. R is the type
// of the advective fluxes and the A_h gradients (double: bitwise the
// reference; float: the mixed step); the rest stays fp64. ZC: the static
// z-level geometry in column form (masks, inverse thicknesses and centre
// depths from the columns' wet-level counts and deepest thicknesses, in
// registers; the same bits).
// Bound by the latency of its fp64 chains (about 600 VALU instructions per
// cell for both components, five divisions in a row on a face), so what counts
// is waves in flight without spills and straight-line code: u and v in
// workgroups of their own (159 registers against 230 for both: 3 waves per
// SIMD), the scheme a template argument (the face values of a level
// interleave), the levels cut into ranges (1024 tiles of 512 x 512 on 768
// resident workgroups left a third of the second round idle, and 64 tiles of
// 128 x 128 three quarters of the chip). Measured per launch, before -> now:
// 128 x 4 x 20 132 -> 11 us, 128 x 128 x 30 204 -> 37, 512 x 512 x 40 600 ->
// 377, 1000 x 1000 x 30 1487 -> 1097. At 4 waves per SIMD it spilled 30
// registers and took 478 us at 512 x 512 x 40 (364 at 3).
template <class R, bool ZC, bool TVD>
__global__ __launch_bounds__(TILE_THREADS) __attribute__((amdgpu_waves_per_eu(3))) void k_momentum_explicit_tiled(
    Dims d, StepParams p, Geo geo, int nk, const double* __restrict__ u,
    const double* __restrict__ v, const double* __restrict__ b, const double* __restrict__ phi,
    const double* __restrict__ w, const double* __restrict__ Km, const double* __restrict__ zs,
    double* __restrict__ pgx, double* __restrict__ pgy, double* __restrict__ dzu,
    double* __restrict__ dzv, double* __restrict__ stu, double* __restrict__ stv) {
  __shared__ MomLds<R> LB[2];
  __shared__ FaceLds<R> F;
  __shared__ std::conditional_t<ZC, NoTile, MomMaskLds> MB[2];
  const BlockTile T = xcd_block((d.nx + TX - 1) / TX, (d.ny + TY - 1) / TY, 2);
  const int k0 = T.z * nk;
  const int k1 = k0 + nk < d.nz ? k0 + nk : d.nz;
  if (T.part == 0)
    momentum_component<R, ZC, TVD, 0>(d, p, geo, T.x * TX, T.y * TY, k0, k1, LB, MB, F, u, v, b,
                                 phi, w, Km, zs, pgx, dzu, stu);
  else
    momentum_component<R, ZC, TVD, 1>(d, p, geo, T.x * TX, T.y * TY, k0, k1, LB, MB, F, v, u, b,
                                 phi, w, Km, zs, pgy, dzv, stv);
}

// Levels per workgroup of a tiled march: all of them where the tiles alone give `target`
// workgroups, else as few as make up that number (each range of levels reads the two levels
// above and below it again and forms its top interface's fluxes a second time).
int levels_per_block(long long tiles, int nz, long long target) {
  const long long parts = tiles >= target ? 1 : (target + tiles - 1) / tiles;
  const int n = (int)((nz + parts - 1) / parts);
  return n < 1 ? 1 : n;
}

void launch_tracers(bool mixed, hipStream_t s, Dims d, StepParams p, Geo geo, const double* T,
                    const double* S, const double* b, const double* u, const double* v,
                    const double* w, const double* Kh, double* cst, double* T_out,
                    double* S_out, double* b_out) {
  const int gx = (d.nx + TX - 1) / TX, gy = (d.ny + TY - 1) / TY;
  const int parts = p.tracers_ts ? 2 : 1;
  // 1024 workgroups, as many as are resident (4 per CU). Measured with 1024 / 2048 / 4096,
  // both tracer kernels: 128 x 128 x 30 63 / 68 / 77 us, 256 x 256 x 30 112 / 119 / 129,
  // 512 x 512 x 40 and 1000 x 1000 x 30 equal.
  const int nk = levels_per_block((long long)parts * gx * gy, d.nz, 1024);
  const unsigned grid = (unsigned)parts * gx * gy * ((d.nz + nk - 1) / nk);
  const bool tvd = p.advection == ADV_UP3_TVD;
  auto rhs = [&](auto kernel) {
    kernel<<<grid, TILE_THREADS, 0, s>>>(d, p, geo, nk, T, S, b, u, v, w, Kh, T_out, S_out,
                                         b_out);
  };
  auto solve = [&](auto kernel) {
    const unsigned nb = (unsigned)((d.n2 + SOLVE_THREADS - 1) / SOLVE_THREADS);
    kernel<<<nb, SOLVE_THREADS, 0, s>>>(d, p, geo, geo.zs, Kh, cst, T_out, S_out, b_out);
  };
  if (p.zcol) {
    if (mixed) rhs(tvd ? k_tracer_rhs<float, true, true> : k_tracer_rhs<float, true, false>);
    else rhs(tvd ? k_tracer_rhs<double, true, true> : k_tracer_rhs<double, true, false>);
    solve(k_tracer_solve<true>);
  } else {
    if (mixed) rhs(k_tracer_rhs<float, false, false>);
    else rhs(tvd ? k_tracer_rhs<double, false, true> : k_tracer_rhs<double, false, false>);
    solve(k_tracer_solve<false>);
  }
}

void launch_momentum_explicit_tiled(bool mixed, hipStream_t s, Dims d, StepParams p, Geo geo,
                                    const double* u, const double* v, const double* b,
                                    const double* phi, const double* w, const double* Km,
                                    double* pgx, double* pgy, double* dzu, double* dzv,
                                    double* stu, double* stv) {
  const int gx = (d.nx + TX - 1) / TX, gy = (d.ny + TY - 1) / TY;
  // 2048 workgroups: 768 are resident at a time (3 per CU). Measured with 2048 / 4096 / 8192:
  // 128 x 128 x 30 37 / 47 / 47 us, 512 x 512 x 40 364 / 366 / 384, 1000 x 1000 x 30 1069 /
  // 1083 / 1116; 128 x 4 x 20 (one level each) 11 us in all three.
  const int nk = levels_per_block(2LL * gx * gy, d.nz, 2048);
  const unsigned grid = 2u * gx * gy * ((d.nz + nk - 1) / nk);
  const bool tvd = p.advection == ADV_UP3_TVD;
  auto go = [&](auto kernel) {
    kernel<<<grid, TILE_THREADS, 0, s>>>(d, p, geo, nk, u, v, b, phi, w, Km, geo.zs, pgx, pgy,
                                         dzu, dzv, stu, stv);
  };
  if (p.zcol) {
    if (mixed) go(tvd ? k_momentum_explicit_tiled<float, true, true>
                      : k_momentum_explicit_tiled<float, true, false>);
    else go(tvd ? k_momentum_explicit_tiled<double, true, true>
                : k_momentum_explicit_tiled<double, true, false>);
  } else if (mixed) {
    go(k_momentum_explicit_tiled<float, false, false>);
  } else {
    go(tvd ? k_momentum_explicit_tiled<double, false, true>
           : k_momentum_explicit_tiled<double, false, false>);
  }
}

}  // namespace hoc
