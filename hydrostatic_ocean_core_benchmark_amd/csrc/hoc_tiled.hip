// LDS-tiled column kernels ("2.5D"): a workgroup owns a TX x TY tile of
// columns and marches down the levels. At each level the fields that enter
// horizontal stencils are staged once in LDS with a 2-cell periodic halo,
// so every value is read from HBM about once instead of once per stencil
// point; the column's own vertical neighbours stay in a register window.
// Arithmetic and operand order are those of the untiled kernels (and of the
// reference's NumPy expressions), so the results are bitwise the same.
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

// Staged tile of one level in the flux type R: what the face pass and the
// cell pass both read (double-buffered, so level k + 1 lands while level k
// is still read) ...
template <class R>
struct TileLds {
  R c[2][SY][SX];           // the tracers (T, S) or b, with halo
  uint8_t m[SY][SX];        // mask3 with halo
  uint8_t mu[TY][TX + 1];   // mask3u
  uint8_t mv[TY + 1][TX];   // mask3v
};

// ... and what only the face pass reads (one buffer: the barrier after the
// face pass ends its reads before level k + 1 is stored).
template <class R>
struct VelLds {
  R u[TY][TX + 1];          // u at i-1 .. i
  R v[TY + 1][TX];          // v at j-1 .. j
  R du[TY][TX + 1];         // dz3u
  R dv[TY + 1][TX];         // dz3v
};

// Advective face fluxes dz_f u_f c_f of one level, each computed once, on
// the x-faces (index q: between tile columns q-1 and q) and y-faces
// (between rows q-1 and q), for both tracers. The K_h face gradients are
// formed by the cell that uses them, from the staged tile (each interior
// gradient twice, from the same operands): with the single velocity buffer
// this holds a workgroup to 33 KB of LDS, so four fit on a CU.
template <class R>
struct FaceLds {
  R fx[2][TY][TX + 1];
  R fy[2][TY + 1][TX];
};

// K_h gradient mask_f (c_1 - c_0) / d across one face of the staged tile.
template <class R>
__device__ __forceinline__ R face_grad(uint8_t mf, R c0, R c1, double d) {
  return R(mk(mf)) * (c1 - c0) / R(d);
}

// Level-k staging of one tile held in registers between its global loads
// and its LDS stores, so the loads of level k + 1 are in flight while
// level k is computed (two LDS buffers, one barrier per level).
constexpr int ST_C = (SX * SY + TILE_THREADS - 1) / TILE_THREADS;        // tracer + mask slots
constexpr int ST_U = (TY * (TX + 1) + TILE_THREADS - 1) / TILE_THREADS;  // u-face slots
constexpr int ST_V = ((TY + 1) * TX + TILE_THREADS - 1) / TILE_THREADS;  // v-face slots

template <class R>
struct TileRegs {
  R c0[ST_C], c1[ST_C];
  uint8_t m[ST_C];
  R u[ST_U], du[ST_U];
  uint8_t mu[ST_U];
  R v[ST_V], dv[ST_V];
  uint8_t mv[ST_V];
};

// Plane offsets of this thread's staging slots (independent of k; -1: no slot).
struct TileOffs {
  int c[ST_C], u[ST_U], v[ST_V];
};

__device__ __forceinline__ TileOffs tile_offsets(int tid, int i0, int j0, int nx, int ny) {
  TileOffs F;
#pragma unroll
  for (int q = 0; q < ST_C; ++q) {
    const int t = tid + q * TILE_THREADS;
    F.c[q] = t < SX * SY ? pmod(j0 + t / SX - HALO, ny) * nx + pmod(i0 + t % SX - HALO, nx) : -1;
  }
#pragma unroll
  for (int q = 0; q < ST_U; ++q) {
    const int t = tid + q * TILE_THREADS;
    F.u[q] = t < TY * (TX + 1) ? pmod(j0 + t / (TX + 1), ny) * nx + pmod(i0 + t % (TX + 1) - 1, nx)
                               : -1;
  }
#pragma unroll
  for (int q = 0; q < ST_V; ++q) {
    const int t = tid + q * TILE_THREADS;
    F.v[q] = t < (TY + 1) * TX ? pmod(j0 + t / TX - 1, ny) * nx + pmod(i0 + t % TX, nx) : -1;
  }
  return F;
}

template <class RT>
__device__ __forceinline__ void tile_load(TileRegs<RT>& R, const TileOffs& F, long long o, bool ts,
                                          const double* A, const double* S, const double* u,
                                          const double* v, const Geo& geo) {
#pragma unroll
  for (int q = 0; q < ST_C; ++q) {
    if (F.c[q] >= 0) {
      const long long g = o + F.c[q];
      R.c0[q] = (RT)A[g];
      R.c1[q] = ts ? (RT)S[g] : RT(0);
      R.m[q] = geo.m3[g];
    }
  }
#pragma unroll
  for (int q = 0; q < ST_U; ++q) {
    if (F.u[q] >= 0) {
      const long long g = o + F.u[q];
      R.u[q] = (RT)u[g];
      R.du[q] = (RT)geo.dz3u[g];
      R.mu[q] = geo.m3u[g];
    }
  }
#pragma unroll
  for (int q = 0; q < ST_V; ++q) {
    if (F.v[q] >= 0) {
      const long long g = o + F.v[q];
      R.v[q] = (RT)v[g];
      R.dv[q] = (RT)geo.dz3v[g];
      R.mv[q] = geo.m3v[g];
    }
  }
}

template <class RT>
__device__ __forceinline__ void tile_store(TileLds<RT>& L, VelLds<RT>& V, const TileRegs<RT>& R,
                                           int tid) {
#pragma unroll
  for (int q = 0; q < ST_C; ++q) {
    const int t = tid + q * TILE_THREADS;
    if (t < SX * SY) {
      const int lx = t % SX, ly = t / SX;
      L.c[0][ly][lx] = R.c0[q];
      L.c[1][ly][lx] = R.c1[q];
      L.m[ly][lx] = R.m[q];
    }
  }
#pragma unroll
  for (int q = 0; q < ST_U; ++q) {
    const int t = tid + q * TILE_THREADS;
    if (t < TY * (TX + 1)) {
      const int lx = t % (TX + 1), ly = t / (TX + 1);
      V.u[ly][lx] = R.u[q];
      V.du[ly][lx] = R.du[q];
      L.mu[ly][lx] = R.mu[q];
    }
  }
#pragma unroll
  for (int q = 0; q < ST_V; ++q) {
    const int t = tid + q * TILE_THREADS;
    if (t < (TY + 1) * TX) {
      const int lx = t % TX, ly = t / TX;
      V.v[ly][lx] = R.v[q];
      V.dv[ly][lx] = R.dv[q];
      L.mv[ly][lx] = R.mv[q];
    }
  }
}

// Both tracers of the tile's columns: advection + K_h Laplacian + explicit
// part of the vertical diffusion + surface flux, the forward sweep on tri_b
// (d* parked in the outputs), then the back-substitution and the EOS
// (libs/core/model3d_v05.py:466-533). R is the type of the horizontal and
// vertical advective fluxes, the K_h gradients and the EOS: double for the
// plain step (bitwise the reference), float for the mixed step; the column
// update, the vertical diffusion and the tridiagonal solve stay fp64.
// The fp32-flux instantiation runs at 4 waves per SIMD (128 VGPRs): measured
// at 1024 x 1024 x 60, 3.65 ms per step against 4.19 ms at the compiler's
// default of 3 waves.
template <class R>
__global__ __launch_bounds__(TILE_THREADS)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 4 : 1))) void k_tracers_tiled(
    Dims d, StepParams p, Geo geo, const double* __restrict__ T, const double* __restrict__ S,
    const double* __restrict__ b, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ w, const double* __restrict__ Kh, double* __restrict__ cst,
    double* __restrict__ T_out, double* __restrict__ S_out, double* __restrict__ b_out) {
  __shared__ TileLds<R> LB[2];
  __shared__ VelLds<R> VL;
  __shared__ FaceLds<R> F;
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  const long long n2 = d.n2;
  const int tid = threadIdx.x;
  const int tx = tid % TX, ty = tid / TX;
  int bx, by;
  xcd_tile(bx, by);
  const int i0 = bx * TX, j0 = by * TY;
  const int i = i0 + tx, j = j0 + ty;
  const bool active = i < nx && j < ny;
  const long long c = active ? (long long)j * nx + i : 0;
  const bool ts = p.tracers_ts != 0;
  const int ntr = ts ? 2 : 1;
  const double* A = ts ? T : b;
  double* Ao = ts ? T_out : b_out;
  const double flux[2] = {ts ? p.flux_T : 0.0, p.flux_S};
  const int adv = p.advection;

  // own-column windows: tracer at k-2..k+2, mask3 at k-2..k+2
  double win[2][5];
  bool mw[5];
  for (int q = 0; q < 5; ++q) {
    win[0][q] = 0.0;
    win[1][q] = 0.0;
    mw[q] = false;
  }
  if (active) {
    for (int q = 2; q < 5; ++q) {
      const int kk = q - 2;
      if (kk < nz) {
        win[0][q] = A[kk * n2 + c];
        if (ts) win[1][q] = S[kk * n2 + c];
        mw[q] = geo.m3[kk * n2 + c] != 0;
      }
    }
  }
  double w_k = active ? w[c] : 0.0;
  double kh_k = active ? Kh[c] : 0.0;
  double dzi_k = active ? geo.dzi[c] : 0.0;
  R cf_top[2] = {R(0), R(0)};  // interface value at the top of level k
  double dprev[2] = {0.0, 0.0};
  double cb_prev = 0.0;  // c* of tri_b at the level above

  TileRegs<R> RG;
  const TileOffs TO = tile_offsets(tid, i0, j0, nx, ny);
  tile_load(RG, TO, 0, ts, A, S, u, v, geo);
  tile_store(LB[0], VL, RG, tid);
  __syncthreads();
  const bool has_adv = adv != ADV_NONE;
  for (int k = 0; k < nz; ++k) {
    const long long o = (long long)k * n2;
    const TileLds<R>& L = LB[k & 1];
    if (k + 1 < nz) tile_load(RG, TO, o + n2, ts, A, S, u, v, geo);
    // the own column's operands of level k, issued before the face pass so
    // their latency hides behind it
    double w_k1 = 0.0, kh_k1 = 0.0, dzi_k1 = 0.0, dz = 0.0;
    if (active) {
      w_k1 = w[o + n2 + c];
      kh_k1 = Kh[o + n2 + c];
      dzi_k1 = geo.dzi[o + n2 + c];
      dz = geo.dz3[o + c];
    }
    // ---- faces: the east and north face of every cell, plus the tile's
    // west column (8) and south row (32) of faces by threads 0..39
    {
      auto xface = [&](int fy_, int q) {
        const int cy = fy_ + HALO, c0x = q - 1 + HALO;
        const R vel = VL.u[fy_][q];
        const R ddu = VL.du[fy_][q];
        const bool wm = L.m[cy][c0x - 1] != 0, w2 = L.m[cy][c0x + 2] != 0;
        for (int r = 0; r < ntr; ++r) {
          const R(*C)[SX] = L.c[r];
          F.fx[r][fy_][q] = ddu * vel * tracer_face<R>(adv, C[cy][c0x - 1], C[cy][c0x],
                                                       C[cy][c0x + 1], C[cy][c0x + 2], vel, wm,
                                                       w2);
        }
      };
      auto yface = [&](int q, int fx_) {
        const int cx = fx_ + HALO, c0y = q - 1 + HALO;
        const R vel = VL.v[q][fx_];
        const R ddv = VL.dv[q][fx_];
        const bool wm = L.m[c0y - 1][cx] != 0, w2 = L.m[c0y + 2][cx] != 0;
        for (int r = 0; r < ntr; ++r) {
          const R(*C)[SX] = L.c[r];
          F.fy[r][q][fx_] = ddv * vel * tracer_face<R>(adv, C[c0y - 1][cx], C[c0y][cx],
                                                       C[c0y + 1][cx], C[c0y + 2][cx], vel, wm,
                                                       w2);
        }
      };
      if (has_adv) {
        xface(ty, tx + 1);
        yface(ty + 1, tx);
        if (tid < TY) xface(tid, 0);
        else if (tid < TY + TX) yface(0, tid - TY);
      }
    }
    __syncthreads();
    if (active) {
      // ---- own-column values for level k
      const double inv = safe_inv(dz);
      const bool m_k = mw[2];
      const bool bot_km1 = k >= 1 && mw[1] && !mw[2];          // cell k-1 is a bottom cell
      const bool bot_k = m_k && !((k + 1 < nz) && mw[3]);      // cell k is a bottom cell
      const int cx = tx + HALO, cy = ty + HALO;
      // row k of tri_b (K_h, no drag), factored here from the operands the
      // diffusion terms read anyway; c* parked in `cst` for the back-substitution
      double sub_k, den_k, cst_k;
      factor_row(p, k, inv, kh_k, kh_k1, safe_inv(dzi_k), safe_inv(dzi_k1), m_k,
                 (k + 1 < nz) && mw[3], p.thv_dt * 0.0, cb_prev, sub_k, den_k, cst_k);
      cst[o + c] = cst_k;
      cb_prev = cst_k;

      for (int r = 0; r < ntr; ++r) {
        const double cc = win[r][2];  // the tile's own cell, in fp64
        double tend = 0.0;
        if (!ts) tend = p.neg_N2 * (0.5 * (w_k + w_k1));
        if (has_adv) {
          const R hdiv = ((F.fx[r][ty][tx + 1] - F.fx[r][ty][tx]) / R(p.dx) +
                          (F.fy[r][ty + 1][tx] - F.fy[r][ty][tx]) / R(p.dy)) * R(inv);
          const R cft = (k == 0) ? R(win[r][2]) : cf_top[r];
          const R cfb = tracer_face_z<R>(adv, k + 1, nz, R(win[r][1]), R(win[r][2]),
                                         R(win[r][3]), R(win[r][4]), mw[1], mw[4], R(w_k1));
          cf_top[r] = cfb;
          const R vdiv = (R(w_k) * cft - R(w_k1) * cfb) * R(inv);
          tend = tend - (double)((hdiv + vdiv) * (m_k ? R(1) : R(0)));
        }
        if (p.has_K_h) {
          const R(*C)[SX] = L.c[r];
          const R ge = face_grad<R>(L.mu[ty][tx + 1], C[cy][cx], C[cy][cx + 1], p.dx);
          const R gw = face_grad<R>(L.mu[ty][tx], C[cy][cx - 1], C[cy][cx], p.dx);
          const R gn = face_grad<R>(L.mv[ty + 1][tx], C[cy][cx], C[cy + 1][cx], p.dy);
          const R gs = face_grad<R>(L.mv[ty][tx], C[cy - 1][cx], C[cy][cx], p.dy);
          tend = tend + p.K_h * (double)((m_k ? R(1) : R(0)) *
                                         ((ge - gw) / R(p.dx) + (gn - gs) / R(p.dy)));
        }
        // explicit vertical diffusion with the surface flux (vertical_var.py:80-106)
        double ft;
        if (k == 0) {
          ft = flux[r];
        } else {
          ft = kh_k * (win[r][1] - win[r][2]) * safe_inv(dzi_k);
          if (bot_km1) ft = 0.0;
        }
        double fb = 0.0;
        if (k + 1 < nz) {
          fb = kh_k1 * (win[r][2] - win[r][3]) * safe_inv(dzi_k1);
          if (bot_k) fb = 0.0;
        }
        const double out = (ft - fb) * inv;
        const double dr = 0.0 * win[r][2] * (bot_k ? 1.0 : 0.0);
        const double dzd = (out - dr * inv) * (m_k ? 1.0 : 0.0);
        double rhs = cc + p.dt * tend + p.c_dzd * dzd;
        if (k == 0) rhs = rhs + p.thv_dt * flux[r] * safe_inv(dz);
        const long long t = o + c;
        const double dd = (k == 0) ? rhs / den_k : (rhs - sub_k * dprev[r]) / den_k;
        dprev[r] = dd;
        (r == 0 ? Ao : S_out)[t] = dd;
      }
      // ---- advance the windows
      for (int r = 0; r < 2; ++r)
        for (int q = 0; q < 4; ++q) win[r][q] = win[r][q + 1];
      for (int q = 0; q < 4; ++q) mw[q] = mw[q + 1];
      const int kn = k + 3;
      if (kn < nz) {
        win[0][4] = A[(long long)kn * n2 + c];
        if (ts) win[1][4] = S[(long long)kn * n2 + c];
        mw[4] = geo.m3[(long long)kn * n2 + c] != 0;
      } else {
        win[0][4] = 0.0;
        win[1][4] = 0.0;
        mw[4] = false;
      }
      w_k = w_k1;
      kh_k = kh_k1;
      dzi_k = dzi_k1;
    }
    if (k + 1 < nz) tile_store(LB[(k + 1) & 1], VL, RG, tid);
    __syncthreads();
  }
  if (!active) return;
  // back-substitution with the next level's operands loaded one level ahead
  double xa = 0.0, xb = 0.0;
  long long t = (long long)(nz - 1) * n2 + c;
  double a_n = Ao[t], s_n = ts ? S_out[t] : 0.0, c_n = cst[t], z_n = ts ? geo.zc[t] : 0.0;
  uint8_t m_n = geo.m3[t];
  for (int k = nz - 1; k >= 0; --k) {
    const double a_k = a_n, s_k = s_n, c_k = c_n, z_k = z_n;
    const double mm = mk(m_n);
    const long long tk = t;
    if (k > 0) {
      t -= n2;
      a_n = Ao[t];
      if (ts) s_n = S_out[t];
      c_n = cst[t];
      if (ts) z_n = geo.zc[t];
      m_n = geo.m3[t];
    }
    xa = (k == nz - 1) ? a_k : a_k - c_k * xa;
    Ao[tk] = xa * mm;
    if (ts) {
      xb = (k == nz - 1) ? s_k : s_k - c_k * xb;
      S_out[tk] = xb * mm;
      if (p.eos_mixed)
        b_out[tk] = buoyancy_mixed(p, xa * mm, xb * mm, z_k) * mm;
      else
        b_out[tk] = buoyancy(p, xa * mm, xb * mm, z_k) * mm;
    }
  }
}

}  // namespace hoc

namespace hoc {

// ------------------------------------------------ column-form geometry
// Column geometry of a tile and its 2-cell halo, staged once per launch:
// wet levels nw and deepest wet thickness hb per column, and the 2D face
// masks. Every thickness, face thickness and 3D mask of the tile at any
// level follows from these (cg_dz, cg_face in hoc_device.h).
struct ColTile {  // [SY + 1][SX + 1]: the face flags of the last halo row and column
  double hb[SY + 1][SX + 1];  // need the column beyond them
  uint8_t nw[SY + 1][SX + 1];
  uint8_t mu[SY + 1][SX + 1];  // mask_u: the east face of the column is open
  uint8_t mv[SY + 1][SX + 1];  // mask_v: the north face of the column is open
};

__device__ __forceinline__ void col_tile_load(ColTile& CG, const Geo& geo, int tid, int i0,
                                              int j0, int nx, int ny) {
  for (int t = tid; t < (SX + 1) * (SY + 1); t += TILE_THREADS) {
    const int lx = t % (SX + 1), ly = t / (SX + 1);
    const long long g = (long long)pmod(j0 + ly - HALO, ny) * nx + pmod(i0 + lx - HALO, nx);
    CG.hb[ly][lx] = geo.hb[g];
    CG.nw[ly][lx] = geo.nw[g];
    CG.mu[ly][lx] = geo.mu2[g];
    CG.mv[ly][lx] = geo.mv2[g];
  }
}

// Level-k wet flags of the east face of tile column (ly, lx) and of its
// north face (mask3u, mask3v).
__device__ __forceinline__ bool col_wet_u(const ColTile& CG, int ly, int lx, int k) {
  return CG.mu[ly][lx] && k < CG.nw[ly][lx] && k < CG.nw[ly][lx + 1];
}
__device__ __forceinline__ bool col_wet_v(const ColTile& CG, int ly, int lx, int k) {
  return CG.mv[ly][lx] && k < CG.nw[ly][lx] && k < CG.nw[ly + 1][lx];
}

// Per-level staging of the column-form tracer tile: the tracers with halo
// and the face velocities; no geometry.
template <class R>
struct TracerLdsC {
  R c[2][SY][SX];
};
template <class R>
struct VelLdsC {
  R u[TY][TX + 1];  // u at i-1 .. i
  R v[TY + 1][TX];  // v at j-1 .. j
};
template <class R>
struct TracerRegsC {
  R c0[ST_C], c1[ST_C];
  R u[ST_U];
  R v[ST_V];
};

template <class RT>
__device__ __forceinline__ void tracer_load_c(TracerRegsC<RT>& R, const TileOffs& F, long long o,
                                              bool ts, const double* A, const double* S,
                                              const double* u, const double* v) {
#pragma unroll
  for (int q = 0; q < ST_C; ++q) {
    if (F.c[q] >= 0) {
      const long long g = o + F.c[q];
      R.c0[q] = (RT)A[g];
      R.c1[q] = ts ? (RT)S[g] : RT(0);
    }
  }
#pragma unroll
  for (int q = 0; q < ST_U; ++q)
    if (F.u[q] >= 0) R.u[q] = (RT)u[o + F.u[q]];
#pragma unroll
  for (int q = 0; q < ST_V; ++q)
    if (F.v[q] >= 0) R.v[q] = (RT)v[o + F.v[q]];
}

template <class RT>
__device__ __forceinline__ void tracer_store_c(TracerLdsC<RT>& L, VelLdsC<RT>& V,
                                               const TracerRegsC<RT>& R, int tid) {
#pragma unroll
  for (int q = 0; q < ST_C; ++q) {
    const int t = tid + q * TILE_THREADS;
    if (t < SX * SY) {
      const int lx = t % SX, ly = t / SX;
      L.c[0][ly][lx] = R.c0[q];
      L.c[1][ly][lx] = R.c1[q];
    }
  }
#pragma unroll
  for (int q = 0; q < ST_U; ++q) {
    const int t = tid + q * TILE_THREADS;
    if (t < TY * (TX + 1)) V.u[t / (TX + 1)][t % (TX + 1)] = R.u[q];
  }
#pragma unroll
  for (int q = 0; q < ST_V; ++q) {
    const int t = tid + q * TILE_THREADS;
    if (t < (TY + 1) * TX) V.v[t / TX][t % TX] = R.v[q];
  }
}

// k_tracers_tiled for a static z-level geometry in column form: the same
// operations on the same operands in the same order (so the same bits),
// with every thickness, face thickness, centre depth and 3D mask formed from
// the tile's column geometry instead of read per cell, and tri_b factored
// in the forward sweep. Per layer cell it reads T, S, u, v, w and K_h, and
// writes T, S, b, with d* (in the outputs) and c* (in `cst`) parked between
// the sweeps.
template <class R>
__global__ __launch_bounds__(TILE_THREADS)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 4 : 1))) void k_tracers_col(
    Dims d, StepParams p, Geo geo, const double* __restrict__ T, const double* __restrict__ S,
    const double* __restrict__ b, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ w, const double* __restrict__ Kh, double* __restrict__ cst,
    double* __restrict__ T_out, double* __restrict__ S_out, double* __restrict__ b_out) {
  __shared__ TracerLdsC<R> LB[2];
  __shared__ VelLdsC<R> VL;
  __shared__ FaceLds<R> F;
  __shared__ ColTile CG;
  const int nx = d.nx, ny = d.ny, nz = d.nz;
  const long long n2 = d.n2;
  const int tid = threadIdx.x;
  const int tx = tid % TX, ty = tid / TX;
  int bx, by;
  xcd_tile(bx, by);
  const int i0 = bx * TX, j0 = by * TY;
  const int i = i0 + tx, j = j0 + ty;
  const bool active = i < nx && j < ny;
  const long long c = active ? (long long)j * nx + i : 0;
  const bool ts = p.tracers_ts != 0;
  const int ntr = ts ? 2 : 1;
  const double* A = ts ? T : b;
  double* Ao = ts ? T_out : b_out;
  const double flux[2] = {ts ? p.flux_T : 0.0, p.flux_S};
  const int adv = p.advection;
  const double dzr = p.dzr;
  const int rule = p.face_rule;
  const int cx = tx + HALO, cy = ty + HALO;

  TracerRegsC<R> RG;
  const TileOffs TO = tile_offsets(tid, i0, j0, nx, ny);
  tracer_load_c(RG, TO, 0, ts, A, S, u, v);
  col_tile_load(CG, geo, tid, i0, j0, nx, ny);
  tracer_store_c(LB[0], VL, RG, tid);
  __syncthreads();
  const int nwc = CG.nw[cy][cx];
  const double hbc = CG.hb[cy][cx];
  auto wet = [&](int kk) { return kk >= 0 && kk < nwc; };

  // own-column window: tracer at k-2..k+2
  double win[2][5];
  for (int q = 0; q < 5; ++q) win[0][q] = win[1][q] = 0.0;
  if (active) {
    for (int q = 2; q < 5; ++q) {
      const int kk = q - 2;
      if (kk < nz) {
        win[0][q] = A[kk * n2 + c];
        if (ts) win[1][q] = S[kk * n2 + c];
      }
    }
  }
  double w_k = active ? w[c] : 0.0;
  double kh_k = active ? Kh[c] : 0.0;
  double dzi_k = cg_dzi(dzr, nwc, hbc, 0, nz);
  R cf_top[2] = {R(0), R(0)};  // interface value at the top of level k
  double dprev[2] = {0.0, 0.0};
  double cb_prev = 0.0;  // c* of tri_b at the level above

  const bool has_adv = adv != ADV_NONE;
  for (int k = 0; k < nz; ++k) {
    const long long o = (long long)k * n2;
    const TracerLdsC<R>& L = LB[k & 1];
    if (k + 1 < nz) tracer_load_c(RG, TO, o + n2, ts, A, S, u, v);
    double w_k1 = 0.0, kh_k1 = 0.0;
    if (active) {
      w_k1 = w[o + n2 + c];
      kh_k1 = Kh[o + n2 + c];
    }
    const double dzi_k1 = cg_dzi(dzr, nwc, hbc, k + 1, nz);
    const double dz = cg_dz(dzr, nwc, hbc, k);
    // ---- faces: the east and north face of every cell, plus the tile's
    // west column (8) and south row (32) of faces by threads 0..39
    if (has_adv) {
      auto xface = [&](int fy_, int q) {
        const int yy = fy_ + HALO, c0x = q - 1 + HALO;
        const R vel = VL.u[fy_][q];
        const R ddu = R(cg_face(rule, dzr, CG.mu[yy][c0x] != 0, CG.nw[yy][c0x], CG.hb[yy][c0x],
                                CG.nw[yy][c0x + 1], CG.hb[yy][c0x + 1], k));
        const bool wm = k < CG.nw[yy][c0x - 1], w2 = k < CG.nw[yy][c0x + 2];
        for (int r = 0; r < ntr; ++r) {
          const R(*C)[SX] = L.c[r];
          F.fx[r][fy_][q] = ddu * vel * tracer_face<R>(adv, C[yy][c0x - 1], C[yy][c0x],
                                                       C[yy][c0x + 1], C[yy][c0x + 2], vel, wm,
                                                       w2);
        }
      };
      auto yface = [&](int q, int fx_) {
        const int xx = fx_ + HALO, c0y = q - 1 + HALO;
        const R vel = VL.v[q][fx_];
        const R ddv = R(cg_face(rule, dzr, CG.mv[c0y][xx] != 0, CG.nw[c0y][xx], CG.hb[c0y][xx],
                                CG.nw[c0y + 1][xx], CG.hb[c0y + 1][xx], k));
        const bool wm = k < CG.nw[c0y - 1][xx], w2 = k < CG.nw[c0y + 2][xx];
        for (int r = 0; r < ntr; ++r) {
          const R(*C)[SX] = L.c[r];
          F.fy[r][q][fx_] = ddv * vel * tracer_face<R>(adv, C[c0y - 1][xx], C[c0y][xx],
                                                       C[c0y + 1][xx], C[c0y + 2][xx], vel, wm,
                                                       w2);
        }
      };
      xface(ty, tx + 1);
      yface(ty + 1, tx);
      if (tid < TY) xface(tid, 0);
      else if (tid < TY + TX) yface(0, tid - TY);
    }
    __syncthreads();
    if (active) {
      const double inv = safe_inv(dz);
      const bool m_k = wet(k);
      const bool m_k1 = wet(k + 1);
      const bool bot_km1 = k >= 1 && wet(k - 1) && !m_k;  // cell k-1 is a bottom cell
      const bool bot_k = m_k && !((k + 1 < nz) && m_k1);   // cell k is a bottom cell
      double sub_k, den_k, cst_k;
      factor_row(p, k, inv, kh_k, kh_k1, safe_inv(dzi_k), safe_inv(dzi_k1), m_k,
                 (k + 1 < nz) && m_k1, p.thv_dt * 0.0, cb_prev, sub_k, den_k, cst_k);
      cst[o + c] = cst_k;
      cb_prev = cst_k;
      const uint8_t mue = col_wet_u(CG, cy, cx, k), muw = col_wet_u(CG, cy, cx - 1, k);
      const uint8_t mvn = col_wet_v(CG, cy, cx, k), mvs = col_wet_v(CG, cy - 1, cx, k);

      for (int r = 0; r < ntr; ++r) {
        const double cc = win[r][2];  // the tile's own cell, in fp64
        double tend = 0.0;
        if (!ts) tend = p.neg_N2 * (0.5 * (w_k + w_k1));
        if (has_adv) {
          const R hdiv = ((F.fx[r][ty][tx + 1] - F.fx[r][ty][tx]) / R(p.dx) +
                          (F.fy[r][ty + 1][tx] - F.fy[r][ty][tx]) / R(p.dy)) * R(inv);
          const R cft = (k == 0) ? R(win[r][2]) : cf_top[r];
          const R cfb = tracer_face_z<R>(adv, k + 1, nz, R(win[r][1]), R(win[r][2]),
                                         R(win[r][3]), R(win[r][4]), wet(k - 1), wet(k + 2),
                                         R(w_k1));
          cf_top[r] = cfb;
          const R vdiv = (R(w_k) * cft - R(w_k1) * cfb) * R(inv);
          tend = tend - (double)((hdiv + vdiv) * (m_k ? R(1) : R(0)));
        }
        if (p.has_K_h) {
          const R(*C)[SX] = L.c[r];
          const R ge = face_grad<R>(mue, C[cy][cx], C[cy][cx + 1], p.dx);
          const R gw = face_grad<R>(muw, C[cy][cx - 1], C[cy][cx], p.dx);
          const R gn = face_grad<R>(mvn, C[cy][cx], C[cy + 1][cx], p.dy);
          const R gs = face_grad<R>(mvs, C[cy - 1][cx], C[cy][cx], p.dy);
          tend = tend + p.K_h * (double)((m_k ? R(1) : R(0)) *
                                         ((ge - gw) / R(p.dx) + (gn - gs) / R(p.dy)));
        }
        // explicit vertical diffusion with the surface flux (vertical_var.py:80-106)
        double ft;
        if (k == 0) {
          ft = flux[r];
        } else {
          ft = kh_k * (win[r][1] - win[r][2]) * safe_inv(dzi_k);
          if (bot_km1) ft = 0.0;
        }
        double fb = 0.0;
        if (k + 1 < nz) {
          fb = kh_k1 * (win[r][2] - win[r][3]) * safe_inv(dzi_k1);
          if (bot_k) fb = 0.0;
        }
        const double out = (ft - fb) * inv;
        const double dr = 0.0 * win[r][2] * (bot_k ? 1.0 : 0.0);
        const double dzd = (out - dr * inv) * (m_k ? 1.0 : 0.0);
        double rhs = cc + p.dt * tend + p.c_dzd * dzd;
        if (k == 0) rhs = rhs + p.thv_dt * flux[r] * safe_inv(dz);
        const double dd = (k == 0) ? rhs / den_k : (rhs - sub_k * dprev[r]) / den_k;
        dprev[r] = dd;
        (r == 0 ? Ao : S_out)[o + c] = dd;
      }
      // ---- advance the window
      for (int r = 0; r < 2; ++r)
        for (int q = 0; q < 4; ++q) win[r][q] = win[r][q + 1];
      const int kn = k + 3;
      if (kn < nz) {
        win[0][4] = A[(long long)kn * n2 + c];
        if (ts) win[1][4] = S[(long long)kn * n2 + c];
      } else {
        win[0][4] = 0.0;
        win[1][4] = 0.0;
      }
      w_k = w_k1;
      kh_k = kh_k1;
    }
    dzi_k = dzi_k1;
    if (k + 1 < nz) tracer_store_c(LB[(k + 1) & 1], VL, RG, tid);
    __syncthreads();
  }
  if (!active) return;
  // back-substitution with the next level's operands loaded one level ahead
  double xa = 0.0, xb = 0.0;
  long long t = (long long)(nz - 1) * n2 + c;
  double a_n = Ao[t], s_n = ts ? S_out[t] : 0.0, c_n = cst[t];
  for (int k = nz - 1; k >= 0; --k) {
    const double a_k = a_n, s_k = s_n, c_k = c_n;
    const double mm = wet(k) ? 1.0 : 0.0;
    const long long tk = t;
    if (k > 0) {
      t -= n2;
      a_n = Ao[t];
      if (ts) s_n = S_out[t];
      c_n = cst[t];
    }
    xa = (k == nz - 1) ? a_k : a_k - c_k * xa;
    Ao[tk] = xa * mm;
    if (ts) {
      xb = (k == nz - 1) ? s_k : s_k - c_k * xb;
      S_out[tk] = xb * mm;
      const double z_k = cg_zc(geo.zs, dzr, nwc, hbc, k);
      if (p.eos_mixed)
        b_out[tk] = buoyancy_mixed(p, xa * mm, xb * mm, z_k) * mm;
      else
        b_out[tk] = buoyancy(p, xa * mm, xb * mm, z_k) * mm;
    }
  }
}

}  // namespace hoc

namespace hoc {

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

// Face fluxes of one component on one level, each computed once: the
// advective flux (advecting velocity times the face value) and the A_h
// gradient, on the x-faces (index q: between tile columns q-1 and q) and the
// y-faces (between rows q-1 and q).
template <class R>
struct MomFaces {
  R fx[TY][TX + 1], gx[TY][TX + 1];
  R fy[TY + 1][TX], gy[TY + 1][TX];
};

constexpr int MS_H = (SX * SY + TILE_THREADS - 1) / TILE_THREADS;              // halo slots
constexpr int MS_O = ((TY + 1) * (TX + 1) + TILE_THREADS - 1) / TILE_THREADS;  // +1 slots

// Level-k staging held in registers between its global loads and its LDS
// stores or its use, and this thread's plane offsets.
template <class R>
struct MomRegs {
  R a[MS_H], o[MS_O];
  double phi[2], b[2];  // at the own point and the next one along the component's direction
  R w[2];               // on interface k + 1
};
struct MomGeoRegs {  // geometry read from the arrays
  uint8_t ma[MS_H], mo[MS_O];
  double zc[2];
};
struct MomOffs {
  unsigned h[MS_H];  // A with its halo
  unsigned o[MS_O];  // the other component's points
};

// Value of a plane at a byte offset. The plane's address is the same in every
// lane and is kept in scalar registers, so that one vector register holds the
// offset for every array (a plane is below 2^32 bytes). Without the empty asm
// the compiler keeps a 64-bit vector address per array across the march, 30
// registers here.
template <class T>
__device__ __forceinline__ T at_byte(const T* plane, unsigned off) {
  unsigned long long a = (unsigned long long)plane;
  __asm__("" : "+s"(a));
  using G = const __attribute__((address_space(1))) char;
  return *(const __attribute__((address_space(1))) T*)((G*)a + off);
}
__device__ __forceinline__ void put_byte(double* plane, unsigned off, double v) {
  unsigned long long a = (unsigned long long)plane;
  __asm__("" : "+s"(a));
  using G = __attribute__((address_space(1))) char;
  *(__attribute__((address_space(1))) double*)((G*)a + off) = v;
}

// Slots beyond the tile read the own point (the value is not stored).
template <int COMP>
__device__ __forceinline__ MomOffs mom_offsets(int tid, int i0, int j0, int nx, int ny) {
  MomOffs F;
#pragma unroll
  for (int q = 0; q < MS_H; ++q) {
    const int t = tid + q * TILE_THREADS;
    const int tt = t < SX * SY ? t : tid;
    F.h[q] = (unsigned)(pmod(j0 + tt / SX - HALO, ny) * nx + pmod(i0 + tt % SX - HALO, nx));
  }
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

struct NoTile {};

// First threads that form the tile's west column of faces (TY of them) and
// its south row (TX).
constexpr int EDGE_X = 64, EDGE_Y = 0;
static_assert(EDGE_X + TY <= TILE_THREADS && EDGE_Y + TX <= TILE_THREADS, "edge threads");

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

// Levels at which the east (axis 0) or north (axis 1) face of column (j, i)
// is wet, for a static z-level geometry.
__device__ __forceinline__ int face_levels(const Geo& geo, int axis, int j, int i, int ny,
                                           int nx) {
  const int c0 = j * nx + i;
  const int c1 = axis == 0 ? j * nx + pmod(i + 1, nx) : pmod(j + 1, ny) * nx + i;
  const int a = geo.nw[c0], b = geo.nw[c1];
  return (axis == 0 ? geo.mu2[c0] : geo.mv2[c0]) ? (a < b ? a : b) : 0;
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
    MomLds<R>* LB, Mask* MB, MomFaces<R>& F, const double* __restrict__ A,
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
  const MomOffs MO = mom_offsets<COMP>(tid, i0, j0, nx, ny);
  auto load = [&](long long o) {
#pragma unroll
    for (int q = 0; q < MS_H; ++q) {
      RG.a[q] = (R)at_byte(A + o, 8u * MO.h[q]);
      if constexpr (!ZC) GG.ma[q] = at_byte(mA + o, MO.h[q]);
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
    for (int q = 0; q < MS_H; ++q) {
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
// 364, 1000 x 1000 x 30 1487 -> 1069. At 4 waves per SIMD it spills 30
// registers and takes 478 us at 512 x 512 x 40.
template <class R, bool ZC, bool TVD>
__global__ __launch_bounds__(TILE_THREADS) __attribute__((amdgpu_waves_per_eu(3))) void k_momentum_explicit_tiled(
    Dims d, StepParams p, Geo geo, int nk, const double* __restrict__ u,
    const double* __restrict__ v, const double* __restrict__ b, const double* __restrict__ phi,
    const double* __restrict__ w, const double* __restrict__ Km, const double* __restrict__ zs,
    double* __restrict__ pgx, double* __restrict__ pgy, double* __restrict__ dzu,
    double* __restrict__ dzv, double* __restrict__ stu, double* __restrict__ stv) {
  __shared__ MomLds<R> LB[2];
  __shared__ MomFaces<R> F;
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

void launch_tracers_tiled(bool mixed, hipStream_t s, Dims d, StepParams p, Geo geo,
                          const double* T, const double* S, const double* b, const double* u,
                          const double* v, const double* w, const double* Kh, double* cst,
                          double* T_out, double* S_out, double* b_out) {
  const dim3 grid((d.nx + TX - 1) / TX, (d.ny + TY - 1) / TY);
  if (p.zcol) {
    if (mixed)
      k_tracers_col<float><<<grid, TILE_THREADS, 0, s>>>(d, p, geo, T, S, b, u, v, w, Kh, cst,
                                                         T_out, S_out, b_out);
    else
      k_tracers_col<double><<<grid, TILE_THREADS, 0, s>>>(d, p, geo, T, S, b, u, v, w, Kh, cst,
                                                          T_out, S_out, b_out);
  } else if (mixed) {
    k_tracers_tiled<float><<<grid, TILE_THREADS, 0, s>>>(d, p, geo, T, S, b, u, v, w, Kh, cst,
                                                         T_out, S_out, b_out);
  } else {
    k_tracers_tiled<double><<<grid, TILE_THREADS, 0, s>>>(d, p, geo, T, S, b, u, v, w, Kh, cst,
                                                          T_out, S_out, b_out);
  }
}

// Levels per workgroup of a tiled march: all of them where the tiles alone give `target`
// workgroups, else as few as make up that number (each range of levels reads the two levels
// above and below it again and forms its top interface's fluxes a second time).
int levels_per_block(long long tiles, int nz, long long target) {
  const long long parts = tiles >= target ? 1 : (target + tiles - 1) / tiles;
  const int n = (int)((nz + parts - 1) / parts);
  return n < 1 ? 1 : n;
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
