"""The V-cycle's fused legs and its one-workgroup coarse cycle at the sizes
where their regions can go wrong: levels smaller than a tile plus its halo
(the region wraps round the level more than once), partial tiles, coarse
levels with odd sides, and first levels of the coarse cycle just below and
above each thread count's cells, with one to three sweeps per side. Solves
from random coefficients, bitwise against the oracle and with its iteration
counts."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import _random_helmholtz

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (ny, nx), levels: a 12-wide level in a 64-wide region; 10-cell sides; 25 x 17
# and 1023-, 1024-, 1056-, 2048-, 2080-, 4050- and 4095-cell last levels (65 x 32,
# 90 x 45 and 63 x 65 with odd sides)
SHAPES = [((512, 24), 5), ((24, 512), 5), ((40, 20), 2), ((100, 50), 5), ((8, 8), 5),
          ((100, 68), 3), ((66, 62), 2), ((64, 64), 2), ((66, 64), 2), ((128, 64), 2),
          ((130, 64), 2), ((180, 90), 2), ((63, 65), 1)]


@pytest.fixture(scope="module")
def hoc(gpu_available):
    from hydrostatic_ocean_core_benchmark_amd import stepper
    return stepper


def _stepper(hoc, shape, bc, tile=None, precision="fp64", seed=17, **kw):
    from hydrostatic_ocean_core_benchmark_amd import _lib
    from hydrostatic_ocean_core_benchmark_amd.types import Physics3D, PhysicsV05, SchemeParams
    grid, dom, mask, Ku, Kv, rhs = _random_helmholtz(shape, bc, seed=seed)
    phys = PhysicsV05(base=Physics3D(g=9.80616, f=1e-4, H=4000.0))
    params = SchemeParams(name="theta", rtol=1e-12, max_iter=5000, **kw)
    st = hoc.HipStepper(dom, phys, params, 600.0, precision=precision)
    if tile is not None:
        _lib.check(st.lib.hoc_stepper_set_mg_tile(st._h, tile))
    return st, grid, mask, Ku, Kv, rhs


@pytest.mark.parametrize("kind,smoother,sweeps", [
    ("pcg_mg", "rbgs", 2), ("pcg_mg", "jacobi", 2), ("multigrid", None, 2), ("pcg_mg", "rbgs", 1),
    ("pcg_mg", "rbgs", 3), ("pcg_mg", "jacobi", 1), ("pcg_mg", "jacobi", 3)])
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_cycle_matches_oracle(hoc, kind, smoother, sweeps, shape, levels):
    from oracle.helmholtz import HelmholtzVar
    kw = {"solver": kind}
    okw = {}
    if kind == "pcg_mg":
        okw = {"mg_levels": levels, "mg_smoother": smoother, "mg_sweeps": sweeps}
    for tile, bc in ((0, "closed"), (2, "periodic")):
        st, grid, mask, Ku, Kv, rhs = _stepper(hoc, shape, bc, tile, **kw, **okw)
        ny, nx = shape
        ref = HelmholtzVar(nx, ny, grid.dx, grid.dy, st.cfg.g * 0.25 * 600.0 ** 2, Ku, Kv, mask,
                           kind=kind, rtol=1e-12, max_iter=5000, **okw)
        want, rep = ref.solve(rhs)
        x, iters, conv = st.helmholtz_solve(Ku, Kv, rhs)
        got = x.detach().cpu().numpy()
        assert conv == rep.converged and iters == rep.iterations, (tile, iters, rep.iterations)
        assert np.array_equal(got, want), (tile, rel_l2(got, want))


def _fp32_oracle(*args, **kw):
    """The oracle's PCG with its V-cycle in float32: coefficients, masks and
    every operation (scalars are rounded to the arrays' type), from the
    rounded residual to the correction, which goes back to float64."""
    import copy

    from oracle.helmholtz import HelmholtzVar

    class Mixed(HelmholtzVar):
        def _precondition(self, r):
            fine = self.levels
            self.levels = []
            for op in fine:
                op = copy.copy(op)
                for k in ("Ku", "Kv", "mask", "inv_diag"):
                    setattr(op, k, getattr(op, k).astype(np.float32))
                self.levels.append(op)
            z = self._mg_precond(r.astype(np.float32))
            self.levels = fine
            assert z.dtype == np.float32
            return z.astype(np.float64)

    return Mixed(*args, **kw)


@pytest.mark.parametrize("sweeps", [1, 2, 3])
@pytest.mark.parametrize("shape,levels", [((160, 232), 3), ((40, 20), 2), ((24, 512), 5),
                                          ((130, 64), 2), ((128, 64), 2), ((63, 65), 1)])
def test_fp32_cycle_matches_oracle(hoc, shape, levels, sweeps):
    """The fp32 preconditioner against the same cycle in NumPy, bitwise, at
    every tile shape (two sweeps; the other numbers have one)."""
    ny, nx = shape
    kw = {"mg_levels": levels, "mg_sweeps": sweeps}
    for tile in range(4 if sweeps == 2 else 1):
        st, grid, mask, Ku, Kv, rhs = _stepper(hoc, shape, "periodic", tile, "mixed",
                                               solver="pcg_mg", **kw)
        if tile == 0:
            ref = _fp32_oracle(nx, ny, grid.dx, grid.dy, st.cfg.g * 0.25 * 600.0 ** 2, Ku, Kv,
                               mask, kind="pcg_mg", rtol=1e-12, max_iter=5000, **kw)
            want, rep = ref.solve(rhs)
        x, iters, conv = st.helmholtz_solve(Ku, Kv, rhs)
        got = x.detach().cpu().numpy()
        assert conv and rep.converged and iters == rep.iterations, (tile, iters, rep.iterations)
        assert np.array_equal(got, want), (tile, rel_l2(got, want))
