"""The V-cycle's fused legs and its one-workgroup coarse cycle at the sizes
where their regions can go wrong: levels smaller than a tile plus its halo
(the region wraps round the level more than once), partial tiles, coarse
levels with odd sides, and first levels of the coarse cycle just below and
above each thread count's cells. Solves from random coefficients, bitwise
against the oracle and with its iteration counts."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import _random_helmholtz

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (ny, nx), levels: a 12-wide level in a 64-wide region; 10-cell sides; 25 x 17
# and 1023-, 1024-, 1056-, 2048- and 2080-cell last levels
SHAPES = [((512, 24), 5), ((24, 512), 5), ((40, 20), 2), ((100, 50), 5), ((8, 8), 5),
          ((100, 68), 3), ((66, 62), 2), ((64, 64), 2), ((66, 64), 2), ((128, 64), 2),
          ((130, 64), 2), ((180, 90), 2)]


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


@pytest.mark.parametrize("kind,smoother", [("pcg_mg", "rbgs"), ("pcg_mg", "jacobi"),
                                           ("multigrid", None)])
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_cycle_matches_oracle(hoc, kind, smoother, shape, levels):
    from oracle.helmholtz import HelmholtzVar
    kw = {"solver": kind}
    okw = {}
    if kind == "pcg_mg":
        okw = {"mg_levels": levels, "mg_smoother": smoother}
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


@pytest.mark.parametrize("sweeps", [1, 2, 3])
def test_fp32_legs_do_not_depend_on_the_tile(hoc, sweeps):
    """The fp32 preconditioner: every tile shape gives the same bits."""
    outs = []
    for tile in range(4):
        st, *_, Ku, Kv, rhs = _stepper(hoc, (160, 232), "periodic", tile, "mixed", solver="pcg_mg",
                                       mg_levels=3, mg_sweeps=sweeps)
        x, iters, conv = st.helmholtz_solve(Ku, Kv, rhs)
        assert conv
        outs.append((x.detach().cpu().numpy(), iters))
    for x, iters in outs[1:]:
        assert iters == outs[0][1] and np.array_equal(x, outs[0][0])
