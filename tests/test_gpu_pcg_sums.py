"""The PCG's dot products over every shape of their partition: fewer than 8
cells, one leaf, leaves of unequal depth (255 cells halve to 120 and 135), a
full trailing chunk less one, whole chunks with and without a trailing one, the
last grid whose totals every workgroup forms and the first whose totals a launch
of its own forms, each in phases and, up to the parts that the cooperative
launch takes, persistent. Bitwise against the oracle, iteration counts equal."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_parity import _random_helmholtz

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [(2, 3), (4, 5), (8, 16), (3, 43), (15, 17), (16, 16), (7, 73), (13, 79), (64, 128),
          (65, 127), (64, 129), (91, 181), (130, 126), (77, 131), (127, 129), (256, 1056),
          (700, 900), (768, 1024), (769, 1024), (1030, 1035)]


@pytest.fixture(scope="module")
def hoc(gpu_available):
    from hydrostatic_ocean_core_benchmark_amd import stepper
    return stepper


@pytest.mark.parametrize("shape", SHAPES)
def test_pcg_matches_oracle(hoc, shape):
    from hydrostatic_ocean_core_benchmark_amd.types import Physics3D, PhysicsV05, SchemeParams
    from oracle.helmholtz import HelmholtzVar
    ny, nx = shape
    grid, dom, mask, Ku, Kv, rhs = _random_helmholtz(shape, "periodic", seed=nx)
    rtol = 1e-12 if ny * nx < 50000 else 1e-5
    phys = PhysicsV05(base=Physics3D(g=9.80616, f=1e-4, H=4000.0))
    params = SchemeParams(name="theta", solver="pcg_jacobi", rtol=rtol, max_iter=400)
    st = hoc.HipStepper(dom, phys, params, 600.0)
    ref = HelmholtzVar(nx, ny, grid.dx, grid.dy, st.cfg.g * 0.25 * 600.0 ** 2, Ku, Kv, mask,
                       kind="pcg_jacobi", rtol=rtol, max_iter=400)
    want, rep = ref.solve(rhs)
    for path in ("multikernel", "persistent"):
        st.solver_path = path
        # 16 parts per whole chunk of 8192 cells: at most 1792 are resident
        taken = path if ny * nx < 900_000 else "multikernel"
        assert st.solver_path == taken, path
        x, iters, conv = st.helmholtz_solve(Ku, Kv, rhs)
        got = x.detach().cpu().numpy()
        assert conv == rep.converged and iters == rep.iterations, (path, iters, rep.iterations)
        assert np.array_equal(got, want), (path, rel_l2(got, want))
