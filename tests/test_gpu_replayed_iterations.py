"""PCG-Jacobi iterations replayed from recorded graphs: steps whose solves
need different numbers of iterations, limits that fall inside, at and past a
replayed run (3 to 8 iterations, where a solve ends unconverged), the default
and a side stream, and a second handle stepped in between. Bitwise against the
oracle, with its iteration and failure counts."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_level_ranges import _problem

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def hoc(gpu_available):
    from hydrostatic_ocean_core_benchmark_amd import stepper
    return stepper


@pytest.mark.parametrize("side_stream", [False, True])
@pytest.mark.parametrize("max_iter", [1, 2, 3, 4, 5, 8, 2000])
def test_steps_match_oracle(hoc, max_iter, side_stream):
    from hydrostatic_ocean_core_benchmark_amd.types import State3D
    from oracle.stepper import OracleStepper, OState
    dom, phys, params, f = _problem(37, 22, 6, "zlevel", "up3_tvd")
    params = dataclasses.replace(params, name="theta", max_iter=max_iter)
    ref = OracleStepper(dom, phys, params, 300.0)
    want = OState(**f)
    stream = torch.cuda.Stream() if side_stream else torch.cuda.default_stream()
    with hoc.HipStepper(dom, phys, params, 300.0) as st, \
            hoc.HipStepper(dom, phys, params, 150.0) as other, torch.cuda.stream(stream):
        got = State3D(**f)
        for n in range(7):  # replayed from the fifth step on
            want = ref.step(want)
            other.step(State3D(**f))
            got = st.step(got)
            stream.synchronize()
            assert st.solver_iterations == ref.solver_iterations, n
            assert st.solver_failures == ref.solver_failures, n
            for k in ("u", "v", "eta", "T", "S"):
                g, w = getattr(got, k).cpu().numpy(), getattr(want, k)
                assert np.array_equal(g, w), (n, k, rel_l2(g, w))
