"""The barotropic substeps of split_explicit, several to a launch: even and odd
numbers of them, one to four Picard passes (four run launch by launch), grids
smaller than a tile with its halo (which then wraps round the grid more than
once), partial tiles, the averaged transports, and closed, periodic and open
edges. Two steps from a random state, bitwise against the oracle."""

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


@pytest.mark.parametrize("n_split,n_picard", [(1, 2), (2, 1), (5, 2), (6, 3), (3, 4)])
@pytest.mark.parametrize("nx,ny", [(5, 4), (16, 17), (33, 15), (70, 41)])
@pytest.mark.parametrize("edges", ["closed", "periodic", "open"])
def test_steps_match_oracle(hoc, nx, ny, edges, n_split, n_picard):
    from hydrostatic_ocean_core_benchmark_amd.types import State3D
    from oracle.stepper import OracleStepper, OState
    dom, phys, params, f = _problem(nx, ny, 3, "zlevel", "up3")
    dom = dataclasses.replace(dom, bc_x=edges, bc_y=edges)
    if edges == "open":
        phys = dataclasses.replace(phys, eta_ext=0.02, u_ext=0.03)
    f["u"] = f["u"] * dom.mask3u
    f["v"] = f["v"] * dom.mask3v
    params = dataclasses.replace(params, name="split_explicit", n_split=n_split, n_picard=n_picard,
                                 barotropic_average="mean" if n_split > 2 else "none")
    ref = OracleStepper(dom, phys, params, 60.0)
    want = ref.step(ref.step(OState(**f)))
    with hoc.HipStepper(dom, phys, params, 60.0) as st:
        got = st.step(st.step(State3D(**f)))
        torch.cuda.synchronize()
        for k in ("u", "v", "eta", "T", "S"):
            g, w = getattr(got, k).cpu().numpy(), getattr(want, k)
            assert np.array_equal(g, w), (k, rel_l2(g, w))
