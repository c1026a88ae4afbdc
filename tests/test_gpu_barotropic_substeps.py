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


@pytest.mark.parametrize("n_picard", [2, 4])
def test_captured_step_replays(hoc, n_picard):
    """A split step and the pressure gradients in a graph of the caller's,
    replayed four times with eager steps and a synchronisation between the
    replays, each time bitwise the eager result: what is cleared inside (the
    averaged transports from four passes on, the pressure gradients' zero
    fields) is cleared by kernels."""
    from hydrostatic_ocean_core_benchmark_amd.types import State3D
    dom, phys, params, f = _problem(33, 15, 3, "zlevel", "up3")
    params = dataclasses.replace(params, name="split_explicit", n_split=3, n_picard=n_picard,
                                 barotropic_average="mean")
    with hoc.HipStepper(dom, phys, params, 60.0) as st:
        fin, out = st._inputs(State3D(**f)), st._new_state_buffers()
        want, other = st._new_state_buffers(), st._new_state_buffers()
        nu, kappa = st.nu.clone(), st.kappa.clone()

        def eager(src, dst):
            st.nu.copy_(nu)
            st.kappa.copy_(kappa)
            st._step_into(src, dst)

        eager(fin, want)
        px, py = st.pressure_gradients(fin["b"])
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            eager(fin, out)
            gx, gy = st.pressure_gradients(fin["b"])
        for n in range(4):
            eager(want, other)
            st.pressure_gradients(other["b"])
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(gx, px) and torch.equal(gy, py), n
            for k, w in want.items():
                assert torch.equal(out[k], w), (n, k)
