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
            # two solves a step; a run of two needs a third iteration
            assert (st.replayed_iterations > 0) == (n >= 4 and max_iter >= 3), n
            assert st.solver_iterations == ref.solver_iterations, n
            assert st.solver_failures == ref.solver_failures, n
            for k in ("u", "v", "eta", "T", "S"):
                g, w = getattr(got, k).cpu().numpy(), getattr(want, k)
                assert np.array_equal(g, w), (n, k, rel_l2(g, w))


def test_steps_while_another_thread_captures(hoc):
    """A handle stepped through its first replayed solves while another thread
    captures a graph (in the thread-local mode: in the global one a polled
    step's synchronisation is refused, with or without replays): the state and
    the graph come out right."""
    import threading
    dom, phys, params, f = _problem(37, 22, 6, "zlevel", "up3_tvd")
    params = dataclasses.replace(params, name="theta")
    got, err = {}, []
    with hoc.HipStepper(dom, phys, params, 300.0) as st, \
            hoc.HipStepper(dom, phys, params, 300.0) as plain:
        runs = []
        for h in (st, plain):
            a, b = h._new_state_buffers(), h._new_state_buffers()
            for k, buf in a.items():
                buf.copy_(torch.as_tensor(f[k]))
            runs.append((a, b))
        want = plain._step_n_into(*runs[1], 8)
        side, cap = torch.cuda.Stream(), torch.cuda.Stream()
        y = torch.zeros(1000, device="cuda")
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()

        def steps():
            try:
                with torch.cuda.stream(side):
                    got.update(st._step_n_into(*runs[0], 8))
            except Exception as e:
                err.append(e)

        with torch.cuda.stream(cap):
            graph.capture_begin(capture_error_mode="thread_local")
            y.add_(1.0)
            t = threading.Thread(target=steps)
            t.start()
            t.join()
            try:
                graph.capture_end()
            except Exception as e:
                err.append(e)
        assert not err, err
        assert st.replayed_iterations > 0
        torch.cuda.synchronize()
        for n in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert torch.all(y == n + 1.0), n
        for k, w in want.items():
            assert torch.equal(got[k], w), k


@pytest.mark.parametrize("dt,replays", [(20.0, False), (600.0, True)])
def test_few_iterations_are_launched(hoc, dt, replays):
    """256 x 256: 7 iterations a solve are launched, 77 replayed (from 32 on at
    this size), with the bits of a handle whose phases are profiled by name,
    which launches all."""
    dom, phys, params, f = _problem(256, 256, 2, "zlevel", "up3_tvd")
    params = dataclasses.replace(params, name="theta")
    ends = []
    for name in (None, "k_pcg_ap"):
        with hoc.HipStepper(dom, phys, params, dt) as st:
            st.profile_kernel(name)
            a, b = st._new_state_buffers(), st._new_state_buffers()
            for k, buf in a.items():
                buf.copy_(torch.as_tensor(f[k]))
            ends.append({k: x.clone() for k, x in st._step_n_into(a, b, 7).items()})
            assert (st.replayed_iterations > 0) == (replays and name is None)
    for k, want in ends[1].items():
        assert torch.equal(ends[0][k], want), k
