"""gdx_phase_times on device 0: refused before a numeric phase has run; after one
of any kind, the stages that launched add up to the total and the others are 0.  A
numeric phase that a caller captures into a graph runs nothing and leaves them."""
import ctypes

import numpy as np
import pytest
import torch

from gridap_amd import _lib, flux_operator_from_workload, problem_from_workload
from gridap_amd import workloads as W
from gridap_amd._lib import GdxError

pytestmark = pytest.mark.gpu

ERR_STATE = -3
MODES = W.fourier_modes(5, 5, 3, 0.4)


def diffusion(cells, **kw):
    dim = len(cells)
    p = dict(dim=dim, order=1, qdeg=2, cells=cells, parts=(1,) * dim, domain=(0.0, 1.0) * dim, strategy="sub",
             coef_const=1.0, modes=np.zeros((0, 5)), rhs="const", rhs_const=1.0, dirichlet=True, uD=(0.0, 1.0, 0.0, 0.0))
    p.update(kw)
    return p


# kind, problem, stages that launch (coefficient, RHS, matrix)
KINDS = {
    "2d constant": (diffusion((9, 7)), (False, False, True)),
    "3d modes": (diffusion((6, 5, 4), modes=MODES), (True, False, True)),
    "3d manufactured": (diffusion((6, 5, 4), modes=MODES, rhs="manufactured"), (True, True, True)),
    "3d cells": (diffusion((6, 5, 4)), (False, False, True)),
    "3d z-marching": (diffusion((6, 5, 4), modes=MODES), (True, None, True)),
    "mapped": (diffusion((6, 5, 4)), (True, False, True)),
    "elasticity": (W.elasticity3d_q2((3, 3, 2), (1, 1, 1)), (False, False, True)),
    "flux": (dict(W.plaplacian3d_q1(6, (1, 1, 1)), flux=(3.0, 0.01, 1.0)), (False, False, True)),
}


def problem(ctx, kind):
    p = KINDS[kind][0]
    if kind == "flux":
        return flux_operator_from_workload(ctx, p)._problem()
    assem, data = problem_from_workload(ctx, p)
    prob = assem._problem_for(data)
    if kind == "3d cells":
        prob.set_cell_coefficient(np.linspace(1.0, 2.0, int(np.prod(p["cells"]))))
    if kind == "3d z-marching":
        prob.set_kernel(0, 16)
    if kind == "mapped":
        prob.set_vertex_coords(W.mapped_vertices(p))
    return prob


def refused(prob):
    with pytest.raises(GdxError) as e:
        prob.phase_times()
    assert e.value.code == ERR_STATE


@pytest.mark.parametrize("kind", KINDS)
def test_stages_add_up(gpu_ctx, kind):
    prob = problem(gpu_ctx, kind)
    refused(prob)
    prob.numeric()
    t = prob.phase_times()
    # every time is a float difference of the same timestamps, at most milliseconds
    assert 0.0 < t[3] < 1e3 and sum(t[:3]) == pytest.approx(t[3], abs=1e-4)
    for ms, launched in zip(t, KINDS[kind][1]):
        assert launched is None or (ms > 0.0 if launched else ms == 0.0)
    prob.close()


@pytest.mark.parametrize("kind", ["3d cells", "elasticity"])
def test_capture_of_the_numeric_phase(gpu_ctx, kind):
    """The numeric phase captured by the program on the library's stream: replays
    assemble with the coefficient of their time, and no time is taken from it."""
    prob = problem(gpu_ctx, kind)
    ncell = int(np.prod(KINDS[kind][0]["cells"]))
    ptr = ctypes.c_void_p()
    _lib.call("gdx_stream", prob.handle, ctypes.byref(ptr))
    stream = torch.cuda.ExternalStream(ptr.value)

    def values():
        prob.sync()
        return np.concatenate([np.concatenate([Q["val"], Q["b"]]) for Q in map(prob.export_part, range(prob.nparts))])

    def capture():
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            graph.capture_begin(capture_error_mode="thread_local")
            prob.numeric()
            graph.capture_end()
        return graph

    prob.set_cell_coefficient(np.full(ncell, 1.0))
    graph = capture()
    refused(prob)  # it has not run
    prob.numeric()
    times = prob.phase_times()
    again = capture()
    assert prob.phase_times() == times
    for k, g in enumerate((graph, again, graph)):
        prob.set_cell_coefficient(np.full(ncell, 2.0 + k))
        with torch.cuda.stream(stream):
            g.replay()
        got = values()
        prob.set_cell_coefficient(np.full(ncell, 9.0))  # other values in between
        prob.numeric()
        prob.sync()
        prob.set_cell_coefficient(np.full(ncell, 2.0 + k))
        prob.numeric()
        assert np.array_equal(got, values())
    del graph, again
    prob.close()
