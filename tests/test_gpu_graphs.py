"""Captured multigrid cycles (use_graph): what a graph was captured with must
be what its replays would be launched with now.  Each run is compared bit for
bit with the same run as plain launches, for variants that are deterministic;
runs are long enough that most of their cycles are replays.
"""
import ctypes as C

import numpy as np
import pytest

import mgcfd
from conftest import perturbed_state

pytestmark = pytest.mark.gpu

DETERMINISTIC = ["gather_exact", "part_coloured", "mixed_coloured"]


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    r.set_flux_variant(mgcfd.FLUX_VARIANTS["gather_exact"])
    yield r
    r.close()


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


def run_bound(rt, cycles, graph):
    """mgcfd_mg_run on the levels bound last (Solver.run_device binds anew)."""
    rms, st = np.zeros(cycles), C.c_int(-1)
    mgcfd._check(rt.L.mgcfd_mg_run(cycles, int(graph), rms.ctypes.data_as(C.POINTER(C.c_double)), C.byref(st)),
                 "mgcfd_mg_run")
    assert st.value == 0
    return rms


def solver(rt, mesh):
    s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
    s.setup()
    rt.upload(s.lv[0].variables, perturbed_state(len(mesh[0]["coords"]), s.fs["ff_variable"], seed=5))
    return s


@pytest.mark.parametrize("variant", DETERMINISTIC + ["nodal_exact"])
def test_constants_changed_between_runs(rt, knn_small, variant):
    """One binding, two runs with different freestreams: the second run's
    replays use the constants declared last."""
    got = []
    for graph in (False, True):
        s = solver(rt, knn_small)
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        s.bind()
        out = []
        for mach, aoa in ((0.5, 3.0), (0.7, -1.0)):
            rt.decl_consts(mgcfd.freestream(mach, aoa))
            out += [run_bound(rt, 6, graph)] + [s.state(l) for l in range(len(knn_small))]
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("variant", ["part_coloured", "mixed_coloured"])
def test_part_plan_changed_between_runs(rt, knn_small, variant):
    """One binding, a run before and after each level was planned anew: the
    replays use the new plan's buffers, grid and kernels."""
    got = []
    for graph in (False, True):
        s = solver(rt, knn_small)
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        s.bind()
        out = [run_bound(rt, 6, graph)]
        for config in ((128, 512), (128, 256), (192, 0)):
            for h in s.lv:
                rt.map_part_config(h.edge_to_node, *config)
            out += [run_bound(rt, 6, graph)] + [s.state(l) for l in range(len(knn_small))]
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))
