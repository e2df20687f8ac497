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
from oracle import Oracle
from test_gpu_fused_stages import random_mesh

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


def replays(rt):
    rt.L.mgcfd_graph_replays.restype = C.c_longlong
    return rt.L.mgcfd_graph_replays()


@pytest.mark.parametrize("variant", DETERMINISTIC + ["gather_fast", "nodal_exact"])
def test_batch_replays_equal_plain_launches(rt, knn_small, variant):
    """Three runs of a batch: the first replays the cycles between its first
    and last, the others all of theirs; states, fluxes and histories are those
    of plain launches."""
    meshes = [mgcfd.mesh_knn(1200, 3720, 4, seed=4), knn_small]
    got = []
    for graph in (False, True):
        b = mgcfd.Batch(rt, meshes, [0.5, 0.7], [3.0, -1.5], variant)
        out, counts = [], []
        for _ in range(3):
            before = replays(rt)
            st, rms = b.run(7, use_graph=graph)
            counts.append(replays(rt) - before)
            assert not st.any()
            out += [rms] + [b.fetch(i, l) for i in range(2) for l in range(4)]
            out += [b.fetch(i, l, "step_factors") for i in range(2) for l in range(4)]
            assert not any(b.fetch(i, l, "fluxes").any() for i in range(2) for l in range(4))
        b.close()
        assert counts == ([5, 7, 7] if graph else [0, 0, 0])
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("variant", DETERMINISTIC + ["nodal_exact"])
@pytest.mark.parametrize("levels,cycles,counts", [(3, 1, [0, 1, 1, 1]), (3, 2, [0, 2, 2, 2]), (3, 4, [2, 4, 4, 4]),
                                                  (1, 1, [0, 1, 1, 1]), (1, 3, [2, 3, 3, 3])])
def test_short_runs_on_one_binding(rt, variant, levels, cycles, counts):
    """Runs of one cycle and more, the state carried on the device between
    them, with fetches and loops of the caller's in between: every run from
    the second on is replayed, and equals plain launches."""
    mesh = mgcfd.mesh_box(8, 3, seed=7)[:levels]
    got = []
    for graph in (False, True):
        s = solver(rt, mesh)
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        s.bind()
        out = []
        for k in range(4):
            # what a run finds in the flux dats, its first stages add to
            for l, h in enumerate(s.lv):
                rt.upload(h.fluxes, 1e-9 * perturbed_state(h.sizes["nodes"], np.ones(5), seed=6 + l + k))
            before = replays(rt)
            out.append(run_bound(rt, cycles, graph))
            assert replays(rt) - before == (counts[k] if graph else 0)
            out += [s.state(l, what) for l in range(levels)
                    for what in ("variables", "old_variables", "step_factors", "residuals", "fluxes")]
        got.append(out)
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("variant", DETERMINISTIC + ["nodal_exact"])
def test_abort_in_a_later_cycle(rt, variant):
    """Volumes so small that the solve blows up: the reference's early return
    on a NaN comes in its eighth cycle, which is a replay when graphs are used,
    begun by the cycle before.  Status, history and the nodes that hold NaN are
    the reference's, and every value is that of plain launches."""
    mesh = random_mesh(515, 4, seed=9)
    o = Oracle("orc")
    state = perturbed_state(515, o.freestream(0.5, 3.0).ff_variable[:], seed=5)
    vol = {}

    def after_setup(levels):
        levels[0]["var"][:] = state
        for l, a in enumerate(levels):
            a["vol"] *= 1e-9
            vol[l] = a["vol"].copy()

    with np.errstate(all="ignore"):
        ref = o.solve(mesh, 12, 0.5, 3.0, after_setup=after_setup)
    assert ref["status"] == 2 and ref["steps"] == 15 and np.isnan(ref["rms"]).nonzero()[0].tolist() == [7]
    got = []
    for graph in (False, True):
        s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
        s.setup()
        rt.upload(s.lv[0].variables, state)
        for l in range(2):
            rt.upload(s.lv[l].volumes, vol[l])
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        before = replays(rt)
        st, rms = s.run_device(12, use_graph=graph)
        assert replays(rt) - before == (10 if graph else 0)
        assert st == 2
        assert np.isnan(rms).nonzero()[0].tolist() == [7] and not rms[8:].any()
        if not variant.startswith("mixed"):
            assert np.allclose(rms[:7], ref["rms"][:7], rtol=1e-6, atol=0)
            for l in range(2):
                assert np.array_equal(np.isnan(s.state(l)), np.isnan(ref["levels"][l]["variables"]))
        got.append([rms] + [s.state(l, w) for l in range(2) for w in ("variables", "residuals")])
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))
