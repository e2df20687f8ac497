"""The kernels that run a Runge-Kutta stage inside the edge flux
(k_gather_stage, k_flux_part_stage) and the device-resident driver around
them, at the sizes where their tiles can go wrong, against the oracle.

Meshes are random graphs, whose parts have halos far larger than a box's or a
nearest-neighbour mesh's: the blocked plan's parts of 256 nodes are split at
its halo limit, and stage one or two halo nodes per thread.  Sizes sit at
the edges of a part (255, 256, 257 nodes) and of several parts; degrees from
2 to 12 per node give halos below 256, between 256 and the limit, and
beyond it.  Every solve starts from a disturbed state and from non-zero flux
dats, which the first cycle has to add to and leave zero.

Bars as in the parity suite: FP64 variants 1e-12 relative per variable on the
state after three cycles (the random graphs' weights are damped by 1e-7 as
every mesh's, so a stage's rounding differences of ~1e-16 are not amplified),
mixed precision 1e-6.
"""
import numpy as np
import pytest

import mgcfd
from conftest import perturbed_state
from oracle import Oracle
from test_gpu_parity import MIXED_STATE_TOL, STATE_TOL, rel_err

pytestmark = pytest.mark.gpu


def random_mesh(n, deg, seed):
    """Two levels of n and n / 2 nodes at random points, node i of the first
    restricting to i / 2 of the second; each level's edges are a ring, so that
    every node has a volume, and random pairs up to 'deg' per node."""
    rng = np.random.default_rng(seed)

    def level(n, ne):
        ring = np.arange(n)
        a = np.concatenate([ring, rng.integers(0, n, max(0, ne - n))])
        b = (a + np.concatenate([np.ones(n, np.int64), rng.integers(1, n, len(a) - n)])) % n
        ne = len(a)
        nb = max(1, n // 7)
        return dict(coords=rng.uniform(0.0, 2.0, (n, 3)), edge_to_node=np.stack([a, b], 1).astype(np.int32),
                    edge_weights=rng.uniform(-0.6, 0.6, (ne, 3)),
                    bnd_to_node=rng.integers(0, n, nb).astype(np.int32),
                    bnd_group=rng.integers(0, 9, nb).astype(np.int32), bnd_weights=rng.uniform(-0.4, 0.4, (nb, 3)))

    fine, coarse = level(n, n * deg // 2), level((n + 1) // 2, n * deg // 3)
    fine["node_to_mg_node"] = (np.arange(n) // 2).astype(np.int32)
    return [fine, coarse]


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    r.set_flux_variant(mgcfd.FLUX_VARIANTS["gather_exact"])
    yield r
    r.close()


@pytest.mark.parametrize("variant", ["gather_exact", "gather_fast", "part_coloured", "part_atomic", "mixed_coloured",
                                     "mixed_atomic"])
@pytest.mark.parametrize("n,deg", [(255, 4), (256, 6), (257, 6), (515, 2), (1100, 2), (1300, 4), (1500, 12)])
def test_fused_solve(rt, n, deg, variant):
    mesh = random_mesh(n, deg, seed=n + deg)
    o = Oracle("orc")
    state = perturbed_state(n, o.freestream(0.5, 3.0).ff_variable[:], seed=5)
    flux = [1e-9 * perturbed_state(len(lv["coords"]), np.ones(5), seed=6 + l) for l, lv in enumerate(mesh)]

    def after_setup(levels):
        levels[0]["var"][:] = state
        for l, a in enumerate(levels):
            a["flux"][:] = flux[l]

    cycles = 3
    ref = o.solve(mesh, cycles, 0.5, 3.0, after_setup=after_setup)
    for graph in (False, True):
        s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
        s.setup()
        rt.upload(s.lv[0].variables, state)
        for l in range(2):
            rt.upload(s.lv[l].fluxes, flux[l])
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        st, rms = s.run_device(cycles, use_graph=graph)
        assert st == ref["status"] == 0
        tol = MIXED_STATE_TOL if variant.startswith("mixed") else STATE_TOL
        for l in range(2):
            err = rel_err(s.state(l), ref["levels"][l]["variables"])
            assert err <= tol, f"level {l} graph {graph}: {err:.3e}"
            assert not s.state(l, "fluxes").any(), f"level {l}: flux not zero after the run"


def test_blocked_plan_blocks(rt):
    """Blocks of the blocked plan: whole 256-node patches where their halo has
    more than 256 and at most 448 nodes, quarters on a level of few patches,
    and smaller ones where the halo is beyond that."""
    import ctypes as C

    def stats(mesh, level):
        s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
        st = (C.c_int * 5)()
        mgcfd._check(rt.L.mgcfd_plan_stats(s.lv[level].edge_to_node, st), "mgcfd_plan_stats")
        return list(st)

    mesh = mgcfd.mesh_knn(70000, 217000, 2, seed=3)
    whole = stats(mesh, 1)
    assert whole[0] == -(-len(mesh[1]["coords"]) // 256) and 512 < whole[1] <= 704 and whole[4] == 80 * whole[1]
    quarter = stats(random_mesh(1100, 2, seed=1102), 0)
    assert quarter[0] == 18 and quarter[1] <= 64 + 128
    split = stats(random_mesh(1500, 12, seed=1512), 0)
    assert split[0] > 24 and split[1] <= 704


@pytest.mark.parametrize("variant", ["part_coloured", "mixed_coloured"])
@pytest.mark.parametrize("n,deg", [(257, 6), (1100, 2), (1300, 4)])
def test_part_shapes_change_nothing(rt, n, deg, variant):
    """Levels with few parts run smaller parts and more threads per part; a
    deterministic variant's state and RMS history do not depend on it, bit for
    bit."""
    mesh = random_mesh(n, deg, seed=n + deg)
    got = []
    # None: as the number of parts selects (64 nodes, 256 threads here)
    for config in (None, (256, 0), (256, 256), (256, 512), (128, 0), (128, 256), (64, 512)):
        s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
        s.setup()
        rt.upload(s.lv[0].variables, perturbed_state(n, s.fs["ff_variable"], seed=5))
        for l in range(2):
            if config:
                rt.map_part_config(s.lv[l].edge_to_node, *config)
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        st, rms = s.run_device(3)
        assert st == 0
        got.append((s.state(0), s.state(1), rms))
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("variant", ["gather_exact", "part_coloured", "mixed_coloured"])
@pytest.mark.parametrize("others", [1, 40, 90, 200])
def test_small_mesh_alone_and_in_a_batch(rt, others, variant):
    """Alone a small mesh's levels run quarter patches; beside others the batch
    has more patches and the shapes change (half and whole patches, fewer
    lanes and threads): its states and RMS history stay the same, bit for bit."""
    small, other = mgcfd.mesh_knn(1500, 4600, 2, seed=3), mgcfd.mesh_knn(700, 2100, 2, seed=4)

    def result(meshes):
        b = mgcfd.Batch(rt, meshes, [0.5] * len(meshes), [3.0] * len(meshes), variant)
        st, rms = b.run(5)
        out = [b.fetch(0, 0), b.fetch(0, 1), rms[0].copy()]
        b.close()
        assert not st.any()
        return out

    for a, b in zip(result([small]), result([small] + [other] * others)):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("variant", ["gather_exact", "part_coloured", "part_atomic", "nodal_exact"])
@pytest.mark.parametrize("level", [0, 1])
@pytest.mark.parametrize("graph", [False, True])
def test_abort_keeps_the_references_state(rt, level, graph, variant):
    """A negative minimum dt (a negative volume) on the second level, whose
    state a restriction has just made, or on the first: every level's
    variables are the reference's at its early return."""
    mesh = random_mesh(515, 4, seed=9)
    o = Oracle("orc")
    state = perturbed_state(515, o.freestream(0.5, 3.0).ff_variable[:], seed=5)
    vol = {}

    def after_setup(levels):
        levels[0]["var"][:] = state
        levels[level]["vol"][3] *= -1.0
        vol[0] = levels[level]["vol"].copy()

    ref = o.solve(mesh, 3, 0.5, 3.0, after_setup=after_setup)
    s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
    s.setup()
    rt.upload(s.lv[0].variables, state)
    rt.upload(s.lv[level].volumes, vol[0])
    rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
    st, _ = s.run_device(3, use_graph=graph)
    assert st == ref["status"] == 1
    for l in range(2):
        err = rel_err(s.state(l), ref["levels"][l]["variables"])
        assert err <= STATE_TOL, f"level {l}: {err:.3e}"
        if variant != "nodal_exact":    # its flux kernel has run by the time its stage kernel aborts
            assert not s.state(l, "fluxes").any()


@pytest.mark.parametrize("n", [65537, 80003, 97537, 131073])
def test_patches_beyond_the_last_full_round(rt, n):
    """Levels of more patches than CUs cut the patches beyond the last full
    round (257, 313, 382 and 513 patches on 256 CUs: quarters, quarters,
    halves, quarters).  Against the oracle, and the coloured variants bit for
    bit as with whole patches."""
    import ctypes as C

    mesh = mgcfd.mesh_knn(n, int(3.1 * n), 2, seed=n)
    o = Oracle("orc")
    state = perturbed_state(n, o.freestream(0.5, 3.0).ff_variable[:], seed=5)
    ref = o.solve(mesh, 2, 0.5, 3.0, after_setup=lambda lv: lv[0]["var"].__setitem__(slice(None), state))

    def solve(variant, part_nodes=0):
        s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
        s.setup()
        rt.upload(s.lv[0].variables, state)
        if part_nodes:
            for l in range(2):
                rt.map_part_config(s.lv[l].edge_to_node, part_nodes, 0)
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
        st, rms = s.run_device(2)
        assert st == 0
        stats = (C.c_int * 6)()
        if not variant.startswith("gather"):
            mgcfd._check(rt.L.mgcfd_part_plan_stats(s.lv[0].edge_to_node, stats), "mgcfd_part_plan_stats")
        return s.state(0), s.state(1), rms, stats[0]

    for variant in ("gather_exact", "gather_fast", "part_atomic", "part_coloured", "mixed_coloured"):
        got = solve(variant)
        tol = MIXED_STATE_TOL if variant.startswith("mixed") else STATE_TOL
        for l in range(2):
            assert rel_err(got[l], ref["levels"][l]["variables"]) <= tol, (variant, l)
        if variant.endswith("coloured"):
            whole = solve(variant, 256)
            assert got[3] > whole[3] == -(-n // 256)
            for a, b in zip(got[:3], whole):
                assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), variant
