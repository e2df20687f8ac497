"""The blocked gather's shapes (nodes per block, lanes per node, halo nodes per
thread) follow the number of a level's blocks, so a mesh's shapes depend on
the batch it is in; the values of the fast form must not, as the exact form's
do not."""
import numpy as np
import pytest

import mgcfd
from conftest import perturbed_state
from oracle import Oracle
from test_gpu_parity import FLUX_FAST_TOL, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


@pytest.mark.parametrize("others", [1, 40, 90, 200])
def test_fast_gather_alone_and_in_a_batch(rt, others):
    small, other = mgcfd.mesh_knn(1500, 4600, 2, seed=3), mgcfd.mesh_knn(700, 2100, 2, seed=4)

    def result(meshes):
        b = mgcfd.Batch(rt, meshes, [0.5] * len(meshes), [3.0] * len(meshes), "gather_fast")
        st, rms = b.run(5)
        out = [b.fetch(0, 0), b.fetch(0, 1), rms[0].copy()]
        b.close()
        assert not st.any()
        return out

    for a, b in zip(result([small]), result([small] + [other] * others)):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("copies", [1, 4, 8, 20])
def test_fast_flux_of_a_mesh_and_of_copies_of_it(rt, copies):
    """One edge-flux pass over a disturbed state: a mesh alone, and several
    unconnected copies of it in one level (more blocks, other shapes)."""
    m = mgcfd.mesh_knn(5000, 15500, 1, seed=8)[0]
    o = Oracle("orc")
    var = perturbed_state(5000, o.freestream(0.5, 3.0).ff_variable[:], seed=11)

    def flux(k, w):
        big = dict(m)
        n, nb = 5000, len(m["bnd_to_node"])
        big["coords"] = np.concatenate([m["coords"] + [10.0 * i, 0, 0] for i in range(k)])
        big["edge_to_node"] = np.concatenate([m["edge_to_node"] + n * i for i in range(k)]).astype(np.int32)
        big["edge_weights"] = np.concatenate([m["edge_weights"]] * k)
        big["bnd_to_node"] = np.concatenate([m["bnd_to_node"] + n * i for i in range(k)]).astype(np.int32)
        big["bnd_group"] = np.concatenate([m["bnd_group"]] * k)
        big["bnd_weights"] = np.concatenate([m["bnd_weights"]] * k)
        s = mgcfd.Solver(rt, [big], 0.5, 3.0)
        s.setup()
        rt.upload(s.lv[0].variables, np.concatenate([var] * k))
        if w is not None:            # the set-up's weights depend on the coordinates' rounding
            rt.upload(s.lv[0].edge_weights, np.concatenate([w] * k))
        rt.set_flux_variant(mgcfd.FLUX_VARIANTS["gather_fast"])
        s.flux_edge(0)
        return s.state(0, "fluxes"), s.state(0, "edge_weights")

    one, w = flux(1, None)
    many, _ = flux(copies, w)
    for i in range(copies):
        part = np.ascontiguousarray(many[5000 * i:5000 * (i + 1)])
        assert np.array_equal(part.view(np.uint64), one.view(np.uint64)), i
    ref = np.zeros((5000, 5))
    o.compute_flux_edge(np.ascontiguousarray(m["edge_to_node"], np.int32), var, np.ascontiguousarray(w), ref,
                        o.freestream(0.5, 3.0))
    assert rel_err(one, ref) <= FLUX_FAST_TOL
