"""Edge fluxes of states in other units: the flux is linear in density,
momentum and energy together, so a state scaled by a power of two has its flux
scaled by the same, as far as the exponents reach (momenta beyond 1e+-154
have squares that FP64 does not hold)."""
import numpy as np
import pytest

import mgcfd
from conftest import perturbed_state
from test_gpu_parity import FLUX_FAST_TOL, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


@pytest.mark.parametrize("variant", ["gather_exact", "gather_fast", "nodal_exact", "part_coloured", "part_atomic",
                                     "atomic"])
def test_flux_of_scaled_states(rt, variant):
    m = mgcfd.mesh_knn(3000, 9300, 1, seed=8)
    s = mgcfd.Solver(rt, m, 0.5, 3.0)
    s.setup()
    rt.set_flux_variant(mgcfd.FLUX_VARIANTS[variant])
    var = perturbed_state(3000, s.fs["ff_variable"], seed=11)

    def flux(scale):
        rt.upload(s.lv[0].variables, var * scale)
        rt.upload(s.lv[0].fluxes, np.zeros((3000, 5)))
        s.flux_edge(0)
        return s.state(0, "fluxes") / scale

    one = flux(1.0)
    assert np.isfinite(one).all() and np.abs(one).max() > 0
    for e in (-600, -520, 520, 600):
        got = flux(2.0 ** e)
        if variant.endswith("exact"):
            assert np.array_equal(got, one), e
        else:
            assert rel_err(got, one) <= FLUX_FAST_TOL, e
