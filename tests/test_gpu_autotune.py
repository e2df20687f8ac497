"""The batch autotuner's trials and the part configurations it chooses from."""
import ctypes as C

import numpy as np
import pytest

import mgcfd
from test_gpu_graphs import bits, replays

pytestmark = pytest.mark.gpu

CANDIDATES = 7          # configurations tried on each level


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


@pytest.mark.parametrize("iters", [1, 2, 5])
@pytest.mark.parametrize("levels", [1, 3])
def test_trials_are_replays(rt, iters, levels):
    """Every timed cycle of a trial is a replay, after as many that are not timed
    and two that capture it (the first of the first trial has no graph); the
    runs after the tuning are those of a batch not tuned."""
    meshes = [m[:levels] for m in (mgcfd.mesh_box(8, 3, seed=7), mgcfd.mesh_knn(3000, 9300, 3, seed=3))]
    tuned, plain = (mgcfd.Batch(rt, meshes, [0.5, 0.7], [3.0, -1.5], "part_coloured") for _ in range(2))
    before = replays(rt)
    tuned.autotune(iters)
    assert replays(rt) - before == levels * CANDIDATES * (2 * iters + 2) - 1
    for _ in range(2):
        (st, rms), (st2, rms2) = tuned.run(5), plain.run(5, use_graph=False)
        assert not st.any() and not st2.any() and np.array_equal(bits(rms), bits(rms2))
        for i in range(2):
            for l in range(levels):
                for what in ("variables", "step_factors", "fluxes"):
                    assert np.array_equal(bits(tuned.fetch(i, l, what)), bits(plain.fetch(i, l, what)))
    tuned.close()
    plain.close()
