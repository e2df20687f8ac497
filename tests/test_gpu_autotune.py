"""The batch autotuner's trials and the part configurations it chooses from."""
import ctypes as C

import numpy as np
import pytest

import hip_shim
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


PREPARE = """
import mgcfd
rt = mgcfd.Runtime()
b = mgcfd.Batch(rt, [mgcfd.mesh_knn(10007, 31000, 2, seed=5)], [0.5], [3.0], "part_atomic")
def shapes():
    b.run(1, use_graph=False)            # packs the plans' weights
    return hip_shim.launch_shapes(shim, lambda: b.run(1, use_graph=False))
own = shapes()
for l in range(2):
    b.set_part_config(l, 128, 512)
other = shapes()
# level 0's 40 patches of 256 nodes as quarters with 256 threads; as halves with 512
assert (157, 256) in own - other and (79, 512) in other - own, (own, other)
"""


def test_own_shape_can_be_returned_to(tmp_path):
    """A small level's own shape, smaller parts than any that can be set with
    as many threads, is what (256, 256, 0) selects after another was set."""
    hip_shim.run_script(tmp_path, PREPARE + """
for l in range(2):
    b.set_part_config(l, 256, 256)
assert shapes() == own
print("ok")
""")


def test_own_shape_is_tried(tmp_path):
    """Tuning tries each level's own shape, also when another was set before."""
    hip_shim.run_script(tmp_path, PREPARE + """
tried = hip_shim.launch_shapes(shim, lambda: b.autotune(1))
assert own <= tried, (own - tried)
print("ok")
""")


def test_map_part_config_zero_is_the_default_shape(rt):
    mesh = mgcfd.mesh_knn(10007, 31000, 2, seed=5)
    s = mgcfd.Solver(rt, mesh, 0.5, 3.0)
    s.setup()

    def stats(l):
        out = (C.c_int * 6)()
        mgcfd._check(rt.L.mgcfd_part_plan_stats(s.lv[l].edge_to_node, out), "mgcfd_part_plan_stats")
        return list(out)

    own = [stats(l) for l in range(2)]
    for l in range(2):
        rt.map_part_config(s.lv[l].edge_to_node, 256)
        assert stats(l)[0] == -(-len(mesh[l]["coords"]) // 256) < own[l][0]
        rt.map_part_config(s.lv[l].edge_to_node, 0)
        assert stats(l) == own[l]
    for bad in (-1, 1, 15, 257):
        with pytest.raises(mgcfd.MgcfdError, match="nodes per part"):
            rt.map_part_config(s.lv[0].edge_to_node, bad)


def test_batch_part_config_limits(rt):
    b = mgcfd.Batch(rt, [mgcfd.mesh_knn(1200, 3720, 2, seed=4)], [0.5], [3.0], "part_atomic")
    for bad in ((0, 256, 0), (15, 256, 0), (257, 256, 0), (256, 0, 0), (256, 1024, 0), (256, 256, 9)):
        with pytest.raises(mgcfd.MgcfdError):
            b.set_part_config(0, *bad)
    b.close()
