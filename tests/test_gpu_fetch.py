"""Fetches (op_fetch_data_char, mgcfd_batch_fetch): the device undoes the
internal element order while it writes 2 MB pieces to pinned memory.  Sizes sit
at the edges of a piece (52,428 rows of five doubles, 524,288 ints) and need
one, a few and more pieces than there are buffers (eight); every value has to
come back as it was declared."""
import numpy as np
import pytest

import mgcfd

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


def ring(rt, n, seed):
    """A set of n elements with an internal order of its own (a ring of edges
    through a random permutation)."""
    order = np.random.default_rng(seed).permutation(n).astype(np.int32)
    nodes, edges = rt.decl_set(n, "nodes"), rt.decl_set(n, "edges")
    rt.decl_map(edges, nodes, 2, np.stack([order, np.roll(order, 1)], 1), "edge-->node")
    xyz = rt.decl_dat(nodes, 3, np.random.default_rng(seed).uniform(size=(n, 3)), "xyz")
    rt.partition(nodes, xyz)
    return nodes, edges


@pytest.mark.parametrize("n,dim,typ", [(1, 5, "double"), (52428, 5, "double"), (52429, 5, "double"),
                                       (524288, 1, "int"), (524289, 1, "int"), (87382, 3, "double"),
                                       (120001, 7, "double"), (500000, 5, "double")])
@pytest.mark.parametrize("ordered", [False, True])
def test_fetch_returns_what_was_declared(rt, n, dim, typ, ordered):
    rng = np.random.default_rng(n + dim)
    data = rng.integers(-2**31, 2**31, (n, dim)).astype(np.int32) if typ == "int" else rng.normal(size=(n, dim))
    st = ring(rt, n, 3)[0] if ordered and n > 1 else rt.decl_set(n, "alone")
    d = rt.decl_dat(st, dim, data, "d", typ)
    for _ in range(2):
        assert np.array_equal(rt.fetch(d), data)
    other = data[::-1].copy()
    rt.upload(d, other)
    assert np.array_equal(rt.fetch(d), other)


def test_batch_fetch_gives_each_mesh_its_own_nodes(rt):
    """Freestream states differ by mesh; volumes differ by node: both come back
    in the mesh's order whatever its place in the batch."""
    meshes = [mgcfd.mesh_knn(n, 3 * n, 2, seed=n) for n in (300, 1000, 60000)]
    alone = []
    for m in meshes:
        b = mgcfd.Batch(rt, [m], [0.5], [3.0])
        alone.append([b.fetch(0, l, "volumes") for l in range(2)])
        b.close()
    b = mgcfd.Batch(rt, meshes, [0.4, 0.5, 0.6], [1.0, 2.0, 3.0])
    for i, mach in enumerate((0.4, 0.5, 0.6)):
        for l in range(2):
            assert np.array_equal(b.fetch(i, l, "volumes"), alone[i][l])
        ff = mgcfd.freestream(mach, float(i + 1))["ff_variable"]
        assert np.allclose(b.fetch(i, 0), ff[None, :], rtol=1e-14, atol=0)
    b.close()
