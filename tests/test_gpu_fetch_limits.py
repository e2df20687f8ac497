"""Fetches beyond what the pinned landing buffers are made for."""
import numpy as np
import pytest

import mgcfd
from test_gpu_fetch import ring

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


@pytest.mark.parametrize("dim,typ", [(262144, "double"), (262145, "double"), (300001, "double"), (524289, "int")])
@pytest.mark.parametrize("ordered", [False, True])
def test_elements_larger_than_a_buffer(rt, dim, typ, ordered):
    """An element that fills a 2 MB buffer exactly, and larger ones, after an
    ordinary fetch has made the buffers."""
    n = 37
    rng = np.random.default_rng(dim)
    st = ring(rt, n, 3)[0] if ordered else rt.decl_set(n, "alone")
    data = rng.integers(-2**31, 2**31, (n, dim)).astype(np.int32) if typ == "int" else rng.normal(size=(n, dim))
    d, little = rt.decl_dat(st, dim, data, "d", typ), rt.decl_dat(st, 5, rng.normal(size=(n, 5)), "little")
    assert rt.fetch(little).shape == (n, 5)
    assert np.array_equal(rt.fetch(d), data)
