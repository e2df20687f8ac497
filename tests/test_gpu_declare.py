"""Dats declared without data start as zeros, and what the first loop writes
into them stays: the zeros are in place before any loop's stream runs."""
import numpy as np
import pytest

import mgcfd

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


def sumsq(rt, st, d):
    g = np.array([0.0])
    rt.par_loop("calc_rms_kernel", st, rt.arg(d, -1, None, 5, acc=mgcfd.OP_READ), rt.gbl(g, mgcfd.OP_INC))
    return g[0]


@pytest.mark.parametrize("n", [1000, 100_000_000])
@pytest.mark.parametrize("late", [False, True])
def test_first_loop_follows_the_zeros(rt, n, late):
    """Ones written by the first loop after the declarations are all there
    (sums of ones are exact), and the dats not written hold zeros.  late: the
    dats are declared on a set that has run a loop already."""
    st = rt.decl_set(n, "s")
    if late:
        rt.par_loop("zero_1d_array_kernel", st, rt.arg(rt.decl_dat(st, 1, None, "x"), -1, None, 1, acc=mgcfd.OP_WRITE))
        rt.sync()
    rt.decl_const("ff_variable", np.ones(5))
    dats = [rt.decl_dat(st, 5, None, f"d{i}") for i in range(3)]
    for d in (dats[2], dats[0]):
        rt.par_loop("initialize_variables_kernel", st, rt.arg(d, -1, None, 5, acc=mgcfd.OP_WRITE))
    assert [sumsq(rt, st, d) for d in dats] == [5.0 * n, 0.0, 5.0 * n]


def test_first_loop_follows_an_upload(rt):
    """A loop right after op_upload_data reads all of the new values."""
    n = 10_000_000
    st = rt.decl_set(n, "s")
    d = rt.decl_dat(st, 5, None, "d")
    ones, twos = np.ones((n, 5)), np.full((n, 5), 2.0)
    for _ in range(3):
        rt.upload(d, ones)
        assert sumsq(rt, st, d) == 5.0 * n
        rt.upload(d, twos)
        assert sumsq(rt, st, d) == 20.0 * n
