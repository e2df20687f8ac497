"""The standalone reduction loops and the elementwise loops through the C ABI,
at the sizes where their grids change: one value, a workgroup's edge, the
largest grid of one value per thread, and beyond it, where each thread takes
a strided share.

Minima, counts and the elementwise loops are exact (one IEEE operation after
the other, as numpy does them).  The sum of squares is compared with
math.fsum: a thread adds ceil(5 n / 2^18) terms, its workgroup at most 4 + 8
levels, the host 256 partials per running sum and 3 more, each addition within
2^-53 of the sum of positive terms, so the relative error is at most
(1 + terms + 12 + 259) * 2^-53 (the first for the squares).
"""
import math

import numpy as np
import pytest

import mgcfd

pytestmark = pytest.mark.gpu

O = mgcfd.OP_READ
SIZES = [1, 51, 52, 256, 257, 52428, 52429, 262144, 262145, 300001]


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


@pytest.mark.parametrize("n", SIZES)
def test_reduction_loops(rt, n):
    rng = np.random.default_rng(n)
    dt = rng.uniform(1e-3, 2.0, (n, 1))
    x = rng.normal(size=(n, 5)) * 1e-4
    x[rng.integers(0, n, max(1, n // 9)), rng.integers(0, 5)] = 0.0
    st = rt.decl_set(n, "s")
    d1, d5 = rt.decl_dat(st, 1, dt, "dt"), rt.decl_dat(st, 5, x, "x")

    def least():
        g = np.array([np.finfo(np.float64).max])
        rt.par_loop("get_min_dt_kernel", st, rt.arg(d1, -1, None, 1, acc=O), rt.gbl(g, mgcfd.OP_MIN))
        return g[0]

    def count(loop):
        c = np.array([3], dtype=np.int32)
        rt.par_loop(loop, st, rt.arg(d5, -1, None, 5, acc=O), rt.gbl(c, mgcfd.OP_INC))
        return c[0] - 3

    assert least() == dt.min()
    for at in (0, n - 1):                       # a minimum in the first and in the last place
        low = dt.copy()
        low[at] = -1e-9
        rt.upload(d1, low)
        assert least() == -1e-9
    g = np.array([0.5])
    rt.par_loop("calc_rms_kernel", st, rt.arg(d5, -1, None, 5, acc=O), rt.gbl(g, mgcfd.OP_INC))
    ref = math.fsum((x * x).ravel().tolist() + [0.5])
    assert abs(g[0] - ref) <= (1 + math.ceil(5 * n / 2**18) + 12 + 259) * 2.0**-53 * ref
    assert count("count_non_zeros") == int((x > 0.0).sum())
    assert count("count_bad_vals") == 0
    x[0, 0], x[n - 1, 4], x[n // 2, 2] = np.nan, np.inf, -np.inf
    rt.upload(d5, x)
    assert count("count_bad_vals") == 3
    assert count("count_non_zeros") == int((x > 0.0).sum())


@pytest.mark.parametrize("n", SIZES)
def test_elementwise_loops(rt, n):
    rng = np.random.default_rng(n + 1)
    st = rt.decl_set(n, "s")
    old, var, flux = (rng.normal(size=(n, 5)) for _ in range(3))
    sf = rng.uniform(0.1, 1.0, (n, 1))
    kids = rng.integers(0, 9, (n, 1)).astype(np.int32)
    d = {k: rt.decl_dat(st, v.shape[1], v, k, "int" if k == "kids" else "double")
         for k, v in
         dict(old=old, var=var, flux=flux, res=np.zeros((n, 5)), sf=sf, kids=kids).items()}
    rt.par_loop("residual_kernel", st, rt.arg(d["old"], -1, None, 5, acc=O), rt.arg(d["var"], -1, None, 5, acc=O),
                rt.arg(d["res"], -1, None, 5, acc=mgcfd.OP_WRITE))
    assert np.array_equal(rt.fetch(d["res"]), var - old)
    for rk in range(3):
        rt.upload(d["flux"], flux)
        rt.par_loop("time_step_kernel", st, rt.gbl(np.array([rk], dtype=np.int32), O),
                    rt.arg(d["sf"], -1, None, 1, acc=O), rt.arg(d["flux"], -1, None, 5, acc=mgcfd.OP_RW),
                    rt.arg(d["old"], -1, None, 5, acc=O), rt.arg(d["var"], -1, None, 5, acc=mgcfd.OP_WRITE))
        new = old + (sf / (4 - rk)) * flux
        assert np.array_equal(rt.fetch(d["var"]), new)
        assert not rt.fetch(d["flux"]).any()
    rt.par_loop("up_post_kernel", st, rt.arg(d["var"], -1, None, 5, acc=mgcfd.OP_RW),
                rt.arg(d["kids"], -1, None, 1, "int", O))
    assert np.array_equal(rt.fetch(d["var"]), new * (1.0 / np.maximum(kids, 1)))
