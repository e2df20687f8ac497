"""Elementwise loops over more doubles than one launch has threads (2^32 - 1):
sets of more than 858,993,459 elements.  Values are checked through the
library's own reductions, which read every double."""
import ctypes as C

import numpy as np
import pytest

import mgcfd

pytestmark = pytest.mark.gpu

N = 858_993_459 + 1_000_001
NEEDED = 150 << 30           # three [N][5] arrays of doubles, and one of [N]


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert r.L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0      # of the HIP runtime the library is linked to
    if free.value < NEEDED:
        r.close()
        pytest.skip("needs 150 GiB of free device memory")
    yield r
    r.close()


def test_elementwise_loops_beyond_one_launch(rt):
    """Residual, time step, the restriction's mean, copy and reset, from states
    whose every value is 1: sums of squares are whole numbers, exact in FP64
    in any order."""
    st = rt.decl_set(N, "s")
    a, b, c = (rt.decl_dat(st, 5, None, k) for k in "abc")
    rt.decl_const("ff_variable", np.ones(5))

    def fill(d, one):
        rt.par_loop("initialize_variables_kernel" if one else "zero_5d_array_kernel", st,
                    rt.arg(d, -1, None, 5, acc=mgcfd.OP_WRITE))

    def sumsq(d):
        g = np.array([0.0])
        rt.par_loop("calc_rms_kernel", st, rt.arg(d, -1, None, 5, acc=mgcfd.OP_READ), rt.gbl(g, mgcfd.OP_INC))
        return g[0]

    fill(a, True)
    rt.par_loop("residual_kernel", st, rt.arg(b, -1, None, 5, acc=mgcfd.OP_READ),
                rt.arg(a, -1, None, 5, acc=mgcfd.OP_READ), rt.arg(c, -1, None, 5, acc=mgcfd.OP_WRITE))
    assert sumsq(c) == 5.0 * N
    # c = old + sf / 4 * flux with sf 0: the old state
    sf = rt.decl_dat(st, 1, None, "sf")
    fill(b, True)
    fill(c, False)
    rt.par_loop("time_step_kernel", st, rt.gbl(np.array([0], dtype=np.int32), mgcfd.OP_READ),
                rt.arg(sf, -1, None, 1, acc=mgcfd.OP_READ), rt.arg(b, -1, None, 5, acc=mgcfd.OP_RW),
                rt.arg(a, -1, None, 5, acc=mgcfd.OP_READ), rt.arg(c, -1, None, 5, acc=mgcfd.OP_WRITE))
    assert sumsq(c) == 5.0 * N
    assert sumsq(b) == 0.0                       # the flux is reset everywhere
    kids = rt.decl_dat(st, 1, None, "kids", "int")
    rt.par_loop("up_post_kernel", st, rt.arg(c, -1, None, 5, acc=mgcfd.OP_RW),
                rt.arg(kids, -1, None, 1, "int", mgcfd.OP_READ))
    assert sumsq(c) == 5.0 * N
    fill(b, True)
    rt.par_loop("copy_double_kernel", st, rt.arg(b, -1, None, 5, acc=mgcfd.OP_READ),
                rt.arg(a, -1, None, 5, acc=mgcfd.OP_WRITE))
    assert sumsq(a) == 5.0 * N
    rt.par_loop("down_v2_kernel_pre", st, rt.arg(sf, -1, None, 1, acc=mgcfd.OP_WRITE),
                rt.arg(a, -1, None, 5, acc=mgcfd.OP_WRITE))
    assert sumsq(a) == 0.0
