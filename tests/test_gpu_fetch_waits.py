"""Fetches from several threads: a fetch waits for the work queued on its own
stream, not for another caller's."""
import threading
import time

import numpy as np
import pytest

import mgcfd

pytestmark = pytest.mark.gpu


@pytest.fixture
def rt():
    r = mgcfd.Runtime()
    yield r
    r.close()


def test_fetch_does_not_wait_for_another_streams_work(rt):
    """The library's stream holds about 0.3 s of queued loops; a thread that
    fetches from it waits for them, a thread that fetches a finished batch
    (a stream of its own) meanwhile does not."""
    n = 20_000_000
    st = rt.decl_set(n, "s")
    a, b, c = (rt.decl_dat(st, 5, None, k) for k in "abc")
    small = rt.decl_dat(rt.decl_set(3, "t"), 5, np.ones((3, 5)), "small")
    batch = mgcfd.Batch(rt, [mgcfd.mesh_knn(3000, 9300, 2, seed=3)], [0.5], [3.0])
    batch.run(2)
    ref = batch.fetch(0, 0)
    assert (rt.fetch(small) == 1.0).all()

    def loops(k):
        for _ in range(k):
            rt.par_loop("residual_kernel", st, rt.arg(a, -1, None, 5, acc=mgcfd.OP_READ),
                        rt.arg(b, -1, None, 5, acc=mgcfd.OP_READ), rt.arg(c, -1, None, 5, acc=mgcfd.OP_WRITE))

    loops(5)
    rt.sync()
    t0 = time.perf_counter()
    loops(20)
    rt.sync()
    per = (time.perf_counter() - t0) / 20
    done = {}

    def waiting():
        assert (rt.fetch(small) == 1.0).all()
        done["queued"] = time.perf_counter()

    loops(max(50, int(0.3 / per)))
    t = threading.Thread(target=waiting)
    t.start()
    time.sleep(0.05)
    assert "queued" not in done
    got = batch.fetch(0, 0)
    done["own"] = time.perf_counter()
    t.join()
    batch.close()
    assert np.array_equal(got, ref)
    assert done["own"] < done["queued"] - 0.05, done
