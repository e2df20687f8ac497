"""Fetches beyond what the pinned landing buffers are made for."""
import numpy as np
import pytest

import hip_shim
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


PREPARE = """
import mgcfd
from test_gpu_fetch import ring
rt = mgcfd.Runtime()
n = 300000
st = ring(rt, n, 3)[0]
data = np.random.default_rng(1).normal(size=(n, 5))
d = rt.decl_dat(st, 5, data, "d")
mgcfd._check(rt.L.op_renumber(None), "op_renumber")
"""


def test_fetch_needs_no_device_memory(tmp_path):
    """Device memory is gone when a set's first dat is fetched; a later fetch,
    with memory again, takes the buffers; no error is left for later calls."""
    hip_shim.run_script(tmp_path, PREPARE + """
shim.shim_refuse_device(1)
for _ in range(2):
    assert np.array_equal(rt.fetch(d), data)
rt.sync()
rt.par_loop("zero_5d_array_kernel", st, rt.arg(d, -1, None, 5, acc=mgcfd.OP_WRITE))
assert not rt.fetch(d).any()
rt.upload(d, data)
shim.shim_refuse_device(0)
assert np.array_equal(rt.fetch(d), data)
print("ok")
""")


@pytest.mark.parametrize("left", [0, 1, 3])
def test_fetch_with_fewer_pinned_buffers(tmp_path, left):
    """Six buffers' worth of pieces with none, one or three buffers to be had."""
    hip_shim.run_script(tmp_path, PREPARE + f"""
shim.shim_pinned_left({left})
for _ in range(2):
    assert np.array_equal(rt.fetch(d), data)
shim.shim_pinned_left(-1)
assert np.array_equal(rt.fetch(d), data)
print("ok")
""")


def test_fetch_without_further_threads(tmp_path):
    """No thread can be started (a limit that holds for ordinary users): the
    calling thread copies every piece."""
    hip_shim.run_script(tmp_path, PREPARE + """
import resource, threading
assert np.array_equal(rt.fetch(d), data)
resource.setrlimit(resource.RLIMIT_NPROC, (1, resource.getrlimit(resource.RLIMIT_NPROC)[1]))
try:
    threading.Thread(target=int).start()
    print("threads still start")
except RuntimeError:
    print("no threads")
for _ in range(2):
    assert np.array_equal(rt.fetch(d), data)
print("ok")
""")


@pytest.mark.parametrize("n", [1000, 300000])
def test_fetch_from_a_thread_on_another_device(tmp_path, n):
    """The library on the second of two devices (one, shown as two): the first
    fetch, made by a thread that has chosen no device, allocates and launches
    on the library's; the thread's own choice is left alone."""
    hip_shim.run_script(tmp_path, "shim.shim_devices(2)\n" + PREPARE.replace("n = 300000", f"n = {n}") + """
import ctypes as C, threading
got = []
def work():
    got.append(rt.fetch(d))
    dev = C.c_int(-1)
    shim.hipGetDevice(C.byref(dev))
    got.append(dev.value)
shim.shim_expect(1)
t = threading.Thread(target=work)
t.start()
t.join()
assert shim.shim_misplaced() == 0, shim.shim_misplaced()
assert np.array_equal(got[0], data) and got[1] == 0
print("ok")
""", MGCFD_DEVICE="1")
