"""Reading fields back on the GPU: arrays on both sides of 16 MiB, from which they pass
through the pinned ring in chunks of 4 MiB, arrive as they were sent, whatever memory
takes them."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solver(nx, ny, nz):
    import cfd_nssolver_forhpc_flowpassingcylinder_amd as pkg
    return pkg.FlowSolver(pkg.default_config(nx=nx, ny=ny, nz=nz, lx=4.0, ly=4.0, lz=4.0,
                                             grid_kind=0, re=100.0, dt=1e-3, z_periodic=1))


def _fields(n, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(n) for _ in range(3)]


# (nx + 4)(ny + 4)(nz + 4) doubles an array: 16 MiB less a row, 16 MiB, one row more, a
# last chunk of five rows, 36 MiB, 73 MB
@pytest.mark.parametrize("nx,ny,nz", [(123, 124, 124), (124, 124, 124), (125, 124, 124),
                                      (81, 124, 237), (284, 124, 124), (512, 256, 64)])
def test_arrays_arrive(nx, ny, nz):
    s = _solver(nx, ny, nz)
    sent = _fields(s.G, nx)
    for _ in range(2):
        s.upload_velocity(1, *sent)
        for a, b in zip(s.download_velocity(1), sent):
            assert np.array_equal(a, b)
        sent = sent[1:] + sent[:1]
    s.set_pressure(sent[2])
    assert np.array_equal(s.pressure(), sent[2])


def _p(a, off=0):
    return C.cast(a.ctypes.data + off, C.POINTER(C.c_double))


def test_destinations():
    """Memory off a page's and a double's alignment, one array for all three components
    (the last one stays), and pinned memory, where the copies go one after the other."""
    s = _solver(140, 140, 124)
    n = s.G
    sent = _fields(n, 1)
    s.upload_velocity(0, *sent)
    raw = [np.zeros(8 * n + 16, np.uint8) for _ in range(3)]
    assert s.L.cfdmx_download_velocity(s.h, 0, _p(raw[0], 4), _p(raw[1], 8), _p(raw[2], 12)) == 0
    for q in range(3):
        at = 4 * (q + 1)
        assert raw[q][at:at + 8 * n].tobytes() == sent[q].tobytes()
        assert not raw[q][:at].any() and not raw[q][at + 8 * n:].any()
    one = np.zeros(n)
    assert s.L.cfdmx_download_velocity(s.h, 0, _p(one), _p(one), _p(one)) == 0
    assert np.array_equal(one, sent[2])
    mem = C.c_void_p()
    assert s.L.hipHostMalloc(C.byref(mem), C.c_size_t(8 * n), C.c_uint(0)) == 0
    pin = np.ctypeslib.as_array(C.cast(mem, C.POINTER(C.c_double)), (n,))
    assert s.L.cfdmx_download_velocity(s.h, 0, _p(pin), _p(raw[1], 8), _p(raw[2], 12)) == 0
    assert np.array_equal(pin, sent[0])
    assert s.L.cfdmx_download_velocity(s.h, 0, _p(pin), None, _p(raw[2], 12)) != 0
    del pin
    assert s.L.hipHostFree(mem) == 0


def test_threads():
    """Two threads read one context, two more a context each."""
    s = [_solver(140, 140, 124) for _ in range(3)]
    sent = [_fields(c.G, 10 + k) for k, c in enumerate(s)]
    for c, f in zip(s, sent):
        c.upload_velocity(0, *f)
    bad = []

    def read(k):
        for _ in range(4):
            got = s[k].download_velocity(0)
            if not all(np.array_equal(a, b) for a, b in zip(got, sent[k])):
                bad.append(k)

    ts = [threading.Thread(target=read, args=(k,)) for k in (0, 0, 1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
