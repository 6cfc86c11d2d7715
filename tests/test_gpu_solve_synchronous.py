"""bx_helm_solve is synchronous: when it returns, its stream is idle and the
solution can be read on any other stream, however the solve ended -- an iterate
in either of the two arrays that multigrid iterations alternate between, an
iteration launched past the end.  Both streams are non-blocking, so nothing
else orders the read behind the solve."""
import ctypes

import numpy as np
import pytest

from bamrex_amd import _lib
from bamrex_amd.imex import dev

from conftest import announce
from test_gpu_multigrid_ahead import solver, system

pytestmark = pytest.mark.gpu

HIP_STREAM_NON_BLOCKING = 1
HIP_MEMCPY_DEVICE_TO_HOST = 2


def hip(name, *args):
    """A HIP runtime call (the library's own dependency)."""
    f = getattr(_lib.lib(), name)
    f.restype = ctypes.c_int
    return f(*args)


@pytest.fixture
def streams():
    s = [ctypes.c_void_p() for _ in range(2)]
    for q in s:
        assert hip("hipStreamCreateWithFlags", ctypes.byref(q), HIP_STREAM_NON_BLOCKING) == 0
    yield s
    for q in s:
        assert hip("hipStreamDestroy", q) == 0


# 160 x 96: small tiles, the iteration ends in the last smoothing's launch; 64 x 64:
# the whole hierarchy in the tail; 1024 x 264: large tiles, a residual of its own.
# maxiter 1, 2, 3: odd and even; 60: a solve that converges
@pytest.mark.parametrize("method", ["mg_fused", "mg", "fgmres_mg"])
@pytest.mark.parametrize("nx,ny", [(160, 96), (64, 64), (1024, 264)], ids=str)
def test_solution_is_there_on_return(streams, nx, ny, method):
    announce("synchronous solve %s %dx%d" % (method, nx, ny))
    solving, reading = streams
    sy = system(nx, ny, 13, False)
    b, zero = dev(sy[4]), np.zeros((ny, nx))
    s = solver(nx, ny, sy, 1e-3)
    x = dev(zero)
    for maxiter in ((60,) if method == "fgmres_mg" else (1, 2, 3, 60)):
        x.upload(zero)
        assert hip("hipDeviceSynchronize") == 0
        st = _lib.bx_solve_stats()
        rc = _lib.lib().bx_helm_solve(s.h, b.ptr, x.ptr, _lib.BX_SOLVE[method], 1e-10, maxiter,
                                      ctypes.byref(st), solving)
        idle = hip("hipStreamQuery", solving)
        got = np.empty((ny, nx))
        copied = hip("hipMemcpyAsync", ctypes.c_void_p(got.ctypes.data), x.ptr,
                     ctypes.c_size_t(got.nbytes), HIP_MEMCPY_DEVICE_TO_HOST, reading)
        assert hip("hipStreamSynchronize", reading) == 0
        assert (rc, copied, idle) == (0, 0, 0)
        assert st.iters == maxiter or st.converged
        x.upload(zero)
        assert s.solve(b, x, method, maxiter=maxiter)["iters"] == st.iters
        assert np.array_equal(got, x.download())
    s.close()
