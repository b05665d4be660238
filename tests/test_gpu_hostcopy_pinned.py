"""Pinned host arrays move without the handle's own pinned slots, pageable ones through them;
both arrive whole, and the arrays' padding stays as the caller had it."""
import ctypes

import numpy as np
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu


def pinned_bytes(st):
    f = gpu.lib().gr_internal_pinned_bytes
    f.restype, f.argtypes = ctypes.c_longlong, [ctypes.c_void_p]
    return f(st._h)


def _array(torch, pinned, shape, dt, fill=None):
    a = torch.empty(shape, dtype=torch.float64 if dt == np.float64 else torch.float32, pin_memory=pinned).numpy()
    a[...] = np.random.default_rng(shape[0]).random(shape) if fill is None else fill
    return a


@pytest.mark.parametrize("dtype,nx,ny,nz,pad", [(gpu.GR_F64, 131, 67, 130, 7), (gpu.GR_F32, 518, 61, 100, 2),
                                                (gpu.GR_F32, 1, 1, 1, 0)])
@pytest.mark.parametrize("pinned", [True, False])
def test_arrays_arrive_whole(dtype, nx, ny, nz, pad, pinned):
    torch = pytest.importorskip("torch")
    dt = np.float64 if dtype == gpu.GR_F64 else np.float32
    shape = (nz + 2, ny + 2, nx + 2 + pad)
    U1, U2 = (_array(torch, pinned, shape, dt) for _ in range(2))
    D1, D2 = (_array(torch, pinned, shape, dt, 7) for _ in range(2))
    with gpu.Stepper(1, nx, ny, nz, dtype=dtype, coef=[0.4, 0.1]) as st:
        st.upload(U1, U2)
        gpu.check(gpu.lib().gr_download(st._h, st._ld(D1), gpu._ptr(D1), gpu._ptr(D2)))
        assert (pinned_bytes(st) == 0) == pinned
    for u, d in ((U1, D1), (U2, D2)):
        np.testing.assert_array_equal(d[:, :, :nx + 2], u[:, :, :nx + 2])
        assert (d[:, :, nx + 2:] == 7).all()


def test_slots_are_no_larger_than_the_copies():
    dt = np.float32
    for n, at_most in (((1, 1, 1), 4096), ((30, 30, 30), 1 << 18), ((254, 254, 126), 16 << 20)):
        U = np.random.default_rng(n[0]).random((n[2] + 2, n[1] + 2, n[0] + 2)).astype(dt)
        small = np.zeros((3, 3, 3), dt)
        with gpu.Stepper(1, *n, dtype=gpu.GR_F32, coef=[0.4, 0.1]) as st, \
                gpu.Stepper(1, 1, 1, 1, dtype=gpu.GR_F32, coef=[0.4, 0.1]) as other:
            other.upload(small, small)
            for _ in range(2):
                st.upload(U, U)
                D1, D2 = st.download(U.shape)
                np.testing.assert_array_equal(D1, U)
                np.testing.assert_array_equal(D2, U)
            assert 0 < pinned_bytes(st) <= min(at_most, U.nbytes + 4096)
            assert pinned_bytes(other) <= 4096
