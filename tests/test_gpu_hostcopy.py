"""Uploads and downloads through the pinned slots: fields of many chunks with a ragged
last one, rows padded in the host array, and the padding left as the caller had it."""
import numpy as np
import pytest

from girih_amd import gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,nx,ny,nz,pad", [(gpu.GR_F64, 131, 67, 301, 7), (gpu.GR_F32, 518, 61, 100, 2),
                                                (gpu.GR_F32, 1, 1, 1, 0), (gpu.GR_F64, 30, 5, 3, 0)])
def test_host_fields_round_trip(dtype, nx, ny, nz, pad):
    dt = np.float64 if dtype == gpu.GR_F64 else np.float32
    rng = np.random.default_rng(nx)
    shape = (nz + 2, ny + 2, nx + 2 + pad)
    U1, U2 = rng.random(shape).astype(dt), rng.random(shape).astype(dt)
    with gpu.Stepper(1, nx, ny, nz, dtype=dtype, coef=[0.4, 0.1]) as st:
        st.upload(U1, U2)
        D1, D2 = np.full(shape, 7, dt), np.full(shape, 7, dt)
        gpu.check(gpu.lib().gr_download(st._h, st._ld(D1), gpu._ptr(D1), gpu._ptr(D2)))
        for u, d in ((U1, D1), (U2, D2)):
            np.testing.assert_array_equal(d[:, :, :nx + 2], u[:, :, :nx + 2])
            assert (d[:, :, nx + 2:] == 7).all()
