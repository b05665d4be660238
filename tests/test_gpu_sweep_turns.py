"""Successive streaming sweeps take the planes up and down z in turn.  Kernels 0 to 4 add the planes
below and above in pairs, so either way every cell equals the CPU oracle's bit for bit
(tolerance 0): every tile variant, chunks that divide z unevenly, one plane, sources on the
first and the last plane, one step per call and several.  The FAST arithmetic has no
oracle; a problem turned upside down must give the turned fields, bit for bit."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import gpu

from test_gpu_parity import _bf16_round, _consts, _pad, _pad_coef, _random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_either_way_equals_oracle(kernel, storage):
    dt = np.float64 if storage == "f64" else np.float32
    if storage == "bf16" and kernel == 1:
        pytest.skip("kernel 1 stores no coefficient field")
    for n, (nx, ny, nz) in enumerate([(70, 19, 21), (9, 34, 1), (131, 5, 6)]):
        u0, v0, roc2, coef = _random_problem(kernel, nx, ny, nz, dt, 900 + n)
        if storage == "bf16":
            roc2 = _bf16_round(roc2) if roc2 is not None else None
            coef = _bf16_round(coef) if kernel in (2, 3, 4) else coef
        R = orc.RADIUS[kernel]
        src = np.linspace(0.5, -1.0, 4)  # ends before the last step
        pt = (R + nx // 2, R, R + (nz - 1 if n % 2 == 0 else 0))
        for variant in range({0: 17, 1: 16}.get(kernel, 1)):
            zchunk, calls = ((0, (2, 3)), (4, (1, 1, 3)), (8, (5,)))[(variant + n) % 3]
            print("turns", kernel, storage, (nx, ny, nz), variant, zchunk, calls, flush=True)
            u, v = u0.copy(), v0.copy()
            with gpu.Stepper(kernel, nx, ny, nz, dtype=gpu.GR_F64 if storage == "f64" else gpu.GR_F32,
                             flags=gpu.GR_COEF_BF16 if storage == "bf16" else 0, coef=_consts(coef, kernel)) as st:
                st.upload(_pad(u), _pad(v), _pad(roc2) if roc2 is not None else None, _pad_coef(coef, kernel))
                st.set_source(*pt, src)
                st.set_streaming((variant + n) % 2 if kernel < 2 else 1)  # streaming sweeps take turns
                st.set_config(variant, zchunk, 1)
                st.set_xcd_order(variant % 3)
                for c in calls:
                    st.step(c)
                U1, U2 = st.download(_pad(u).shape)
            for a in range(5):
                w, r = (u, v) if a % 2 == 0 else (v, u)
                orc.sweep(kernel, coef, w, r, roc2)
                if a < src.size:
                    w[pt[2], pt[1], pt[0]] += dt(src[a])
            np.testing.assert_array_equal(U1[:, :, :u.shape[2]], u)
            np.testing.assert_array_equal(U2[:, :, :u.shape[2]], v)


@pytest.mark.parametrize("roc", ["scalar", "field", "bf16"])
def test_fast_turned_problem(roc):
    nx, ny, nz = 77, 21, 23
    u, v, roc2, coef = _random_problem(0, nx, ny, nz, np.float32, 31)
    roc2 = _bf16_round(roc2)
    src, out = np.linspace(0.5, -1.0, 4), []
    flags = gpu.GR_FAST | {"scalar": gpu.GR_ROC2_SCALAR, "field": 0, "bf16": gpu.GR_COEF_BF16}[roc]
    for turned in (False, True):
        t = (lambda a: np.ascontiguousarray(a[::-1])) if turned else (lambda a: a)
        with gpu.Stepper(0, nx, ny, nz, dtype=gpu.GR_F32, flags=flags, roc2=0.04, coef=_consts(coef, 0)) as st:
            st.upload(_pad(t(u)), _pad(t(v)), None if roc == "scalar" else _pad(t(roc2)), None)
            k = 4 + 2
            st.set_source(40, 9, nz + 7 - k if turned else k, src)
            st.set_streaming(1)
            st.set_config(0, 8, 1)
            st.step(5)
            out.append([t(a) for a in st.download(_pad(u).shape)])
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
