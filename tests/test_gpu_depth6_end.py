"""Kernel 5 at depth 6 in FP32 and FP64, whose pass ends no call: the last six steps run as
two shallower passes.  Fields equal the CPU oracle's bit for bit (tolerance 0)."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import gpu

from test_gpu_parity import _pad, _pad_coef, _random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "f64"])
def test_last_six_steps(storage):
    dt, dtype = (np.float64, gpu.GR_F64) if storage == "f64" else (np.float32, gpu.GR_F32)
    u, v, _, coef = _random_problem(5, 66, 19, 13, dt, 9)
    with gpu.Stepper(5, 66, 19, 13, dtype=dtype) as st:
        st.upload(_pad(u), _pad(v), None, _pad_coef(coef, 5))
        st.set_config(zchunk=5, t_block=6)
        a = 0
        # 4 + 2; 6 + 4 + 2; 6 + a sweep; 6 + 6 + a sweep; 6 + 2; 6 + 4 + a sweep
        for napply, launches in ((6, 2), (12, 3), (7, 2), (13, 3), (8, 2), (11, 3)):
            print("depth 6", storage, napply, flush=True)
            st.step(napply)
            assert st.stats()["last_launches"] == launches
            for a in range(a, a + napply):
                w, r = (u, v) if a % 2 == 0 else (v, u)
                orc.sweep(5, coef, w, r, None)
            a += 1
            U1, U2 = st.download(_pad(u).shape)
            np.testing.assert_array_equal(U1[:, :, :68], u)
            np.testing.assert_array_equal(U2[:, :, :68], v)
