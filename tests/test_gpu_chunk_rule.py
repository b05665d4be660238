"""The tile of a sweep nobody tuned, under a z chunk of the caller's: 128 wide only where that
leaves at least 256 workgroups (kernel 0) or 150; and kernel 4's own chunks.  The sweeps
equal the CPU oracle's bit for bit (tolerance 0)."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import gpu

from test_gpu_parity import _consts, _pad, _pad_coef, _random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1, 5])
def test_tile_under_a_given_chunk(kernel):
    for n, chunk, wide in [((250, 120, 200), 64, False), ((250, 120, 200), 16, kernel != 0), ((512, 512, 256), 64, True),
                           ((512, 512, 256), 0, False), ((256, 256, 256), 64, False), ((64, 64, 64), 8, False),
                           ((129, 300, 128), 4, False), ((1024, 512, 32), 0, True), ((896, 512, 32), 0, kernel != 0)]:
        with gpu.Stepper(kernel, *n, dtype=gpu.GR_F32, coef=None if kernel == 5 else [0.4, 0.1, 0, 0, 0]) as st:
            st.set_config(zchunk=chunk)
            s = st.stats()
            assert (s["tile_x"], s["zchunk"]) == (128 if wide else 64, chunk), (kernel, n, chunk)


def test_kernel4_chunks():
    for n, dtype, chunk in [((512, 512, 256), gpu.GR_F64, 16), ((512, 512, 256), gpu.GR_F32, 4),
                            ((448, 330, 100), gpu.GR_F64, 4), ((500, 400, 3), gpu.GR_F64, 4)]:
        with gpu.Stepper(4, *n, dtype=dtype) as st:
            assert st.stats()["zchunk"] == chunk, (n, dtype)


@pytest.mark.parametrize("kernel", [0, 1, 5])
def test_given_chunks_equal_oracle(kernel):
    for seed, (nx, ny, nz, chunk) in enumerate([(128, 100, 37, 1), (130, 33, 20, 4), (64, 17, 9, 64)]):  # 259 wide tiles in the first
        u, v, roc2, coef = _random_problem(kernel, nx, ny, nz, np.float64, 40 + seed)
        with gpu.Stepper(kernel, nx, ny, nz, coef=_consts(coef, kernel)) as st:
            st.upload(_pad(u), _pad(v), _pad(roc2) if roc2 is not None else None, _pad_coef(coef, kernel))
            st.set_config(zchunk=chunk)
            assert st.stats()["tile_x"] == (128 if seed == 0 else 64)
            st.step(3)
            U1, U2 = st.download(_pad(u).shape)
        orc.run(kernel, coef, u, v, roc2, nt=2)
        orc.sweep(kernel, coef, u, v, roc2)
        np.testing.assert_array_equal(U1[:, :, :u.shape[2]], u)
        np.testing.assert_array_equal(U2[:, :, :u.shape[2]], v)
