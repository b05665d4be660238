"""The launch settings that untuned sweeps choose by kernel and box: both sides of the
rule's line between the 64- and the 128-wide tile (2^21 cells, equal overhang), short
boxes and whole-plane chunks.  Every setting keeps girih's operand order, so the sweep
entry point and an untuned stepper equal the CPU oracle bit for bit (tolerance 0)."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import gpu

from test_gpu_parity import _consts, _pad, _pad_coef, _random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("prec", ["dp", "sp"])
def test_untuned_sweeps_equal_oracle(kernel, prec):
    torch = pytest.importorskip("torch")
    dt, dtype = (np.float64, gpu.GR_F64) if prec == "dp" else (np.float32, gpu.GR_F32)
    R = orc.RADIUS[kernel]
    # the wide tile applies from 128 x 128 x 128 on; one plane less and 129 cells do not take it
    grids = [(5, 3, 2), (67, 33, 9), (128, 128, 127)] + ([(128, 128, 128), (129, 130, 126)] if kernel in (0, 1, 5) else [])
    for n, (nx, ny, nz) in enumerate(grids):
        print("untuned", kernel, prec, (nx, ny, nz), flush=True)
        u, v, roc2, coef = _random_problem(kernel, nx, ny, nz, dt, 60 + n)
        pu, pv, pr = _pad(u), _pad(v), _pad(roc2) if roc2 is not None else None
        pc = _pad_coef(coef, kernel)
        dev = [torch.tensor(a, device="cuda") if a is not None else None for a in (pu, pv, pr, pc)]
        c = np.array(coef[:R + 1], dtype=dt) if pc is None else dev[3].data_ptr()
        nnz, nny, nnx = pu.shape
        gpu.sweep_dev(kernel, dtype, (nnx, nny, nnz), (R, R, R, nx + R, ny + R, nz + R), c, dev[0].data_ptr(),
                      dev[1].data_ptr(), dev[2].data_ptr() if pr is not None else None)
        with gpu.Stepper(kernel, nx, ny, nz, dtype=dtype, coef=_consts(coef, kernel)) as st:
            st.upload(pu, pv, pr, pc)
            st.step(1)
            s = st.stats()
            U1, _ = st.download(pu.shape)
        if kernel in (0, 1, 5):
            assert s["tile_x"] == (128 if (nx, nz) == (128, 128) else 64)
        assert 4 <= s["zchunk"] <= 32
        orc.sweep(kernel, coef, u, v, roc2)
        np.testing.assert_array_equal(dev[0].cpu().numpy()[:, :, :u.shape[2]], u)
        np.testing.assert_array_equal(U1[:, :, :u.shape[2]], u)
