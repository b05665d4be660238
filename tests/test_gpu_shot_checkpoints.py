"""Shots whose sweeps write the checkpoints and read them in place: every checkpoint
spacing where states share or miss a checkpoint's fields (1, 2, 3, one before and all
of nt), twice on one shot, against the FP64 CPU shot and adjoint bit for bit (tolerance 0)."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import adjoint, gpu, physics

pytestmark = pytest.mark.gpu

NT, DT_OVER_H = 11, 0.4 / 4725.0


@pytest.mark.parametrize("nx,ny,nz", [(67, 18, 9), (5, 3, 2)])
def test_every_checkpoint_spacing_bitexact(nx, ny, nz):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(nx)
    shp = orc.shape_of(0, nx, ny, nz)
    m = 1.0 / rng.uniform(1500.0, 4500.0, (nz, ny, nx)) ** 2
    roc2 = np.zeros(shp)
    roc2[4:-4, 4:-4, 4:-4] = DT_OVER_H ** 2 / m
    pt, rec_k = (4 + nx // 2, 4 + ny // 2, 4 + nz // 2), 4 + nz // 2
    src = physics.ricker(90.0, 0.4 * 10 / 4725.0, NT - 2, t0=0.003)  # ends before the run does
    res = rng.uniform(-1, 1, (NT, ny, nx))
    tr_cpu, g_cpu = orc.shot(physics.fd8_coef(), roc2, NT, pt, np.append(src, [0.0, 0.0]), rec_k, res=res,
                             dt_over_h=DT_OVER_H)
    mt, rt = torch.tensor(m, device="cuda"), torch.tensor(res, device="cuda")
    for ckpt in (1, 2, 3, 4, NT - 1, NT):
        print("shot planes", (nx, ny, nz), ckpt, flush=True)
        shot = adjoint.Shot(nx, ny, nz, NT, DT_OVER_H, pt, src, rec_k, ckpt=ckpt, dtype=gpu.GR_F64, tune=False)
        for _ in range(2):
            np.testing.assert_array_equal(shot.forward(mt).cpu().numpy(), tr_cpu)
            np.testing.assert_array_equal(shot.vjp(mt, rt).cpu().numpy(), g_cpu)
        shot.close()
