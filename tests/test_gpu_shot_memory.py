"""What a shot's first backward pass allocates: K states and K + 2 adjoint fields for
checkpoints every K applications, and the dense accumulator."""
import ctypes

import pytest

from girih_amd import adjoint, gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,ckpt", [(12, 4), (3, 1), (5, 5)])
def test_backward_buffers(nt, ckpt):
    torch = pytest.importorskip("torch")
    n, held = 160, []
    m = torch.full((n, n, n), 1.0 / 2000.0 ** 2, device="cuda")
    res, grad = torch.ones((nt, n, n), device="cuda"), torch.empty((n, n, n), device="cuda")
    for _ in range(2):  # the first shot loads the kernels
        shot = adjoint.Shot(n, n, n, nt, 0.4 / 4725.0, (84, 84, 84), [1.0], 84, ckpt=ckpt, tune=False)
        shot.forward(m)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        gpu.check(gpu.lib().gr_shot_adjoint(shot._s, ctypes.c_void_p(res.data_ptr()), ctypes.c_void_p(grad.data_ptr())))
        held.append(before - torch.cuda.mem_get_info()[0])
        s = shot.stepper.stats()
        field = 4 * s["pitch_x"] * s["rows_y"] * s["planes_z"]
        shot.close()
    want = (2 * ckpt + 2) * field + 4 * n ** 3
    print("backward buffers", nt, ckpt, held, want, flush=True)
    assert want <= held[1] <= want + field  # a field is 22 MB; allocations are rounded up to 2 MB
