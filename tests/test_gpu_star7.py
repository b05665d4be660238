"""The fused passes of the 7-point kernels at the edges of their tiles: grids that end
inside a lane's slot of 2 or 4 cells, one cell short of and beyond a tile, whose rows
fill their pitch, and chunks of one plane.  The passes keep girih's operand order, so
every cell equals the CPU oracle's bit for bit (tolerance 0)."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import gpu

from test_gpu_parity import _bf16_round, _consts, _pad, _pad_coef, _random_problem

pytestmark = pytest.mark.gpu

# (kernel, storage, depth, tile variants of that depth)
PASSES = [(1, "f32", 2, 2), (1, "f32", 3, 2), (1, "f32", 4, 5), (1, "f32", 5, 1), (1, "f32", 6, 1), (1, "f64", 2, 2),
          (1, "f64", 3, 1), (1, "f64", 4, 3), (1, "f64", 5, 1), (1, "f64", 6, 1),
          (5, "f64", 2, 1), (5, "f64", 4, 2), (5, "f32", 2, 2), (5, "f32", 4, 3), (5, "bf16", 2, 1), (5, "bf16", 4, 3),
          (5, "bf16", 6, 2), (5, "f32", 6, 1), (5, "f64", 6, 1)]
# nx = 31, 63: the last halo cell is the last word of its row's pitch; 129 and 65 cross a tile by one cell
GRIDS = [(31, 9, 5), (63, 17, 9), (129, 33, 7), (66, 65, 3), (3, 2, 1)]


@pytest.mark.parametrize("kernel,storage,depth,tiles", PASSES)
@pytest.mark.parametrize("zchunk,order", [(0, 0), (1, 2), (4, 1)])
def test_pass_edges_bitexact(kernel, storage, depth, tiles, zchunk, order):
    dt = np.float64 if storage == "f64" else np.float32
    for tile in range(tiles):
        for n, (nx, ny, nz) in enumerate(GRIDS):
            # one pass; two; a rest of one, of two and (where there is such a depth) of three
            calls = (depth, 2 * depth, depth + 1, 2 * depth + 2, depth, 3 * depth + 3)
            print("star7", kernel, storage, depth, tile, (nx, ny, nz), zchunk, calls, flush=True)
            u, v, _, coef = _random_problem(kernel, nx, ny, nz, dt, 300 + n)
            if storage == "bf16":
                coef = _bf16_round(coef)
            src = np.linspace(0.5, -1.0, 4 * depth + 3)  # ends inside a call
            pt = (nx, ny, nz) if n % 2 else (1 + nx // 2, 1, nz)  # the last interior cell, or on an edge
            with gpu.Stepper(kernel, nx, ny, nz, dtype=gpu.GR_F64 if storage == "f64" else gpu.GR_F32,
                             flags=gpu.GR_COEF_BF16 if storage == "bf16" else 0, coef=_consts(coef, kernel)) as st:
                st.upload(_pad(u), _pad(v), None, _pad_coef(coef, kernel))
                if n > 0:
                    st.set_source(*pt, src)
                st.set_streaming(n % 2)  # both cache policies of the kernel-1 passes
                st.set_config(tile, zchunk, depth)
                st.set_xcd_order(order)
                a = 0
                for napply in calls:
                    st.step(napply)
                    assert st.stats()["last_launches"] < napply
                    U1, U2 = st.download(_pad(u).shape)
                    for a in range(a, a + napply):
                        w, r = (u, v) if a % 2 == 0 else (v, u)
                        orc.sweep(kernel, coef, w, r, None)
                        if n > 0 and a < src.size:
                            w[pt[2], pt[1], pt[0]] += dt(src[a])
                    a += 1
                    np.testing.assert_array_equal(U1[:, :, :u.shape[2]], u)
                    np.testing.assert_array_equal(U2[:, :, :u.shape[2]], v)
