"""Boundary values rewritten through gr_field_ptr between calls: the fused passes read the
halo from whichever buffers they rotate through, so every call must use what the caller
left in U1 and U2.  Fields and halos equal the CPU oracle's bit for bit (tolerance 0)."""
import numpy as np
import pytest

import oracle as orc
from girih_amd import gpu

from test_gpu_parity import _bf16_round, _consts, _pad, _pad_coef, _random_problem

pytestmark = pytest.mark.gpu


class _Memory:
    def __init__(self, ptr, shape, strides, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "strides": strides, "typestr": typestr, "data": (ptr, False),
                                         "version": 2}


def _view(torch, st, which):
    """Field `which` as a tensor [nz + 2R, ny + 2R, nx + 2R] on its own memory."""
    s, size = st.stats(), 8 if st.dtype == gpu.GR_F64 else 4
    at = st.field_ptr(which) + size * s["x_offset"]
    shape = (s["planes_z"], s["rows_y"], st.nx + 2 * st.R)
    return torch.as_tensor(_Memory(at, shape, (s["pitch_x"] * s["rows_y"] * size, s["pitch_x"] * size, size),
                                   "<f%d" % size), device="cuda")


def _new_halo(rng, u, v, R):
    """One set of boundary values for both fields (interiors kept)."""
    h = rng.uniform(-1, 1, u.shape).astype(u.dtype)
    for f in (u, v):
        c = f[R:-R, R:-R, R:-R].copy()
        f[...] = h
        f[R:-R, R:-R, R:-R] = c


@pytest.mark.parametrize("kernel,storage,depth", [(1, "f32", 4), (1, "f64", 3), (5, "f64", 4), (5, "f32", 2),
                                                  (5, "bf16", 6), (5, "f32", 6), (0, "f64", 2), (0, "f32", 2)])
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("n", [(37, 18, 11), (131, 40, 9)])
def test_rewritten_halos_reach_fused_passes(kernel, storage, depth, graph, n):
    torch = pytest.importorskip("torch")
    dt = np.float64 if storage == "f64" else np.float32
    nx, ny, nz = n
    u, v, roc2, coef = _random_problem(kernel, nx, ny, nz, dt, 77)
    if storage == "bf16":
        coef = _bf16_round(coef)
    R, rng = orc.RADIUS[kernel], np.random.default_rng(5)
    with gpu.Stepper(kernel, nx, ny, nz, dtype=gpu.GR_F64 if storage == "f64" else gpu.GR_F32,
                     flags=gpu.GR_COEF_BF16 if storage == "bf16" else 0, coef=_consts(coef, kernel)) as st:
        _new_halo(rng, u, v, R)  # the same halo in both fields, as fused passes need
        st.upload(_pad(u), _pad(v), _pad(roc2) if roc2 is not None else None, _pad_coef(coef, kernel))
        st.set_config(zchunk=5, t_block=depth)
        st.set_graph(graph)
        a = 0
        # one pass (first-order kernels trade a field for the spare), several, a rest of one
        for call, napply in enumerate((depth, 3 * depth, depth, depth, 2 * depth + 1, 2 * depth)):
            print("halo", kernel, storage, depth, graph, napply, flush=True)
            if call > 0:
                _new_halo(rng, u, v, R)
                for which, f in ((0, u), (1, v)):
                    _view(torch, st, which).copy_(torch.tensor(f[:, :, :nx + 2 * R].copy(), device="cuda"))
                torch.cuda.synchronize()
            st.step(napply)
            assert st.stats()["last_launches"] < napply
            for a in range(a, a + napply):
                w, r = (u, v) if a % 2 == 0 else (v, u)
                orc.sweep(kernel, coef, w, r, roc2)
            a += 1
            U1, U2 = st.download(_pad(u).shape)
            np.testing.assert_array_equal(U1[:, :, :nx + 2 * R], u[:, :, :nx + 2 * R])
            np.testing.assert_array_equal(U2[:, :, :nx + 2 * R], v[:, :, :nx + 2 * R])


def test_rewritten_halos_reach_batch_blocks():
    torch = pytest.importorskip("torch")
    sizes = [(40, 20, 12), (33, 18, 16)]
    rng = np.random.default_rng(6)
    coef = np.asarray([-2.8472, 1.6, -0.2, 0.0254, -0.0018])
    with gpu.Batch(sizes, flags=gpu.GR_FAST, coef=list(coef)) as b:
        ref = []
        for i, (nx, ny, nz) in enumerate(sizes):
            u, v, roc2, _ = _random_problem(0, nx, ny, nz, np.float32, 80 + i)
            _new_halo(rng, u, v, 4)
            roc2 *= np.float32(0.1)
            b.problems[i].upload(_pad(u), _pad(v), _pad(roc2), None)
            st = gpu.Stepper(0, nx, ny, nz, dtype=gpu.GR_F32, flags=gpu.GR_FAST, coef=list(coef))
            st.upload(_pad(u), _pad(v), _pad(roc2), None)
            ref.append((st, u, v))
        b.set_time_block(2)
        for n in range(3):
            for i, (st, u, v) in enumerate(ref):
                if n == 0:
                    break
                h = rng.uniform(-1, 1, u.shape).astype(np.float32)
                for s in (st, b.problems[i]):  # single sweeps hold no other copy of the halo
                    for which in (0, 1):
                        t = _view(torch, s, which)
                        c = t[4:-4, 4:-4, 4:-4].clone()
                        t.copy_(torch.tensor(h[:, :, :t.shape[2]].copy(), device="cuda"))
                        t[4:-4, 4:-4, 4:-4] = c
            torch.cuda.synchronize()
            b.step(4)
            assert b.stats()["last_launches"] == 2  # two-step blocks
            for i, (st, u, v) in enumerate(ref):
                st.step(4)
                A, B = b.problems[i].download(_pad(u).shape), st.download(_pad(u).shape)
                for x, y in zip(A, B):
                    np.testing.assert_array_equal(x, y, err_msg="problem %d call %d" % (i, n))
        for st, _, _ in ref:
            st.close()
