"""The work a user has this framework do, as measurable cases.

Five kinds, each through its public entry point:

  step    gpu.Stepper.step(n): n time steps of one resident grid (gr_step)
  sweep   gpu.sweep_dev: single sweeps on the caller's own device arrays (gr_sweep_dev)
  girih   gpu.Stepper.run_ts + download: what girih's driver calls around its host arrays
  batch   gpu.Batch.step(n): uneven wave problems advanced together (gr_batch_step)
  shot    adjoint.shot_traces and its backward pass: one seismic shot and its gradient

Kernels are girih's: 0 the 25-point wave (with FP32: girih's operand order, or "fast"
GR_FAST arithmetic; roc2 "scalar", "field" or "bf16"), 1 the 7-point Jacobi, 5 the 7-point
stencil with seven coefficient arrays ("bf16": stored as bfloat16).  Fields are sums of
smooth standing waves, as a wave or heat simulation holds; coefficients form a convex
average per cell (a heat step with a variable conductivity).
"""
import ctypes
import math

import numpy as np
import torch

from girih_amd import adjoint, gpu, physics

RADIUS = {0: 4, 1: 1, 5: 1}
NCOEF = {0: 0, 1: 0, 5: 7}
JACOBI = [0.4, 0.1]                      # kernel 1: centre and neighbour weight
FD8 = physics.fd8_coef()                 # kernel 0: 8th-order weights
ROC2 = 0.16                              # (v dt / h)^2 of the constant-velocity wave at CFL 0.4
H, VMIN, VMAX = 10.0, 1500.0, 4500.0     # metres, m/s: the layered velocity models
DT = physics.cfl_dt(VMAX * 1.05, H, 0.4)
FLOPS = {0: 40, 1: 10, 5: 13}            # per lattice update


# ------------------------------------------------------------------ what there is to do
def listed():
    return [
        # one application of a caller's own small FP64 grid, twice: launch and call latency
        {"name": "sweep_jacobi7_f64_64", "kind": "sweep", "kernel": 1, "dtype": "f64", "nx": 64, "ny": 64, "nz": 64},
        # the sweep entry point under a caller's own FP32 wave loop, ragged
        {"name": "sweep_wave25_f32_ragged", "kind": "sweep", "kernel": 0, "dtype": "f32", "nx": 403, "ny": 300,
         "nz": 219},
        # the smallest benchmark grid: launch-bound, replayed from a graph
        {"name": "jacobi7_f64_128_graph", "kind": "step", "kernel": 1, "dtype": "f64", "roc2": "", "fast": False,
         "nx": 128, "ny": 128, "nz": 128, "steps": 100, "tune": True, "graph": True},
        # the Jacobi stencil on a grid far larger than the caches
        {"name": "jacobi7_f32_512", "kind": "step", "kernel": 1, "dtype": "f32", "roc2": "", "fast": False,
         "nx": 512, "ny": 512, "nz": 512, "steps": 50, "tune": True, "graph": False},
        # variable coefficients, the benchmark's grid and precisions, and a ragged one
        {"name": "var7_f64_512", "kind": "step", "kernel": 5, "dtype": "f64", "roc2": "", "fast": False,
         "nx": 512, "ny": 512, "nz": 512, "steps": 20, "tune": True, "graph": False},
        {"name": "var7_f32_ragged", "kind": "step", "kernel": 5, "dtype": "f32", "roc2": "", "fast": False,
         "nx": 389, "ny": 270, "nz": 331, "steps": 30, "tune": True, "graph": False},
        {"name": "var7_f32_bf16_512", "kind": "step", "kernel": 5, "dtype": "f32", "roc2": "bf16", "fast": False,
         "nx": 512, "ny": 512, "nz": 512, "steps": 50, "tune": True, "graph": False},
        # the headline: constant-velocity wave with a Ricker source (the largest case)
        {"name": "wave25_f32_1024", "kind": "step", "kernel": 0, "dtype": "f32", "roc2": "scalar", "fast": True,
         "nx": 1024, "ny": 1024, "nz": 1024, "steps": 10, "tune": True, "graph": False},
        # girih's own double-precision wave with a velocity model, ragged
        {"name": "wave25_f64_ragged", "kind": "step", "kernel": 0, "dtype": "f64", "roc2": "field", "fast": False,
         "nx": 500, "ny": 330, "nz": 270, "steps": 20, "tune": True, "graph": False},
        # 16 uneven shots' grids stepped together, bf16 velocity models
        {"name": "batch16_wave25_bf16", "kind": "batch", "roc2": "bf16", "count": 16, "lo": 192, "hi": 512,
         "sizes": 2024, "steps": 10, "graph": True},
        # one shot of an inversion: forward run and gradient
        {"name": "shot_f32_400", "kind": "shot", "dtype": "f32", "nx": 400, "ny": 400, "nz": 400, "steps": 100,
         "ckpt": 50},
        # girih's driver with this stepper: diamond semantics, results back in its host arrays
        {"name": "girih_wave25_f32_256", "kind": "girih", "kernel": 0, "dtype": "f32", "ts": 2, "t_dim": 3,
         "nx": 256, "ny": 256, "nz": 128, "steps": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, lo, hi):
    return {"nx": _log_int(rng, lo, hi), "ny": _log_int(rng, lo, hi), "nz": _log_int(rng, lo, hi)}


def draw(rng):
    kind = rng.choices(["step", "sweep", "girih", "batch", "shot"], [12, 3, 1, 1, 2])[0]
    if kind == "step":
        c = {"kind": kind, "kernel": rng.choice([0, 1, 5]), "dtype": rng.choice(["f32", "f64"]), "roc2": "",
             "fast": False}
        if c["kernel"] == 0:
            c["fast"] = c["dtype"] == "f32" and rng.random() < 0.75
            c["roc2"] = rng.choice(["scalar", "field", "bf16"] if c["dtype"] == "f32" else ["scalar", "field"])
        elif c["kernel"] == 5 and c["dtype"] == "f32" and rng.random() < 0.5:
            c["roc2"] = "bf16"
        c.update(_dims(rng, 48, 640))
        cells = c["nx"] * c["ny"] * c["nz"]
        c["steps"] = _log_int(rng, 4, max(8, min(100, int(4e9 / cells))))
        c["tune"] = rng.random() < 0.75
        c["graph"] = cells < 4e6 and rng.random() < 0.5
        return c
    if kind == "sweep":
        return {"kind": kind, "kernel": rng.choice([0, 1, 5]), "dtype": rng.choice(["f32", "f64"]),
                **_dims(rng, 32, 512)}
    if kind == "girih":
        return {"kind": kind, "kernel": rng.choice([0, 1, 5]), "dtype": rng.choice(["f32", "f64"]), "ts": 0,
                "t_dim": 1, **_dims(rng, 48, 256), "steps": _log_int(rng, 10, 200)}
    if kind == "batch":
        return {"kind": kind, "roc2": rng.choice(["bf16", "field"]), "count": rng.randint(3, 16), "lo": 96, "hi": 320,
                "sizes": rng.randint(1, 9999), "steps": _log_int(rng, 6, 20), "graph": rng.random() < 0.5}
    return {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64"]), **_dims(rng, 64, 224),
            "steps": _log_int(rng, 30, 160), "ckpt": rng.randint(10, 50)}


# ------------------------------------------------------------------ inputs, from the seed alone
def _torch_dtype(c):
    return torch.float64 if c.get("dtype") == "f64" else torch.float32


def _gr_dtype(c):
    return gpu.GR_F64 if c.get("dtype") == "f64" else gpu.GR_F32


def _gen(seed, stream):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + stream) % (1 << 62))


def _smooth(seed, stream, shape, dtype, shift=0.0):
    """A sum of six standing waves over the interior [nz, ny, nx], of amplitude about 1;
    `shift` moves every wave along, as a time step does."""
    rng = np.random.default_rng([int(seed), stream])
    out = torch.zeros(shape, dtype=dtype, device="cuda")
    for _ in range(6):
        amp = rng.uniform(0.3, 1.0)
        axes = []
        for n in shape:
            k = rng.integers(1, max(2, n // 12))
            x = np.cos(np.arange(1, n + 1) * (math.pi * k / (n + 1)) + rng.uniform(0, 2 * math.pi) + shift)
            axes.append(torch.tensor(x, dtype=dtype, device="cuda"))
        out += (amp * axes[0])[:, None, None] * (axes[1][:, None] * axes[2][None, :])
    return out


def _speeds(seed, stream, shape, dtype):
    """A layered velocity model [nz, ny, nx]: 8 layers along z, 5% lateral variation."""
    rng = np.random.default_rng([int(seed), stream, 1])
    cuts = np.sort(rng.integers(0, shape[0], 7))
    layer = np.searchsorted(cuts, np.arange(shape[0]), side="right")
    v = torch.tensor(VMIN + (VMAX - VMIN) * layer / 7.0, dtype=dtype, device="cuda")[:, None, None]
    return v * (1.0 + 0.0125 * _smooth(seed, stream + 100, shape, dtype).clamp(-4, 4))


def _roc2_field(seed, stream, shape, storage, dtype):
    r = ((_speeds(seed, stream, shape, torch.float32) * (DT / H)) ** 2).to(dtype)
    return r.to(torch.bfloat16) if storage == "bf16" else r


def _coefs(seed, shape, storage, dtype):
    """Seven coefficient arrays [7, nz, ny, nx]: neighbours U[0, 0.1), centre one minus their sum."""
    c = torch.empty((7,) + shape, dtype=dtype, device="cuda")
    c.uniform_(0.0, 0.1, generator=_gen(seed, 7))
    c[0] = 1.0 - c[1:].sum(0)
    return c.to(torch.bfloat16) if storage == "bf16" else c


def _inputs(c, seed, stream=0):
    """The interior arrays of one problem, in the types that the problem stores."""
    shape, dtype, storage = (c["nz"], c["ny"], c["nx"]), _torch_dtype(c), c.get("roc2", "field")
    x = {"U1": _smooth(seed, stream, shape, dtype), "U2": _smooth(seed, stream, shape, dtype, 0.05)}
    if c["kernel"] == 0 and storage != "scalar":
        x["roc2"] = _roc2_field(seed, stream, shape, storage, dtype)
    if NCOEF[c["kernel"]]:
        x["coef"] = _coefs(seed, shape, storage, dtype)
    return x


def _source(c, steps):
    """A Ricker wavelet at the grid centre, scaled like a pressure injection."""
    r = RADIUS[0]
    return (r + c["nx"] // 2, r + c["ny"] // 2, r + c["nz"] // 2), ROC2 * physics.ricker(15.0, DT, steps)


# ------------------------------------------------------------------ views of the library's fields
class _DeviceArray:
    """Memory of `owner` for torch.as_tensor: the tensor keeps this object, and so its owner."""

    def __init__(self, owner, ptr, shape, strides, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "strides": strides, "typestr": typestr, "data": (ptr, False),
                                         "version": 2}


def _field(st, which, index=0, bf16=False, owner=None):
    """Field `which` of a Stepper as a tensor [nz + 2R, ny + 2R, nx + 2R] on its own memory,
    which the tensor keeps alive through `owner` (the Stepper, or the Batch it belongs to)."""
    s = st.stats()
    size = 2 if bf16 else (8 if st.dtype == gpu.GR_F64 else 4)
    pitch, rows, planes = s["pitch_x"], s["rows_y"], s["planes_z"]
    at = st.field_ptr(which) + size * (s["x_offset"] + index * pitch * rows * planes)
    shape = (planes, rows, st.nx + 2 * st.R)
    kind = "<i2" if bf16 else "<f%d" % size
    t = torch.as_tensor(_DeviceArray(owner or st, at, shape, (pitch * rows * size, pitch * size, size), kind), device="cuda")
    return t.view(torch.bfloat16) if bf16 else t


def _inner(t, r):
    return t[r:-r, r:-r, r:t.shape[2] - r]


def _fill(st, x, bf16):
    r = st.R
    st.init_fields(2)
    _inner(_field(st, 0), r).copy_(x["U1"])
    _inner(_field(st, 1), r).copy_(x["U2"])
    if "roc2" in x:
        _inner(_field(st, 2, bf16=bf16), r).copy_(x["roc2"])
    for m in range(7 if "coef" in x else 0):
        _inner(_field(st, 3, index=m, bf16=bf16), r).copy_(x["coef"][m])
    torch.cuda.synchronize()


class _Fields:
    """U1 and U2 of a Stepper as tensors (its buffers trade places between calls)."""

    def __init__(self, st, owner=None):
        self.st, self.owner, self.seen = st, owner, {}

    def __call__(self):
        out = []
        for which in (0, 1):
            p = self.st.field_ptr(which)
            if p not in self.seen:
                self.seen[p] = _field(self.st, which, owner=self.owner)
            out.append(self.seen[p])
        return out


# ------------------------------------------------------------------ prepare and run
def _flags(c):
    return ((gpu.GR_FAST if c.get("fast") else 0) | (gpu.GR_ROC2_SCALAR if c["roc2"] == "scalar" else 0) |
            (gpu.GR_COEF_BF16 if c["roc2"] == "bf16" else 0))


def _consts(kernel):
    return FD8 if kernel == 0 else JACOBI if kernel == 1 else None


def _padded(a, r, alignment=8):
    """An interior array in girih's padded host layout (zero halo)."""
    nz, ny, nx = a.shape
    nnx = nx + 2 * r
    out = torch.zeros((nz + 2 * r, ny + 2 * r, nnx + (-nnx) % alignment), dtype=a.dtype, device=a.device)
    out[r:nz + r, r:ny + r, r:nx + r] = a
    return out


def _batch_sizes(c):
    rng = np.random.default_rng(c["sizes"])
    return [tuple(int(x) for x in rng.choice(np.arange(c["lo"], c["hi"] + 1, 16), 3)) for _ in range(c["count"])]


def _batch_problem(c, size):
    return {"kernel": 0, "dtype": "f32", "roc2": c["roc2"], "nx": size[0], "ny": size[1], "nz": size[2]}


def _shot_model(c, seed, stream):
    return (1.0 / _speeds(seed, stream, (c["nz"], c["ny"], c["nx"]), torch.float64) ** 2).to(_torch_dtype(c))


def _shot_geometry(c):
    """Source 50 m below the top, receivers at z = 8 cells."""
    src = (ROC2 * physics.ricker(15.0, DT, c["steps"])).astype(np.float32).astype(np.float64)
    return (4 + c["nx"] // 2, 4 + c["ny"] // 2, 4 + 5), src, 4 + 8


def _start_model(c):
    """The inversion's first guess: a velocity that grows with depth."""
    v = torch.linspace(VMIN, VMAX, c["nz"], dtype=torch.float64, device="cuda")
    return (1.0 / v ** 2)[:, None, None].expand(c["nz"], c["ny"], c["nx"]).to(_torch_dtype(c)).contiguous()


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "step":
        st = gpu.Stepper(c["kernel"], c["nx"], c["ny"], c["nz"], dtype=_gr_dtype(c), flags=_flags(c), roc2=ROC2,
                         coef=_consts(c["kernel"]))
        _fill(st, _inputs(c, seed), c["roc2"] == "bf16")
        if c["roc2"] == "scalar":
            st.set_source(*_source(c, 1000)[0], _source(c, 1000)[1])
        if c["tune"]:
            st.autotune(4)
        if c["graph"]:
            st.set_graph(True)
        return {"kind": kind, "st": st, "steps": c["steps"], "fields": _Fields(st)}
    if kind == "sweep":
        r, x = RADIUS[c["kernel"]], _inputs(c, seed)
        s = {"kind": kind, "kernel": c["kernel"], "dtype": _gr_dtype(c), "U1": _padded(x["U1"], r),
             "U2": _padded(x["U2"], r), "roc2": None}
        np_type = np.float64 if c["dtype"] == "f64" else np.float32
        s["coef"] = np.array(_consts(c["kernel"]), dtype=np_type) if c["kernel"] != 5 else None
        if "roc2" in x:
            s["roc2"] = _padded(x["roc2"], r)
        if "coef" in x:
            s["coefs"] = torch.stack([_padded(a, r) for a in x["coef"]])
            s["coef"] = s["coefs"].data_ptr()
        nnz, nny, nnx = s["U1"].shape
        s["shape"] = (nnx, nny, nnz)
        s["box"] = (r, r, r, c["nx"] + r, c["ny"] + r, c["nz"] + r)
        return s
    if kind == "girih":
        r, x = RADIUS[c["kernel"]], _inputs(c, seed)
        host = {k: _padded(a, r).cpu().numpy() for k, a in x.items() if k != "coef"}
        if "coef" in x:
            host["coef"] = torch.stack([_padded(a, r) for a in x["coef"]]).cpu().numpy()
        st = gpu.Stepper(c["kernel"], c["nx"], c["ny"], c["nz"], dtype=_gr_dtype(c), t_block=0,
                         coef=_consts(c["kernel"]))
        st.upload(host["U1"], host["U2"], host.get("roc2"), host.get("coef"))
        st.autotune(3)
        return {"kind": kind, "st": st, "steps": c["steps"], "ts": c["ts"], "t_dim": c["t_dim"],
                "shape": host["U1"].shape}
    if kind == "batch":
        b = gpu.Batch(_batch_sizes(c), flags=gpu.GR_FAST | (gpu.GR_COEF_BF16 if c["roc2"] == "bf16" else 0), coef=FD8)
        for i, size in enumerate(_batch_sizes(c)):
            p = _batch_problem(c, size)
            _fill(b[i], _inputs(p, seed, stream=10 * i), c["roc2"] == "bf16")
            b[i].set_source(*_source(p, 1000)[0], _source(p, 1000)[1])
        b.autotune(4, use_graph=c["graph"])
        return {"kind": kind, "b": b, "steps": c["steps"], "graph": c["graph"],
                "fields": [_Fields(p, b) for p in b.problems]}
    at, src, rec_k = _shot_geometry(c)
    shot = adjoint.Shot(c["nx"], c["ny"], c["nz"], c["steps"], DT / H, at, src, rec_k, ckpt=c["ckpt"],
                        dtype=_gr_dtype(c), coef=FD8)
    observed = shot.forward(_shot_model(c, seed, 0))
    return {"kind": kind, "shot": shot, "observed": observed, "m": _start_model(c).requires_grad_(True)}


def run(s):
    kind = s["kind"]
    if kind == "step":
        s["st"].step(s["steps"])
        return s["fields"]()
    if kind == "sweep":
        # the loop body of girih's naive stepper: U1 <- f(U2), U2 <- f(U1)
        u1, u2 = s["U1"], s["U2"]
        r = s["roc2"].data_ptr() if s["roc2"] is not None else None
        gpu.sweep_dev(s["kernel"], s["dtype"], s["shape"], s["box"], s["coef"], u1.data_ptr(), u2.data_ptr(), r)
        gpu.sweep_dev(s["kernel"], s["dtype"], s["shape"], s["box"], s["coef"], u2.data_ptr(), u1.data_ptr(), r)
        return [u1, u2]
    if kind == "girih":
        s["st"].run_ts(s["ts"], s["steps"], s["t_dim"])
        return list(s["st"].download(s["shape"]))
    if kind == "batch":
        s["b"].step(s["steps"], use_graph=s["graph"])
        return [f() for f in s["fields"]]
    s["m"].grad = None
    traces = adjoint.shot_traces(s["m"], s["shot"])
    (0.5 * ((traces - s["observed"]) ** 2).sum()).backward()
    return {"traces": traces.detach(), "grad": s["m"].grad}


# ------------------------------------------------------------------ what a pass cannot do without
def _applications(c):
    if c["kind"] == "sweep":
        return 2
    if c["kind"] == "girih":
        if c["ts"] != 2:
            return 2 * ((c["steps"] + 1) // 2)
        w = 2 * (c["t_dim"] + 1)
        return c["steps"] + (-(c["steps"] - 2)) % w - 1
    return c["steps"]


def work(case):
    """Every input array read once and every output array written once, and the arithmetic."""
    c = case
    if c["kind"] == "batch":
        w = {"bytes": 0, "flops": 0}
        for size in _batch_sizes(c):
            p = dict(_batch_problem(c, size), kind="step", fast=True, steps=c["steps"])
            one = work(p)
            w = {k: w[k] + one[k] for k in w}
        return w
    cells, word = c["nx"] * c["ny"] * c["nz"], 8 if c["dtype"] == "f64" else 4
    if c["kind"] == "shot":
        # m and the observed traces in, the traces and the gradient out; the forward run,
        # the adjoint run and one multiply-add per cell and step
        plane = c["nx"] * c["ny"] * c["steps"]
        return {"bytes": word * (2 * cells + 2 * plane), "flops": cells * c["steps"] * (2 * FLOPS[0] + 4)}
    n = _applications(c)
    storage = c.get("roc2", "field")
    arrays = NCOEF[c["kernel"]] + (1 if c["kernel"] == 0 and storage != "scalar" else 0)
    reads = 2 if c["kernel"] == 0 else 1
    return {"bytes": cells * (word * (reads + 2) + arrays * (2 if storage == "bf16" else word)),
            "flops": cells * n * FLOPS[c["kernel"]]}


# ------------------------------------------------------------------ the same in 64 bits, plain torch
def _lap8(p):
    """The 25-point operator of a padded FP64 array, over its interior."""
    n = [x - 8 for x in p.shape]

    def at(dz, dy, dx):
        return p[4 + dz:4 + dz + n[0], 4 + dy:4 + dy + n[1], 4 + dx:4 + dx + n[2]]

    out = FD8[0] * at(0, 0, 0)
    for r in range(1, 5):
        s = at(0, 0, r) + at(0, 0, -r)
        for d in ((0, r, 0), (0, -r, 0), (r, 0, 0), (-r, 0, 0)):
            s += at(*d)
        out.add_(s, alpha=FD8[r])
    return out


def _pad64(a, r):
    nz, ny, nx = a.shape
    out = torch.zeros((nz + 2 * r, ny + 2 * r, nx + 2 * r), dtype=torch.float64, device=a.device)
    out[r:-r, r:-r, r:-r] = a
    return out


def _steps64(c, x, n):
    """(U1, U2) padded in FP64 after n applications of the kernel to the inputs x."""
    r = RADIUS[c["kernel"]]
    u = [_pad64(x["U1"], r), _pad64(x["U2"], r)]
    src = None
    if c["kernel"] == 0 and (c.get("roc2") == "scalar" or c["kind"] == "batch"):
        src = _source(c, 1000)
    roc2 = x["roc2"].double() if "roc2" in x else ROC2
    coef = x["coef"].double() if "coef" in x else None
    for a in range(n):
        w, v = u[a % 2], u[1 - a % 2]
        wi, vi = _inner(w, r), _inner(v, r)
        if c["kernel"] == 0:
            lap = _lap8(v)
            lap *= roc2
            wi.neg_().add_(vi, alpha=2.0).add_(lap)
            if src is not None:
                i, j, k = src[0]
                w[k, j, i] += float(src[1][a])
        else:
            nb = [v[1:-1, 1:-1, :-2], v[1:-1, 1:-1, 2:], v[1:-1, :-2, 1:-1], v[1:-1, 2:, 1:-1], v[:-2, 1:-1, 1:-1],
                  v[2:, 1:-1, 1:-1]]
            if c["kernel"] == 1:
                out = JACOBI[0] * vi
                for b in nb:
                    out.add_(b, alpha=JACOBI[1])
            else:
                out = coef[0] * vi
                for m, b in enumerate(nb):
                    out.addcmul_(coef[m + 1], b)
            wi.copy_(out)
    return u


def _shot64(c, seed):
    """Traces and gradient of a shot in FP64: every state kept, then the reversed recurrence."""
    at, src, rec_k = _shot_geometry(c)
    k2, nt = (DT / H) ** 2, c["steps"]
    shape = (c["nz"], c["ny"], c["nx"])

    def forward(m, keep):
        roc2 = k2 / m
        prev, cur = _pad64(torch.zeros(shape, device="cuda"), 4), _pad64(torch.zeros(shape, device="cuda"), 4)
        traces = torch.empty((nt,) + shape[1:], dtype=torch.float64, device="cuda")
        states = []
        for a in range(nt):
            if keep:
                states.append(_inner(cur, 4).clone())
            lap = _lap8(cur)
            lap *= roc2
            _inner(prev, 4).neg_().add_(_inner(cur, 4), alpha=2.0).add_(lap)
            prev[at[2], at[1], at[0]] += float(src[a])
            prev, cur = cur, prev
            traces[a] = _inner(cur, 4)[rec_k - 4]
        return traces, states

    observed, _ = forward(_shot_model(c, seed, 0).double(), False)
    m = _start_model(c).double()
    roc2 = k2 / m
    traces, states = forward(m, True)
    res = traces - observed
    grad = torch.zeros(shape, dtype=torch.float64, device="cuda")
    # cotangents of x_{a+2} (l2) and x_{a+1} (l1)
    l2, l1 = torch.zeros(shape, dtype=torch.float64, device="cuda"), torch.zeros(shape, dtype=torch.float64, device="cuda")
    for a in range(nt - 1, -1, -1):
        l2[rec_k - 4] += res[a]
        grad.addcmul_(l2, _lap8(_pad64(states.pop(), 4)))
        below = -l2
        l1 = l1 + 2.0 * l2 + _lap8(_pad64(roc2 * l2, 4))
        l2, l1 = l1, below
    return {"traces": traces, "grad": grad * (-k2 / m ** 2)}


def exact(case, seed):
    c = case
    if c["kind"] == "shot":
        return _shot64(c, seed)
    if c["kind"] == "batch":
        return [_steps64(dict(_batch_problem(c, size), kind="batch"), _inputs(_batch_problem(c, size), seed, stream=10 * i),
                         c["steps"]) for i, size in enumerate(_batch_sizes(c))]
    u = _steps64(c, _inputs(c, seed), _applications(c))
    if c["kind"] == "step":
        return u
    r = RADIUS[c["kernel"]]
    u = [_padded(_inner(a, r), r) for a in u]
    return u if c["kind"] == "sweep" else [a.cpu().numpy() for a in u]
