"""What the performance of this framework is measured on.

Four kinds of work, each through the package's public entry points:

  step   solver.Stepper: the fused solver loop.  A pass advances the system by a
         fixed number of accepted steps (`steps`, Stepper.run) or by a fixed time
         (`until_ps`, Stepper.run_until, the reference's solve(Time(t))) and reads
         the magnetisation back, as a script does between two snapshots.
  batch  solver.Ensemble: independent systems of uneven sizes stepped together
         (parameter studies), then every member's magnetisation.
  conv   magneto.SymmetricMatrixVectorConvolution_FFT.execute: the stray field
         alone, in the drop-in form, on device arrays.
  rhs    the drop-in form of one LLG evaluation in FP64: stray field, exchange,
         uniaxial anisotropy, right-hand side and the Runge-Kutta stage algebra, one
         magneto call each, as the reference's front end issues them.

FP32 magnetisation is read back and kept as float32 (what the state holds).  FP64
steppers use the FP64 norm (normalize_mode=1).  Seeds make the initial states; meshes
and materials belong to the case.
"""
import functools
import math

import numpy as np
import torch

from micromagnum_amd import magneto as mg
from micromagnum_amd.device import empty, to_device
from micromagnum_amd.solver import Ensemble, Stepper

MU0 = 4.0e-7 * math.pi
GAMMA = 2.211e5

# Materials and fields by name; all but "disk" are those of bench.py's workloads.
PHYSICS = {
    # permalloy film: stray field and exchange
    "plain": dict(Ms=8e5, alpha=0.5, A=1.3e-11),
    # perpendicular block: uniaxial anisotropy and a uniform field of 20 mT
    "uniaxial": dict(Ms=1.1e6, alpha=0.02, A=1.5e-11, k_uni=5e5, axis1=(0.0, 0.0, 1.0), h_ext=(0.02 / MU0, 0.0, 0.0)),
    # current through a film (Zhang-Li torque)
    "torque": dict(Ms=8.6e5, alpha=0.1, A=1.3e-11, P=0.7, xi=0.05, j=(1e12, 0.0, 0.0)),
    # relaxation with cubic anisotropy
    "cubic": dict(Ms=8e5, alpha=1.0, A=1.3e-11, k_cub=-5e3, axis1=(1.0, 0.0, 0.0), axis2=(0.0, 1.0, 0.0)),
    # a round body: Ms and A per cell, zero outside the inscribed ellipse
    "disk": dict(Ms=8e5, alpha=0.1, A=1.3e-11),
}


def _step(name, shape, delta, method, precision, physics, state, steps=0, until_ps=0.0, tol=1e-4):
    return dict(name=name, kind="step", nx=shape[0], ny=shape[1], nz=shape[2], dx=delta[0], dy=delta[1], dz=delta[2],
                method=method, precision=precision, physics=physics, state=state, steps=steps, until_ps=until_ps,
                tol=tol)


def _field(name, kind, shape, precision):
    return dict(name=name, kind=kind, nx=shape[0], ny=shape[1], nz=shape[2], dx=2e-9, dy=2e-9, dz=2e-9,
                precision=precision)


def listed():
    return [
        # the smallest mesh in use: fixed-step RK4, <M> and M every ten steps; launches and latency
        _step("film_128x32x1_rk4_fp64", (128, 32, 1), (4e-9, 4e-9, 3e-9), "rk4", "fp64", "plain", "random", steps=10),
        # a standard-problem strip (500 nm x 125 nm x 3 nm) at 2 nm: odd sizes, 500-point lines
        _step("strip_250x63x1_rkf45_fp64", (250, 63, 1), (2e-9, 2e-9, 3e-9), "rkf45", "fp64", "plain", "vortex",
              steps=40),
        # a vortex disk in a box that is mostly used, per-cell material
        _step("disk_200x200x5_rkf45_fp64", (200, 200, 5), (3e-9, 3e-9, 4e-9), "rkf45", "fp64", "disk", "vortex",
              steps=40),
        # a ragged block in mixed precision
        _step("block_150x90x14_rkf45_fp32", (150, 90, 14), (2e-9, 2e-9, 2e-9), "rkf45", "fp32", "uniaxial", "random",
              until_ps=1.0),
        # the headline block in both precisions
        _step("block_256x256x16_rkf45_fp32", (256, 256, 16), (2e-9, 2e-9, 2e-9), "rkf45", "fp32", "uniaxial",
              "vortex", until_ps=2.0),
        _step("block_256x256x16_rkf45_fp64", (256, 256, 16), (2e-9, 2e-9, 2e-9), "rkf45", "fp64", "uniaxial",
              "random", steps=40),
        # vortex film under a current, Dormand-Prince
        _step("film_1024x1024x2_dp54_fp32", (1024, 1024, 2), (3e-9, 3e-9, 2e-9), "dp54", "fp32", "torque", "vortex",
              until_ps=1.0, tol=1e-5),
        # the largest mesh: relaxation of a thick grid
        _step("grid_512x512x32_rkf45_fp32", (512, 512, 32), (2e-9, 2e-9, 2e-9), "rkf45", "fp32", "cubic", "random",
              until_ps=1.0),
        # a parameter study: 48 systems, 32..256 cells in the plane, 1..4 layers
        dict(name="ensemble_48_rkf45_fp32", kind="batch", count=48, draw=7, precision="fp32", steps=20),
        # the stray field alone: the block's mesh in FP64, and a ragged small one in FP32
        _field("conv_256x256x16_fp64", "conv", (256, 256, 16), "fp64"),
        _field("conv_99x85x7_fp32", "conv", (99, 85, 7), "fp32"),
        # one evaluation of the drop-in route
        _field("rhs_192x120x10_fp64", "rhs", (192, 120, 10), "fp64"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["conv"] * 2 + ["rhs", "batch"])
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(6, 32), draw=rng.randint(100, 10 ** 6),
                    precision=rng.choice(["fp32", "fp32", "fp64"]), steps=rng.randint(5, 15))
    while True:
        nx, ny = _log_int(rng, 24, 640), _log_int(rng, 16, 640)
        nz = rng.choice([1, 1, 2, 3]) if rng.random() < 0.5 else _log_int(rng, 4, 32)
        if 4000 <= nx * ny * nz <= 1500000:
            break
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, dx=rng.choice([2e-9, 3e-9, 4e-9]), dy=2e-9, dz=rng.choice([2e-9, 3e-9]),
             precision=rng.choice(["fp32", "fp64"]) if kind != "rhs" else "fp64")
    if kind == "step":
        c["physics"] = rng.choice(sorted(PHYSICS))
        c["method"] = rng.choice(["rkf45", "rkf45", "dp54", "rk4"])
        # dp54 carries the last stage of a rejected step over, as the reference does,
        # which from random directions magnifies the last bit
        c["state"] = rng.choice(["random", "vortex"]) if c["method"] != "dp54" else "vortex"
        fixed = c["method"] == "rk4" or c["precision"] == "fp64"
        c["steps"] = rng.randint(8, 15 if c["method"] == "dp54" else 30) if fixed else 0
        c["until_ps"] = 0.0 if fixed else round(rng.uniform(0.3, 0.8) * (1 if c["state"] == "random" else 2), 3)
        c["tol"] = 1e-5 if c["method"] == "dp54" else 1e-4
    return c


# ------------------------------------------------------------------ inputs
def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _delta(case):
    return case["dx"], case["dy"], case["dz"]


@functools.lru_cache(maxsize=64)
def _tensor(shape, delta):
    """The demag tensor of a mesh, which a program computes (or loads) once."""
    gpu = shape[0] * shape[1] * shape[2] >= 1 << 18
    return mg.GenerateDemagTensor(*shape, *delta, device="gpu" if gpu else None)


def _inside(shape):
    """1 in the ellipse inscribed in the mesh's plane, 0 outside."""
    nx, ny, nz = shape
    x, y = (np.arange(nx) + 0.5) / nx * 2 - 1, (np.arange(ny) + 0.5) / ny * 2 - 1
    return np.broadcast_to(x[None, :] ** 2 + y[:, None] ** 2 < 1.0, (nz, ny, nx)).astype(np.float64)


def _state(shape, Ms, kind, seed):
    """Directions from the seed ("random"), or a vortex around a seeded centre
    with 1 % noise; |M| = Ms, zero where Ms is."""
    nx, ny, nz = shape
    rng = np.random.Generator(np.random.PCG64(seed))
    m = rng.standard_normal((3, nz, ny, nx))
    if kind == "vortex":
        cx, cy = (0.5 + 0.1 * rng.uniform(-1, 1, 2)) * (nx, ny)
        X, Y = (np.arange(nx) + 0.5 - cx)[None, None, :], (np.arange(ny) + 0.5 - cy)[None, :, None]
        r2 = X * X + Y * Y
        v = np.stack(np.broadcast_arrays(-Y + 0 * X, X + 0 * Y, 3.0 + 5.0 * np.exp(-r2 / 25.0)))
        m = v / np.sqrt((v ** 2).sum(axis=0)) + 0.01 * m
    m *= Ms / np.sqrt((m ** 2).sum(axis=0))
    return m


def _material(case):
    kw = dict(PHYSICS[case["physics"]])
    if case["physics"] == "disk":
        inside = _inside(_shape(case))
        kw.update(Ms=kw["Ms"] * inside, A=kw["A"] * inside)
    return kw


def _members(case):
    """The systems of an ensemble, as bench.py's 512-system draw makes them."""
    rng = np.random.Generator(np.random.PCG64(case["draw"]))
    out = []
    for _ in range(case["count"]):
        shape = (int(rng.integers(32, 257)), int(rng.integers(32, 257)), int(rng.integers(1, 5)))
        axis = rng.standard_normal(3)
        out.append(dict(shape=shape, delta=tuple(float(v) for v in rng.uniform(2e-9, 5e-9, 3)),
                        Ms=float(rng.uniform(4e5, 1.4e6)), alpha=0.5, A=float(rng.uniform(5e-12, 2e-11)),
                        k_uni=float(rng.uniform(0.0, 1e6)), axis1=tuple(float(v) for v in axis / np.linalg.norm(axis))))
    return out


class _View:
    """A device array as torch sees it: the same memory, nothing copied."""

    def __init__(self, d):
        self.keep = d
        self.__cuda_array_interface__ = dict(shape=d.shape, typestr=d.dtype.str, data=(d.ptr.value, False), version=2)


def _rhs_inputs(case, seed):
    """The arrays of an LLG evaluation and of the stage that follows it."""
    shape, p = _shape(case), PHYSICS["uniaxial"]
    sc, vec = shape[::-1], (3,) + shape[::-1]
    gp = GAMMA / (1.0 + p["alpha"] ** 2)
    M = _state(shape, p["Ms"], "vortex", seed)
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    return dict(M=M, Ms=np.full(sc, p["Ms"]), A=np.full(sc, p["A"]), k=np.full(sc, p["k_uni"]),
                axis=np.broadcast_to(np.array(p["axis1"]).reshape(3, 1, 1, 1), vec).copy(), f1=np.full(sc, -gp),
                f2=np.full(sc, -p["alpha"] * gp / p["Ms"]), k0=1e16 * rng.standard_normal(vec))


def prepare(case, seed):
    seed = int(seed)
    if case["kind"] == "batch":
        specs = _members(case)
        tol = dict(method="rkf45", eps_abs=1e-4, eps_rel=1e-4, precision=case["precision"],
                   normalize_mode=int(case["precision"] == "fp64"))
        ens = Ensemble([dict(s, N=_tensor(s["shape"], s["delta"]), **tol) for s in specs])
        for i, s in enumerate(specs):
            ens.set_m(i, _state(s["shape"], s["Ms"], "random", seed * 1000 + i))
        return dict(case=case, ens=ens)
    shape, delta = _shape(case), _delta(case)
    N = _tensor(shape, delta)
    if case["kind"] == "step":
        kw = _material(case)
        st = Stepper(shape, delta, N=N, precision=case["precision"], method=case["method"], eps_abs=case["tol"],
                     eps_rel=case["tol"], h0=1e-13, normalize_mode=int(case["precision"] == "fp64"), **kw)
        st.set_m(_state(shape, kw["Ms"], case["state"], seed))
        return dict(case=case, st=st, t=0.0)
    dt = np.float64 if case["precision"] == "fp64" else np.float32
    conv = mg.SymmetricMatrixVectorConvolution_FFT(N, *shape, precision=case["precision"])
    if case["kind"] == "conv":
        M, H = to_device(_state(shape, 8e5, "random", seed), dt), empty((3,) + shape[::-1], dt)
        return dict(case=case, conv=conv, M=M, H=H, out=torch.as_tensor(_View(H), device="cuda"))
    d = {k: to_device(v) for k, v in _rhs_inputs(case, seed).items()}
    new = {k: empty(d["M"].shape) for k in ("Hd", "He", "Ha", "dM", "y")}
    return dict(case=case, conv=conv, tab=mg.ButcherTableau("rkf45"), d=d, new=new,
                out={k: torch.as_tensor(_View(v), device="cuda") for k, v in new.items()})


def run(s):
    case = s["case"]
    f32 = case["precision"] == "fp32"
    if case["kind"] == "step":
        st = s["st"]
        if case["until_ps"]:
            s["t"] += case["until_ps"] * 1e-12
            st.run_until(s["t"])
        else:
            st.run(case["steps"])
        M = st.get_m()
        return M.astype(np.float32) if f32 else M
    if case["kind"] == "batch":
        ens = s["ens"]
        ens.run(case["steps"])
        Ms = [ens.get_m(i) for i in range(len(ens))]
        return [M.astype(np.float32) for M in Ms] if f32 else Ms
    if case["kind"] == "conv":
        s["conv"].execute(s["M"], s["H"])
        return s["out"]
    nx, ny, nz = _shape(case)
    d, new = s["d"], s["new"]
    s["conv"].execute(d["M"], new["Hd"])
    e_exch = mg.exchange(nx, ny, nz, *_delta(case), 0, 0, 0, d["Ms"], d["A"], d["M"], new["He"])
    e_aniso = mg.uniaxial_anisotropy(d["axis"], d["k"], d["Ms"], d["M"], new["Ha"])
    mg.llge(d["f1"], d["f2"], d["M"], new["He"], new["dM"])
    mg.rk_prepare_step(2, 1e-13, s["tab"], [d["k0"], new["dM"]], d["M"], new["y"])
    return dict(s["out"], e_exch=e_exch, e_aniso=e_aniso)


# ------------------------------------------------------------------ what a pass needs
def _round4(n):
    return 1 if n == 1 else (2 * n - 1 + 3) // 4 * 4


def _field_work(shape, b):
    """One field evaluation: M read, the tensor's octant read, the result
    written; forward and inverse real transforms of three components."""
    n = shape[0] * shape[1] * shape[2]
    P = [_round4(v) for v in shape]
    pts = P[0] * P[1] * P[2]
    return 12.0 * b * n, 3 * 2 * 2.5 * pts * math.log2(max(2, pts)) + 15.0 * pts + 100.0 * n


def work(case):
    b = 8 if case["precision"] == "fp64" else 4
    if case["kind"] == "batch":
        got = [_field_work(s["shape"], b) for s in _members(case)]
        k = 6 * case["steps"]
        return dict(bytes=k * sum(g[0] for g in got), flops=k * sum(g[1] for g in got))
    nbytes, flops = _field_work(_shape(case), b)
    if case["kind"] == "conv":
        return dict(bytes=nbytes, flops=flops)
    if case["kind"] == "rhs":
        n = case["nx"] * case["ny"] * case["nz"]
        # M, k0 and the tensor in, Ms, A, k, axis, f1, f2 in, five vector fields out
        return dict(bytes=8.0 * n * (6 + 6 + 8 + 15), flops=flops + 100.0 * n)
    stages = {"rk4": 4, "rkf45": 6, "dp54": 6}[case["method"]]
    # a step of these systems takes about 0.1 ps under step control
    steps = case["steps"] or case["until_ps"] / 0.1
    return dict(bytes=steps * stages * nbytes, flops=steps * stages * flops)


# ------------------------------------------------------------------ 64-bit values
_RKF45_B = [[], [1 / 4], [3 / 32, 9 / 32], [1932 / 2197, -7200 / 2197, 7296 / 2197], [439 / 216, -8, 3680 / 513, -845 / 4104],
            [-8 / 27, 2, -3544 / 2565, 1859 / 4104, -11 / 40]]
_RKF45_C4 = [25 / 216, 0, 1408 / 2565, 2197 / 4104, -1 / 5, 0]
_RKF45_C5 = [16 / 135, 0, 6656 / 12825, 28561 / 56430, -9 / 50, 2 / 55]


class _Exact:
    """The field terms in float64 with torch's FFT."""

    def __init__(self, shape, delta, kw):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.shape, self.delta = shape, delta
        put = lambda a, d: torch.as_tensor(np.array(np.broadcast_to(np.asarray(a, dtype=np.float64), d)), device=self.dev)  # noqa: E731
        sc = shape[::-1]
        self.Ms, self.A = put(kw["Ms"], sc), put(kw["A"], sc)
        self.alpha, self.kw = kw["alpha"], kw
        N = torch.as_tensor(_tensor(shape, delta), device=self.dev)
        self.P = tuple(N.shape[:3])
        self.K = [torch.fft.rfftn(N[..., e].contiguous()) for e in range(6)]

    def demag(self, M):
        F = [torch.fft.rfftn(M[c], s=self.P) for c in range(3)]
        K, (nx, ny, nz) = self.K, self.shape
        rows = [(0, 1, 2), (1, 3, 4), (2, 4, 5)]
        return torch.stack([torch.fft.irfftn(sum(K[e] * F[c] for c, e in enumerate(r)), s=self.P)[:nz, :ny, :nx]
                            for r in rows])

    def exchange(self, M):
        """2 A / (mu0 Ms) times the Laplacian of m over the neighbours that have material."""
        on = (self.Ms != 0).double()
        ms = torch.where(self.Ms != 0, self.Ms, torch.ones_like(self.Ms))
        m, s = M / ms * on, torch.zeros_like(M)
        for axis, d in ((3, self.delta[0]), (2, self.delta[1]), (1, self.delta[2])):
            n = M.shape[axis]
            if n == 1:
                continue
            up, dn = m.narrow(axis, 1, n - 1), m.narrow(axis, 0, n - 1)
            both = on.unsqueeze(0).narrow(axis, 1, n - 1) * on.unsqueeze(0).narrow(axis, 0, n - 1)
            g = (up - dn) * both / d ** 2
            s.narrow(axis, 0, n - 1).add_(g)
            s.narrow(axis, 1, n - 1).sub_(g)
        return 2.0 / MU0 * self.A / ms * on * s

    def _vec(self, v):
        return torch.tensor(v, dtype=torch.float64, device=self.dev).reshape(3, 1, 1, 1)

    def uniaxial(self, M):
        a = self._vec(self.kw["axis1"])
        return 2.0 * self.kw["k_uni"] / (MU0 * self.Ms ** 2) * (M * a).sum(0) * a

    def cubic(self, M):
        u = [self._vec(self.kw["axis1"]), self._vec(self.kw["axis2"])]
        u.append(torch.linalg.cross(u[0], u[1], dim=0))
        c = [(M * v).sum(0) / M.square().sum(0).sqrt() for v in u]
        s = [v * v for v in c]
        f = -2.0 / MU0 * self.kw["k_cub"] / self.Ms
        return f * ((s[1] + s[2]) * c[0] * u[0] + (s[0] + s[2]) * c[1] * u[1] + (s[0] + s[1]) * c[2] * u[2])

    def torque(self, M):
        """Zhang-Li: central differences inside, one-sided at the faces."""
        P, xi, al, ms, j = self.kw["P"], self.kw["xi"], self.alpha, self.Ms, self.kw["j"]
        bj = P * 9.2740154e-24 / (1.602176487e-19 * ms * (1 + xi * xi)) / (1 + al * al)
        g = torch.zeros_like(M)
        for c, (axis, d) in enumerate(((3, self.delta[0]), (2, self.delta[1]), (1, self.delta[2]))):
            if M.shape[axis] > 1 and j[c]:
                g += j[c] * torch.gradient(M, spacing=d, dim=axis, edge_order=1)[0]
        B = torch.linalg.cross(M, g, dim=0)
        return -bj / ms ** 2 * (1 + al * xi) * torch.linalg.cross(M, B, dim=0) - bj / ms * (xi - al) * B

    def dmdt(self, M):
        H = self.demag(M) + self.exchange(M)
        if "k_uni" in self.kw:
            H = H + self.uniaxial(M)
        if "k_cub" in self.kw:
            H = H + self.cubic(M)
        if "h_ext" in self.kw:
            H = H + self._vec(self.kw["h_ext"])
        gp = GAMMA / (1 + self.alpha ** 2)
        on = self.Ms != 0
        f2 = torch.where(on, -self.alpha * gp / torch.where(on, self.Ms, torch.ones_like(self.Ms)), torch.zeros_like(self.Ms))
        X = torch.linalg.cross(M, H, dim=0)
        k = -gp * on * X + f2 * torch.linalg.cross(M, X, dim=0)
        return k + self.torque(M) if "P" in self.kw else k

    def norm(self, M):
        n = M.square().sum(0).sqrt()
        return torch.where(n > 0, M * (self.Ms / torch.where(n > 0, n, torch.ones_like(n))), M)

    def scaled_max(self, v):
        on = self.Ms != 0
        return float((v.square().sum(0).sqrt()[on] / self.Ms[on]).max())


def _exact_rk4(x, M, h, steps):
    for _ in range(steps):
        k1 = x.dmdt(M)
        k2 = x.dmdt(M + h / 2 * k1)
        k3 = x.dmdt(M + h / 2 * k2)
        k4 = x.dmdt(M + h * k3)
        M = x.norm(M + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4))
    return M


def _exact_rkf45(x, M, h, tol, steps, t_end):
    """RKF45 with the step control of the reference (headroom 0.85, factors in
    [0.2, 5], steps in [1e-15, 1e-10]); a step that would pass t_end is taken again
    up to it."""
    t, done = 0.0, 0
    while t < t_end if t_end else done < steps:
        k = []
        for row in _RKF45_B:
            k.append(x.dmdt(M + h * sum(b * v for b, v in zip(row, k)) if row else M))
        e_abs = x.scaled_max(h * sum((a - b) * v for a, b, v in zip(_RKF45_C4, _RKF45_C5, k)))
        e_rel = e_abs / (h * x.scaled_max(k[0]))
        sc = 0.85 * min((tol / e_abs) ** 0.2, (tol / e_rel) ** 0.25)
        hn = min(max(h * min(max(sc, 0.2), 5.0), 1e-15), 1e-10)
        if (e_abs <= tol and e_rel <= tol) or hn == 1e-15:
            if t_end and t + h > t_end:
                h, k = t_end - t, []
                for row in _RKF45_B:
                    k.append(x.dmdt(M + h * sum(b * v for b, v in zip(row, k)) if row else M))
                return x.norm(M + h * sum(c * v for c, v in zip(_RKF45_C4, k)))
            M, t, done = x.norm(M + h * sum(c * v for c, v in zip(_RKF45_C4, k))), t + h, done + 1
        h = hn
    return M


def exact(case, seed):
    if case["kind"] == "batch":
        return None
    shape, delta = _shape(case), _delta(case)
    if case["kind"] == "conv":
        M = _state(shape, 8e5, "random", int(seed)).astype(np.float64 if case["precision"] == "fp64" else np.float32)
        x = _Exact(shape, delta, PHYSICS["plain"])
        return x.demag(torch.as_tensor(M, dtype=torch.float64, device=x.dev))
    if case["kind"] == "rhs":
        p, d = PHYSICS["uniaxial"], _rhs_inputs(case, int(seed))
        x = _Exact(shape, delta, p)
        M, k0 = (torch.as_tensor(d[k], device=x.dev) for k in ("M", "k0"))
        Hd, He, Ha = x.demag(M), x.exchange(M), x.uniaxial(M)
        X = torch.linalg.cross(M, He, dim=0)
        gp = GAMMA / (1 + p["alpha"] ** 2)
        dM = -gp * X - p["alpha"] * gp / p["Ms"] * torch.linalg.cross(M, X, dim=0)
        y = M + 1e-13 * (_RKF45_B[2][0] * k0 + _RKF45_B[2][1] * dM)
        V = delta[0] * delta[1] * delta[2]
        a = x._vec(p["axis1"])
        return dict(Hd=Hd, He=He, Ha=Ha, dM=dM, y=y, e_exch=float((M / p["Ms"] * He).sum()) * -MU0 / 2 * V,
                    e_aniso=float((p["k_uni"] * torch.linalg.cross(a.expand_as(M), M / p["Ms"], dim=0).square().sum(0)).sum()))
    # whole trajectories: where plain torch follows them in seconds
    if case["method"] == "dp54" or case["nx"] * case["ny"] * case["nz"] > 250000:
        return None
    kw = _material(case)
    x = _Exact(shape, delta, kw)
    M = torch.as_tensor(_state(shape, kw["Ms"], case["state"], int(seed)), device=x.dev)
    if case["precision"] == "fp32":
        M = M.float().double()
    if case["method"] == "rk4":
        return _exact_rk4(x, M, 1e-13, case["steps"])
    return _exact_rkf45(x, M, 1e-13, case["tol"], case["steps"], case["until_ps"] * 1e-12)
