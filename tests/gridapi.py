"""Grids through the C ABI of fdtd_hip.h, for what the solvers' entry points do not
set: eps maps of any values, runs with and without the blocked steps, and a plain
NumPy restatement of the four UPML solvers without an absorbing layer."""
import ctypes

import numpy as np

TM, TE = 0, 1
MPI, PLAIN, SPLIT, NS = 0, 1, 2, 3
C0 = 0.7071
MU0 = 1.0 / C0**2


class Desc(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_int) for n in ("mode", "flavour", "precision", "N_PX", "N_PY", "N_PML", "top", "bottom",
                                             "left", "right", "cx", "cy")] + [("rf_per_c", ctypes.c_double)] +
                [(n, ctypes.c_int) for n in ("array_size", "max_time")] +
                [(n, ctypes.c_double) for n in ("c0", "mu0", "z0", "eps0")] +
                [(n, ctypes.c_int) for n in ("ntff_time", "point_source")])


class Tables(ctypes.Structure):
    _dp = ctypes.POINTER(ctypes.c_double)
    _fields_ = [("x", _dp * 5), ("sx", _dp), ("y", _dp * 4), ("sy", _dp)]


class Step(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_double) for n in ("time", "ray_coef", "omega", "k", "angle_deg", "ps_re", "ps_im", "dot_x",
                                                "dot_y")] + [(n, ctypes.c_int) for n in ("use_x", "use_y")])


class Grid:
    """A grid of `mode` and `flavour`, every coefficient 1 but those of an absorbing
    layer of `pml` cells on the rows (sigma rising to `sig`); eps 1."""

    def __init__(self, mode, flavour, nx, ny, pml=0, sig=0.4):
        import mpifdtd_amd as m
        from mpifdtd_amd._native import check, dptr
        self.L, self.check, self.dptr = m.lib(), check, dptr
        self.mode, self.flavour = mode, flavour
        self.off = 1 if flavour == MPI else 0
        self.shape = (nx + 2 * self.off, ny + 2 * self.off)
        L = self.L
        V, I, P = ctypes.c_void_p, ctypes.c_int, ctypes.POINTER
        for name, args in (("create", (P(Desc), P(V))), ("destroy", (V,)), ("set_coefs", (V, P(Tables))),
                           ("set_eps", (V, I, V)), ("get_field", (V, I, V)), ("set_field", (V, I, V)), ("reset", (V,)),
                           ("step", (V, P(Step))), ("steps", (V, P(Step), I)), ("set_dft", (V, V, I)),
                           ("get_dft", (V, V))):
            f = getattr(L, "fdtd_hip_grid_" + name)
            f.restype, f.argtypes = I, list(args)
        b = max(2, pml + 2)
        d = Desc(mode, flavour, 0, nx, ny, pml, ny - b, b, b, nx - b, nx // 2, ny // 2, 0.0, 64, 64, C0, MU0, 1.0 / C0, 1.0,
                 0, 0)
        self.h = V()
        check(L.fdtd_hip_grid_create(ctypes.byref(d), ctypes.byref(self.h)), "create")
        x = np.ones((6, nx))
        y = np.ones((5, ny))
        x[5] = y[4] = 0.0
        if pml:
            i = np.arange(nx)
            depth = np.maximum(0, np.maximum(pml - i, i - (nx - 1 - pml))) / pml
            s = sig * depth**2
            if mode == TM:
                x[0], x[1], x[2], x[3], x[4] = (2 - s) / (2 + s), 2 / (2 + s), (2 + s) / 2, (2 - s) / 2, (2 - s) / (2 + s)
            else:
                x[0], x[1], x[2], x[3], x[4] = (2 + s) / 2, (2 - s) / 2, (2 - s) / (2 + s), (2 - s) / (2 + s), 2 / (2 + s)
            x[5] = s
        t = Tables()
        for q in range(5):
            t.x[q] = dptr(x[q])
        for q in range(4):
            t.y[q] = dptr(y[q])
        t.sx, t.sy = dptr(x[5]), dptr(y[4])
        check(L.fdtd_hip_grid_set_coefs(self.h, ctypes.byref(t)), "set_coefs")
        self.set_eps([np.ones(self.shape)] * 3)

    def set_eps(self, maps):
        for q, e in enumerate(maps):
            e = np.ascontiguousarray(e, np.float64)
            self.check(self.L.fdtd_hip_grid_set_eps(self.h, q, e.ctypes.data), "set_eps")

    def params(self, t0, n, omega=0.2, angle=35.0):
        """The parameters of the steps of times t0 .. t0 + n - 1: a wave of that frequency and angle."""
        p = (Step * n)()
        co, si = np.cos(np.deg2rad(angle + 90)), np.sin(np.deg2rad(angle + 90))
        for q in range(n):
            t = t0 + q
            p[q] = Step(t, 1.0 - np.exp(-0.1 * t), omega, omega / C0, angle, 0, 0, co, si, 1, 1)
        return p

    def steps(self, p):
        self.check(self.L.fdtd_hip_grid_steps(self.h, p, len(p)), "steps")

    def step(self, p):
        self.check(self.L.fdtd_hip_grid_step(self.h, ctypes.byref(p)), "step")

    def field(self, q):
        a = np.empty(self.shape, np.complex128)
        self.check(self.L.fdtd_hip_grid_get_field(self.h, q, a.ctypes.data), "get_field")
        return a

    def set_field(self, q, a):
        a = np.ascontiguousarray(a, np.complex128)
        self.check(self.L.fdtd_hip_grid_set_field(self.h, q, a.ctypes.data), "set_field")

    def reset(self):
        self.check(self.L.fdtd_hip_grid_reset(self.h), "reset")

    def set_dft(self, omega):
        w = np.ascontiguousarray(omega, np.float64)
        self.nf = w.size
        self.check(self.L.fdtd_hip_grid_set_dft(self.h, w.ctypes.data, w.size), "set_dft")

    def dft(self):
        out = np.empty((self.nf, 3, 360), np.complex128)
        self.check(self.L.fdtd_hip_grid_get_dft(self.h, out.ctypes.data), "get_dft")
        return out

    def close(self):
        self.L.fdtd_hip_grid_destroy(self.h)


def reference(mode, flavour, nx, ny, eps, params):
    """The nine arrays after the steps `params` without an absorbing layer, every cell
    E = D / eps + source: mpiTM_UPML.c:196-217, mpiTE_UPML.c:290-304,
    fdtdTM_upml.c:54-66, fdtdTE_upml.c:168-192 with sigma = 0."""
    off = 1 if flavour == MPI else 0
    X, Y = nx + 2 * off, ny + 2 * off
    F = np.zeros((9, X, Y), np.complex128)
    i, j = np.meshgrid(np.arange(X) - off, np.arange(Y) - off, indexing="ij")
    c = np.s_[1:-1, 1:-1]

    def source(p, e, gx, gy, dot):
        a = np.deg2rad(p.angle_deg)
        with np.errstate(divide="ignore"):
            f = np.where(e == 1.0, 0.0, 1.0 / e - 1.0)
        if flavour == MPI:
            return p.ray_coef * f * np.exp(1j * ((i * np.cos(a) + j * np.sin(a)) * p.k - p.omega * p.time))
        cp, sp = np.cos(a) / C0, np.sin(a) / C0
        t0 = -((nx / 2.0 + gx) * cp + (ny // 2 + gy) * sp) + 500
        r = (i + gx) * cp + (j + gy) * sp - (p.time - t0)
        return dot * np.exp(-(r / 50.0)**2) * f * np.exp(1j * r * p.omega)

    def d(k, q, dk):  # field q at the neighbour, minus at the cell
        return np.roll(F[q], -k, dk)[c] - F[q][c]

    def ehalf(p):
        if mode == TM:
            curl = -d(-1, 6, 0) + d(-1, 3, 1)
            F[1][c] += curl
            F[2][c] += curl
            F[0][c] = (F[2] / eps[0] + source(p, eps[0], 0, 0, 1.0))[c]
        else:
            for q, m, curl in ((0, 0, -d(-1, 6, 1)), (3, 1, d(-1, 6, 0))):
                F[q + 1][c] += curl
                F[q + 2][c] += curl
                gx, gy = (0, 0) if flavour == MPI else ((0.5, 0.0) if q == 0 else (0.0, 0.5))
                s = source(p, eps[m], gx, gy, p.dot_x if q == 0 else p.dot_y)
                F[q][c] = (F[q + 2] / eps[m] + (0 if flavour == MPI and q == 0 else s))[c]

    def hhalf():
        if mode == TM:
            for q, v in ((3, -d(1, 0, 1)), (6, d(1, 0, 0))):
                F[q + 1][c] += v
                F[q + 2][c] += v
                F[q][c] = F[q + 2][c] / MU0
        else:
            v = -(d(1, 3, 0) - d(1, 0, 1))
            F[7][c] += v
            F[8][c] += v
            F[6][c] = F[8][c] / MU0

    for p in params:
        if flavour == MPI:
            ehalf(p)
            hhalf()
        else:
            hhalf()
            ehalf(p)
    return F
