"""Cases of the framework's performance measurement: whole simulations through
`Simulator` (every solver family, FP64 and FP32, with and without the NTFF's
per-step work), batched sweeps through `Batch`, and the surrogate network
through its C entry points.

A simulation case runs what a program runs for one result: create the solver
(grid, coefficients, structure fill), advance it, read the outputs, finish.  The
C API holds one active solver per process, so a state is the description of
the run and every pass builds its own solver.  Outputs of FP32 runs are handed
on in single precision, which is what they carry; FP64 runs stay in FP64.
"""
import ctypes
import math

import numpy as np
import torch

import mpifdtd_amd as m
from mpifdtd_amd import batch as mb

SOLVERS = {"mpi_tm": m.MPI_TM_UPML_2D, "mpi_te": m.MPI_TE_UPML_2D, "tm": m.TM_UPML_2D, "te": m.TE_UPML_2D,
           "split_tm": m.TM_2D, "split_te": m.TE_2D, "ns_tm": m.NS_TM_2D, "ns_te": m.NS_TE_2D}
MODELS = {"vacuum": m.NO_MODEL, "mie": m.MIE_CYLINDER, "layer": m.LAYER, "zigzag": m.ZIGZAG, "morpho": m.MORPHO_SCALE}
SWEEP_NM = np.arange(380.0, 781.0, 5.0)  # the sweep's 81 wavelengths
MLP_DIMS = (13, 512, 512, 512, 180)
MLP_BATCH = 1024


def _sim(name, solver, model, nx, ny, h, pml, steps, prec, out, **kw):
    """One simulation: nx x ny cells (UPML / PML included) of h nm; out: the outputs read, joined by '+'."""
    d = dict(kind="sim", solver=solver, model=model, nx=nx, ny=ny, h=h, pml=pml, steps=steps, prec=prec, out=out,
             ntff=False, T=0, R=16, launch=0, angle=0, c0=0.7071, point=False)
    d.update(kw)
    if name:
        d["name"] = name
    return d


def listed():
    return [
        # the smallest runs of the reference's flow (its sample grids, h = 50 nm), everything at its
        # default: FP64 and the per-step NTFF; launches and set-up are the time
        _sim("mpi_tm64_mie_80x80_ntff", "mpi_tm", "mie", 80, 80, 50, 10, 200, "fp64", "fields+far", ntff=True),
        # vacuum with a point source on 256 x 256 + 10 UPML cells, Courant 0.5, 2000 steps, FP64 fields
        _sim("mpi_tm64_point_276x276", "mpi_tm", "vacuum", 276, 276, 5, 10, 2000, "fp64", "fields", c0=0.5, point=True),
        # the Mie cylinder at full length, FP64: the drop-in for the reference's solver
        _sim("mpi_tm64_mie_1056x1056", "mpi_tm", "mie", 1056, 1056, 5, 16, 8000, "fp64", "fields+far"),
        # the plain pulse solver with the per-step NTFF and the spectra the reference writes, odd and non-square
        _sim("te64_mie_531x402_spectra", "te", "mie", 531, 402, 10, 10, 3000, "fp64", "fields+spectra", ntff=True, angle=30),
        # the solver the reference's main.c selects (non-standard FDTD TE), on the Mie grid
        _sim("ns_te64_mie_1056x1056", "ns_te", "mie", 1056, 1056, 5, 16, 4000, "fp64", "fields"),
        # the split-field PML solver, odd and non-square
        _sim("split_tm64_mie_901x653", "split_tm", "mie", 901, 653, 5, 16, 3000, "fp64", "fields"),
        # the Mie cylinder in FP32, the tuned blocking of that grid, 8000 steps
        _sim("mpi_tm32_mie_1056x1056", "mpi_tm", "mie", 1056, 1056, 5, 16, 8000, "fp32", "fields+far", T=8),
        # the same with the reference's per-step time-domain NTFF, TE
        _sim("mpi_te32_mie_1056x1056_ntff", "mpi_te", "mie", 1056, 1056, 5, 16, 4000, "fp32", "far+spectra", ntff=True, T=8),
        # the wavelength sweep on the Morpho-scale grid, the library's headline: FP32 pulse run with the
        # running DFT at 81 wavelengths (a full run has 20000 steps, each the same work)
        _sim("tm32_sweep81_8256x4160", "tm", "morpho", 8256, 4160, 5, 32, 8000, "fp32", "dft", angle=90, T=10, R=20, launch=8),
        # uneven multilayer / zigzag instances, TM and TE, advanced as one batch
        dict(kind="batch", name="batch_uneven_16", n=16, grid="sweep", side=0, h=5, steps=800, T=8, R=16),
        # one inference sweep of a surrogate member: 65536 queries in batches of 1024
        dict(kind="mlp_forward", name="mlp_forward_65536", rows=65536),
        # one training epoch of a surrogate member over 20000 spectra in batches of 1024
        dict(kind="mlp_epoch", name="mlp_epoch_20000", rows=20000),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("sim64", "sim32", "batch", "mlp_forward", "mlp_epoch"), (6, 5, 2, 1, 1))[0]
    if kind == "mlp_forward":
        return dict(kind=kind, rows=_logint(rng, 1, 65536))
    if kind == "mlp_epoch":
        return dict(kind=kind, rows=_logint(rng, 300, 20000))
    if kind == "batch":
        if rng.random() < 0.5:
            return dict(kind=kind, n=rng.randint(2, 16), grid="sweep", side=0, h=5, steps=rng.randint(200, 800), T=8, R=16)
        # the surrogate's data generator: morpho-scale structures on one reduced square grid, CW
        return dict(kind=kind, n=_logint(rng, 4, 64), grid="morpho", side=rng.randint(300, 600), h=10,
                    steps=rng.randint(200, 1000), T=8, R=16)
    f64 = kind == "sim64"
    solver = rng.choice(list(SOLVERS) if f64 else ["mpi_tm", "mpi_te", "tm", "te"])
    pml = rng.choice((10, 16, 32))
    small = 2 * pml + 40
    nx, ny = _logint(rng, small, 1400 if f64 else 3000), _logint(rng, small, 1400 if f64 else 3000)
    ny = min(max(ny, nx // 3), 3 * nx)
    steps = min(rng.randint(200, 3000), int((4e9 if f64 else 4e10) / (nx * ny)))
    upml = solver in ("mpi_tm", "mpi_te", "tm", "te")
    ntff = upml and rng.random() < 0.4
    mode = rng.choice(("fields", "far", "dft")) if upml else "fields"
    out = {"fields": "fields", "far": "fields+far", "dft": "dft+far"}[mode]
    if ntff:
        out += "+spectra"
    T = rng.choice((4, 8, 10))
    return _sim("", solver, rng.choice(("mie", "mie", "layer", "zigzag", "morpho")), nx, ny, rng.choice((5, 10)), pml, steps,
                "fp64" if f64 else "fp32", out, ntff=ntff, angle=rng.choice((0, 30, 90, 135)), T=0 if f64 else T,
                R=16, launch=0)


# ---------------------------------------------------------------- inputs

def _run_params(case, seed):
    """Wavelength and structure of a run, from the seed: (lambda_nm, model parameters)."""
    r = np.random.RandomState((seed * 7919 + 17) % (1 << 31))
    lam = int(r.randint(450, 701))
    size = min(case["nx"], case["ny"]) * case["h"]
    p = {}
    if case["model"] == "mie":
        p = dict(circle_radius_nm=float(int(size * (0.1 + 0.08 * r.rand()))), circle_n=1.4 + 0.4 * float(r.rand()))
    elif case["model"] == "layer":
        t0, t1 = int(r.randint(50, 150)), int(r.randint(50, 150))
        p = dict(ml_n0=1.2 + 0.8 * float(r.rand()), ml_n1=1.0, ml_thick_nm0=t0, ml_thick_nm1=t1,
                 ml_layer_num=max(1, int(0.5 * size / (t0 + t1))) if 0.5 * size < 20 * (t0 + t1) else 20,
                 ml_width_nm0=int(0.4 * size), ml_width_nm1=int(0.4 * size), ml_branch_nm=0, ml_use_gap=0)
    elif case["model"] == "zigzag":
        p = dict(zz_width_nm=max(50, int(0.1 * size)), zz_thick_nm=max(30, int(0.04 * size)), zz_degree=int(r.randint(20, 70)),
                 zz_n=1.3 + 0.4 * float(r.rand()), zz_layer_num=3)
    elif case["model"] == "morpho":
        p = dict(mo_n=1.3 + 0.4 * float(r.rand()), mo_layer_num=int(r.randint(4, 9)), mo_randomness=0, mo_seed=0)
    return lam, p


def _weights(seed):
    """One surrogate member's weights as the library initialises them: uniform in +-1/sqrt(fan in); biases small."""
    r = np.random.RandomState((seed * 104729 + 3) % (1 << 31))
    return [(((2 * r.rand(o, i) - 1) / math.sqrt(i)).astype(np.float32), (0.02 * (r.rand(o) - 0.5)).astype(np.float32))
            for i, o in zip(MLP_DIMS[:-1], MLP_DIMS[1:])]


def _spectra(seed, rows):
    """Features in [0, 1] and targets like scaled reflectances: smooth positive curves over the angles."""
    r = np.random.RandomState((seed * 31337 + 5) % (1 << 31))
    x = r.rand(rows, MLP_DIMS[0]).astype(np.float32)
    ang = np.linspace(0, math.pi, MLP_DIMS[-1], dtype=np.float32)
    c = r.rand(MLP_DIMS[0], 6).astype(np.float32)
    y = np.abs(np.sin(x @ c) @ np.cos(np.outer(np.arange(6, dtype=np.float32), ang))) / 3
    return x, y.astype(np.float32)


class _Net:
    """A network of the C interface (mpifdtd_surrogate.h), destroyed with the state."""

    def __init__(self, weights):
        L = m.lib()
        dims = (ctypes.c_int * len(MLP_DIMS))(*MLP_DIMS)
        self.h = ctypes.c_void_p()
        _ok(L.mlp_create(len(MLP_DIMS) - 1, dims, MLP_BATCH, ctypes.c_ulonglong(1), ctypes.byref(self.h)))
        self.set(weights)

    def set(self, weights):
        for l, (w, b) in enumerate(weights):
            _ok(m.lib().mlp_set_params(self.h, l, _fp(w), _fp(b)))

    def get(self):
        out = []
        for i, o in zip(MLP_DIMS[:-1], MLP_DIMS[1:]):
            w, b = np.empty((o, i), np.float32), np.empty(o, np.float32)
            _ok(m.lib().mlp_get_params(self.h, len(out), _fp(w), _fp(b)))
            out.append((w, b))
        return out

    def __del__(self):
        if self.h:
            m.lib().mlp_destroy(self.h)
            self.h = None


def _ok(rc):
    if rc != 0:
        raise RuntimeError("library call failed (%d): %s" % (rc, m.lib().fdtd_hip_last_error().decode()))


def _fp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def _batch_items(case, seed):
    if case["grid"] == "sweep":
        # the instances' sizes and modes are the case's own (every seed the same amount of work);
        # structures, wavelengths and optics come from the seed
        shape, spec = mb.sweep_spec(seed=1, n=case["n"], h_nm=case["h"]), mb.sweep_spec(seed=seed + 2, n=case["n"], h_nm=case["h"])
        items = []
        for a, b in zip(shape, spec):
            q = dict(b, mode=a["mode"], width_nm=a["width_nm"], height_nm=a["height_nm"], steps=case["steps"], params=dict(b["params"]))
            span = 0.8 * a["side"] * case["h"]
            if q["kind"] == "multilayer":
                p = q["params"]
                p["ml_layer_num"] = min(p["ml_layer_num"], max(1, int(span // (p["ml_thick_nm0"] + p["ml_thick_nm1"]))))
                p["ml_width_nm0"] = p["ml_width_nm1"] = int(0.5 * a["side"] * case["h"])
            else:
                q["params"]["zz_layer_num"] = min(q["params"]["zz_layer_num"], 3)
            items.append(q)
        return mb.sweep_instances(items)
    from mpifdtd_amd import surrogate as ms
    w = case["side"] * case["h"]
    return [mb.item(m.MPI_TM_UPML_2D, m.MORPHO_SCALE, w, w, case["h"], 16, d["lambda_nm"], 90, case["steps"],
                    mo_randomness=0, mo_seed=0, **{k: d[k] for k, *_ in ms.GEOMETRY})
            for d in ms.morpho_spec(seed=seed, n=case["n"])]


def prepare(case, seed):
    if case["kind"] == "sim":
        lam, p = _run_params(case, seed)
        return dict(case=case, params=m.model_params(**p),
                    fi=m.field_info(case["nx"] * case["h"], case["ny"] * case["h"], case["h"], case["pml"], lam, case["angle"],
                                    case["steps"]))
    if case["kind"] == "batch":
        return dict(case=case, items=_batch_items(case, seed))
    w = _weights(seed)
    x, y = _spectra(seed, case["rows"])
    return dict(case=case, w=w, net=_Net(w), x=torch.from_numpy(x).cuda(), t=torch.from_numpy(y).cuda())


# ---------------------------------------------------------------- one pass

def _run_sim(s):
    c = s["case"]
    f32 = c["prec"] == "fp32"
    kw = dict(T=c["T"], R=c["R"]) if f32 else {}
    sim = m.Simulator(SOLVERS[c["solver"]], MODELS[c["model"]], s["fi"], params=s["params"], c0=c["c0"], point_source=c["point"],
                      ntff_time=c["ntff"], precision=c["prec"], **kw)
    try:
        if c["launch"]:
            sim.set_launch_mode(c["launch"])
        want = c["out"].split("+")
        if "dft" in want:
            sim.set_dft(SWEEP_NM)
        sim.calc(c["steps"])
        out = {}
        if "fields" in want:
            out["fields"] = [a.astype(np.complex64) if f32 else a for a in sim.fields()]
        if "far" in want:
            out["far"] = sim.far_field()
        if "spectra" in want:
            out["spectra"] = sim.time_spectra()
        if "dft" in want:
            out["dft"] = sim.dft()
            out["dft_spectra"] = sim.dft_spectra()
    finally:
        sim.finish()
    if f32:
        for k in ("far", "dft"):
            if k in out:
                out[k] = out[k].astype(np.complex64)
        for k in ("spectra", "dft_spectra"):
            if k in out:
                out[k] = out[k].astype(np.float32)
    return out


def _run_batch(s):
    c = s["case"]
    with mb.Batch(s["items"], T=c["T"], R=c["R"]) as b:
        b.run()
        return dict(far=np.stack([b.far_field(i) for i in range(c["n"])]).astype(np.complex64))


def run(state):
    c = state["case"]
    if c["kind"] == "sim":
        return _run_sim(state)
    if c["kind"] == "batch":
        return _run_batch(state)
    L, net, x, rows = m.lib(), state["net"], state["x"], c["rows"]
    if c["kind"] == "mlp_forward":
        y = torch.empty((rows, MLP_DIMS[-1]), dtype=torch.float32, device="cuda")
        for i in range(0, rows, MLP_BATCH):  # as MLP.forward_into does
            n = min(MLP_BATCH, rows - i)
            _ok(L.mlp_forward(net.h, x[i].data_ptr(), n, y[i].data_ptr()))
        return y
    net.set(state["w"])  # the epoch starts from the state's weights; Adam's moments go on, as in a fit
    loss = ctypes.c_float()
    _ok(L.mlp_train_epoch(net.h, x.data_ptr(), state["t"].data_ptr(), rows, MLP_BATCH, ctypes.c_ulonglong(7), ctypes.c_float(1e-3),
                          ctypes.byref(loss)))
    return dict(loss=np.float32(loss.value), params=[a for wb in net.get() for a in wb])


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    if case["kind"] == "mlp_forward":
        nw = sum(i * o for i, o in zip(MLP_DIMS[:-1], MLP_DIMS[1:]))
        return {"bytes": 4.0 * case["rows"] * (MLP_DIMS[0] + MLP_DIMS[-1]) + 4.0 * nw, "flops": 2.0 * nw * case["rows"]}
    if case["kind"] == "mlp_epoch":
        nw = sum(i * o for i, o in zip(MLP_DIMS[:-1], MLP_DIMS[1:]))
        return {"bytes": 4.0 * case["rows"] * (MLP_DIMS[0] + MLP_DIMS[-1]) + 8.0 * nw, "flops": 6.0 * nw * case["rows"]}
    if case["kind"] == "batch":
        if case["grid"] == "sweep":
            cells = sum((a["side"] + 32) ** 2 for a in mb.sweep_spec(seed=1, n=case["n"], h_nm=case["h"]))
        else:
            cells = case["n"] * case["side"] ** 2
        return {"bytes": cells * (4.0 + 24.0), "flops": 22.0 * cells * case["steps"]}
    cells, word = case["nx"] * case["ny"], 8.0 if case["prec"] == "fp64" else 4.0
    neps = 2 if case["solver"].endswith("te") else 1
    flops = 22.0 * cells * case["steps"]  # two curls of complex values per cell and step
    ring = 2 * (case["nx"] + case["ny"] - 4 * (case["pml"] + 5))
    if case["ntff"]:  # 360 angles x E and H x three complex taps
        flops += 360.0 * ring * 2 * 12 * case["steps"]
    if "dft" in case["out"]:
        flops += SWEEP_NM.size * ring * 2 * 8.0 * case["steps"]
    return {"bytes": cells * (word * neps + 6 * word), "flops": flops}


# ---------------------------------------------------------------- the same in 64 bits, without the framework

def _circle_eps(case, p, sx, sy, col, row):
    """Relative permittivity at every cell centre + (sx, sy): the cylinder, its rim sampled 10 x 10."""
    nx, ny, pml = case["nx"], case["ny"], case["pml"]
    X = (torch.arange(nx, dtype=torch.float64, device="cuda") + sx)[:, None]
    Y = (torch.arange(ny, dtype=torch.float64, device="cuda") + sy)[None, :]
    one = torch.ones((nx, ny), dtype=torch.float64, device="cuda")
    if case["model"] == "vacuum":
        return one
    r, e = p["circle_radius_nm"] / case["h"], p["circle_n"] ** 2
    dx, dy = X - nx // 2, Y - ny // 2
    part = torch.zeros_like(one)
    for i in np.arange(-4.5, 5):
        for j in np.arange(-4.5, 5):
            part += ((dx + col * i / 10) ** 2 + (dy + row * j / 10) ** 2 <= r * r).double()
    part /= 100
    len2 = dx * dx + dy * dy
    part = torch.where(len2 >= (r + 1) ** 2, torch.zeros_like(part), torch.where(len2 <= (r - 1) ** 2, torch.ones_like(part), part))
    out = (X < pml) | (Y < pml) | (X > nx - pml) | (Y > ny - pml)
    return torch.where(out, one, e * part + (1 - part))


def _sigma(n, pml, shift):
    x = np.arange(n) + shift
    v = np.where(x < pml, (pml - x) / pml, np.where(x < n - pml, 0.0, (x - (n - pml - 1)) / pml))
    return v * v


class _Exact:
    """The UPML solvers (MPI and plain, TM and TE) step by step on whole arrays in complex128."""

    def __init__(self, case, seed):
        self.case, (lam, self.p) = case, _run_params(case, seed)
        self.tm, self.mpi = case["solver"].endswith("tm"), case["solver"].startswith("mpi")
        nx, ny, pml, c0 = case["nx"], case["ny"], case["pml"], case["c0"]
        self.k = 2 * math.pi / (lam / case["h"])
        self.w = c0 * self.k
        self.mu0 = 1.0 / c0 / c0
        smax = 3.0 * c0 / 2 / pml * math.log(1e8) * (1 / math.cos(math.pi / 3) if self.tm else 1)
        col = lambda v: torch.from_numpy(smax * v).cuda()[:, None]  # noqa: E731
        row = lambda v: torch.from_numpy(smax * v).cuda()[None, :]  # noqa: E731
        self.x0, self.xh = col(_sigma(nx, pml, 0)), col(_sigma(nx, pml, 0.5))
        self.y0, self.yh = row(_sigma(ny, pml, 0)), row(_sigma(ny, pml, 0.5))
        z = lambda: torch.zeros((nx + 2, ny + 2), dtype=torch.complex128, device="cuda")  # noqa: E731
        self.f = [z() for _ in range(3)]  # TM Ez Hx Hy, TE Ex Ey Hz, with a ring of zeros around the cells
        self.a = [torch.zeros((nx, ny), dtype=torch.complex128, device="cuda") for _ in range(6)]
        self.eps = [_circle_eps(case, self.p, 0, 0, 1, 1)] if self.tm else [
            _circle_eps(case, self.p, 0.5, 0, 0, 1), _circle_eps(case, self.p, 0, 0.5, 1, 0)]
        self.live = torch.ones((nx, ny), dtype=torch.float64, device="cuda")
        if not self.mpi:  # the plain solvers leave the edge cells alone
            self.live[0], self.live[-1], self.live[:, 0], self.live[:, -1] = 0, 0, 0, 0

    def source(self, q, t):
        """The incident field's term on component q at time t."""
        c, nx, ny = self.case, self.case["nx"], self.case["ny"]
        rad = c["angle"] * math.pi / 180
        e = self.eps[q]
        gx, gy = (0.5, 0) if not self.mpi and not self.tm and q == 0 else (0, 0.5) if not self.mpi and not self.tm else (0, 0)
        X = (torch.arange(nx, dtype=torch.float64, device="cuda") + gx)[:, None]
        Y = (torch.arange(ny, dtype=torch.float64, device="cuda") + gy)[None, :]
        if self.mpi:
            amp = (1 - math.exp(-(0.01 * t) ** 2)) * (1 / e - 1)
            ph = X * (math.cos(rad) * self.k) + Y * (math.sin(rad) * self.k) - self.w * t
        else:
            cx, cy = math.cos(rad) / c["c0"], math.sin(rad) / c["c0"]
            t0 = -((nx / 2 + gx) * cx + (ny // 2 + gy) * cy) + 500
            r = X * cx + Y * cy - (t - t0)
            dot = 1.0 if self.tm else (math.cos, math.sin)[q]((c["angle"] + 90) * math.pi / 180)
            amp, ph = dot * torch.exp(-(r / 50) ** 2) * (1 / e - 1), r * self.w
        return torch.polar(torch.ones_like(ph), ph) * amp

    def e_half(self, t):
        f, a, i = self.f, self.a, (slice(1, -1), slice(1, -1))
        lo_x, lo_y = (slice(0, -2), slice(1, -1)), (slice(1, -1), slice(0, -2))
        if self.tm:
            curl = f[2][i] - f[2][lo_x] - f[1][i] + f[1][lo_y]
            j = (2 - self.x0) / (2 + self.x0) * a[0] + 2 / (2 + self.x0) * curl
            a[1] = ((2 - self.y0) * a[1] + 2 * (j - a[0])) / (2 + self.y0)
            a[0] = j
            e = a[1] / self.eps[0]
            if self.case["point"]:
                ray = 1 - math.exp(-(0.01 * t) ** 2)
                e[self.case["nx"] // 2, self.case["ny"] // 2] += complex(ray * math.cos(self.w * t), ray * math.sin(self.w * t))
            f[0][i] = (e + self.source(0, t)) * self.live
        else:
            j = (2 - self.y0) / (2 + self.y0) * a[0] + 2 / (2 + self.y0) * (f[2][i] - f[2][lo_y])
            a[1] = a[1] + ((2 + self.xh) * j - (2 - self.xh) * a[0]) / 2
            a[0] = j
            j = a[2] + f[2][lo_x] - f[2][i]
            a[3] = ((2 - self.x0) * a[3] + (2 + self.yh) * j - (2 - self.yh) * a[2]) / (2 + self.x0)
            a[2] = j
            f[0][i] = (a[1] / self.eps[0] + (0 if self.mpi else self.source(0, t))) * self.live
            f[1][i] = (a[3] / self.eps[1] + self.source(1, t)) * self.live

    def h_half(self):
        f, a, i = self.f, self.a, (slice(1, -1), slice(1, -1))
        hi_x, hi_y = (slice(2, None), slice(1, -1)), (slice(1, -1), slice(2, None))
        if self.tm:
            n = ((2 - self.yh) * a[2] - 2 * (f[0][hi_y] - f[0][i])) / (2 + self.yh)
            a[3] = a[3] + ((2 + self.x0) * n - (2 - self.x0) * a[2]) / 2
            a[2] = n
            n = a[4] + f[0][hi_x] - f[0][i]
            a[5] = ((2 - self.xh) * a[5] + (2 + self.y0) * n - (2 - self.y0) * a[4]) / (2 + self.xh)
            a[4] = n
            f[1][i], f[2][i] = a[3] / self.mu0 * self.live, a[5] / self.mu0 * self.live
        else:
            curl = f[1][hi_x] - f[1][i] - f[0][hi_y] + f[0][i]
            n = ((2 - self.xh) * a[4] - 2 * curl) / (2 + self.xh)
            a[5] = ((2 - self.yh) * a[5] + 2 * (n - a[4])) / (2 + self.yh)
            a[4] = n
            f[2][i] = a[5] / self.mu0 * self.live

    def advance(self):
        for t in range(self.case["steps"]):
            if self.mpi:
                self.e_half(t)
                self.h_half()
            else:
                self.h_half()
                self.e_half(t)
            self.a = [v * self.live for v in self.a] if not self.mpi else self.a

    def far(self):
        """The far field at 360 angles from the fields on the closed contour 5 cells inside the UPML."""
        c, nx, ny = self.case, self.case["nx"], self.case["ny"]
        lo, rt, tp = c["pml"] + 5, nx - c["pml"] - 5, ny - c["pml"] - 5
        cx, cy, Z0 = nx // 2, ny // 2, math.sqrt(self.mu0)
        r0 = 1e6 * 500 / c["h"]
        coef = np.sqrt(1j * self.k / (8 * math.pi * r0)) * np.exp(1j * self.k * r0) * math.sqrt(c["h"])
        ang = torch.arange(360, dtype=torch.float64, device="cuda") * math.pi / 180
        cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
        f, s = self.f, 0 if self.tm else -1  # TE: the contour's indices count the ring
        xs, ys = torch.arange(lo, rt, device="cuda"), torch.arange(lo, tp, device="cuda")
        N, M, K = [torch.zeros(360, dtype=torch.complex128, device="cuda") for _ in range(3)]
        for horiz, at, sg in ((1, lo, 1.0), (0, rt, 1.0), (1, tp, -1.0), (0, lo, -1.0)):
            i, j = (xs, torch.full_like(xs, at)) if horiz else (torch.full_like(ys, at), ys)
            g = 0.0 if self.tm else 0.5
            ph = self.k * (cs * (i - cx + (g if horiz else 0.0)) + sn * (j - cy + (0.0 if horiz else g)))
            w = sg * torch.polar(torch.ones_like(ph), ph)
            at2 = lambda v, di, dj: v[i + 1 + s + di, j + 1 + s + dj]  # noqa: E731
            back = (0, -1) if horiz else (-1, 0)
            hf = (f[1] if horiz else f[2]) if self.tm else f[2]
            h = 0.5 * (at2(hf, 0, 0) + at2(hf, *back))
            ef = f[0] if self.tm or horiz else f[1]
            if self.tm:
                N += (w * h).sum(1)
                (M if horiz else K).add_((w * at2(ef, 0, 0)).sum(1))
            else:
                (M if horiz else K).sub_((w * h).sum(1))
                N -= (w * at2(ef, 0, 0)).sum(1)
        cs, sn = cs[:, 0], sn[:, 0]
        proj = -M * sn + K * cs
        return coef * (Z0 * N + proj if self.tm else Z0 * proj - N)

    def fields(self):
        i = (slice(None), slice(None)) if self.mpi else (slice(1, -1), slice(1, -1))
        return [v[i].contiguous() for v in self.f]


def _exact_mlp(case, seed):
    W = [(torch.from_numpy(w).cuda().double(), torch.from_numpy(b).cuda().double()) for w, b in _weights(seed)]
    x, t = (torch.from_numpy(a).cuda().double() for a in _spectra(seed, case["rows"]))

    def forward(x):
        for l, (w, b) in enumerate(W):
            x = x @ w.T + b
            x = torch.nn.functional.gelu(x) if l + 1 < len(W) else x
        return x

    if case["kind"] == "mlp_forward":
        return torch.cat([forward(x[i:i + 8192]) for i in range(0, case["rows"], 8192)])
    # the epoch: SplitMix64 Fisher-Yates order, mean squared error, Adam
    mask, s, perm = (1 << 64) - 1, 7, list(range(case["rows"]))
    for i in range(case["rows"] - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        q = (z ^ (z >> 31)) % (i + 1)
        perm[i], perm[q] = perm[q], perm[i]
    perm = torch.tensor(perm, device="cuda")
    par = [a.requires_grad_() for wb in W for a in wb]
    opt = torch.optim.Adam(par, lr=1e-3)
    total = 0.0
    for i in range(0, case["rows"], MLP_BATCH):
        sel = perm[i:i + MLP_BATCH]
        loss = ((forward(x[sel]) - t[sel]) ** 2).mean()
        opt.zero_grad()
        loss.backward()
        opt.step()
        total += float(loss.detach()) * len(sel)
    return dict(loss=total / case["rows"], params=[a.detach() for a in par])


def exact(case, seed):
    if case["kind"].startswith("mlp"):
        return _exact_mlp(case, seed)
    # The UPML solvers on a cylinder or in vacuum.  None for the others: the batches' and the
    # large grid's steps would take minutes here; the split-field and non-standard solvers and the
    # layered structures have no independent restatement in this file; nor have the spectra.
    if case["kind"] != "sim" or case["solver"] not in ("mpi_tm", "mpi_te", "tm", "te") or case["model"] not in ("vacuum", "mie"):
        return None
    if case["steps"] * (case["nx"] * case["ny"] * 1.3e-9 + 0.6e-3) > 18:
        return None
    sim = _Exact(case, seed)
    sim.advance()
    want = case["out"].split("+")
    out = {k: None for k in want}
    if "fields" in want:
        out["fields"] = sim.fields()
    if "far" in want:
        out["far"] = sim.far()
    if "dft" in want:
        out["dft_spectra"] = None
    return out
