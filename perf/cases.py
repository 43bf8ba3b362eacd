"""Performance cases: the work a user has the library do, at real sizes.

A case is a dict of plain values.  ``prepare`` makes a program's state (device
arrays, a context, a simulation or ensembles) from the case and a seed,
``run`` makes one pass through the public entry points, ``exact`` computes the
same outputs with torch alone in 64 bits, ``work`` counts the bytes and
operations a pass cannot do without.

Kinds of cases (the public calls they make):

* ``rhs``: one mk_rhs (``Gpu.mk_rhs``), with the filter, the observables and
  the FP32 GW source as options: what a host with its own stepper calls;
* ``fft``: the 3D r2c and c2r transforms (ihg_fft_r2c, ihg_fft_c2r);
* ``rk4``: ``Sim.run_rk4`` over a number of fixed steps;
* ``dopri``: ``Sim.run_dopri853`` over a given step sequence, optionally with
  time-based (dense) outputs;
* ``gsl``: ``Sim.run_gsl`` over one output interval (one step of the method);
* ``ens``: RK4 steps of ensembles of up to three grid sizes
  (``ensemble.run``), per size in graphs, eager, or grouped.

States: phi and dphi homogeneous plus Gaussian fluctuations with the vacuum
spectrum cut at a quarter of the grid, small psi, dpsi and tensor modes, the
values a run passes through.
"""
import math

import torch

import instaheat_amd as ih
from instaheat_amd import ensemble

MASS, PHI0, DPHI0 = 1.0, 1.0093, -0.7137
RTOL, ATOL = 1e-10, 1e-14


def _rhs(name, nx, ny, nz, gw, filt, output=False, fp32=False, bins=64):
    return dict(name=name, kind="rhs", nx=nx, ny=ny, nz=nz, gw=gw, filt=filt,
                output=output, fp32=fp32, bins=bins)


def listed():
    return [
        # the smallest call: one right-hand side of a 16^3 grid, scalar
        # fields alone; launches and latency
        _rhs("rhs 16^3", 16, 16, 16, False, False, bins=16),
        # the plain small configuration: 32^3, no tensors, RK4 dt = 0.01
        dict(name="rk4 32^3", kind="rk4", nx=32, ny=32, nz=32, gw=False,
             filt=True, bins=32, steps=50, dt=0.01),
        # the 64^3 configuration: GW on, DOPRI853, power spectra in 64 log
        # bins at given times (dense output)
        dict(name="dopri 64^3 dense", kind="dopri", nx=64, ny=64, nz=64,
             gw=True, filt=True, bins=64, steps=6, dt=0.02, t_out=2),
        # a box longer in one direction than the others, every axis its own
        # length (a ragged shape), GW on
        _rhs("rhs 64x256x32", 64, 256, 32, True, False),
        # what each save of a run costs: filter, GW and all observables
        _rhs("rhs 128^3 output", 128, 128, 128, True, True, output=True),
        # the same size without tensors, as inside a step
        _rhs("rhs 128^3 scalar", 128, 128, 128, False, False),
        # one step of GSL's RK8PD at 128^3 (13 stages), GW on
        dict(name="gsl 128^3", kind="gsl", nx=128, ny=128, nz=128, gw=True,
             filt=True, bins=64, dt=0.02),
        # the batched configuration: realizations of three grid sizes
        dict(name="ens 48x32 16x64 4x128", kind="ens", n1=32, r1=48, n2=64,
             r2=16, n3=128, r3=4, gw=True, filt=True, bins=32, steps=5,
             dt=0.005, graph=True, grouped=False),
        # few small realizations, an odd number of them
        dict(name="ens 7x16 3x32", kind="ens", n1=16, r1=7, n2=32, r2=3,
             n3=0, r3=0, gw=True, filt=True, bins=32, steps=20, dt=0.005,
             graph=True, grouped=False),
        # the headline configuration: DOPRI853 steps at 256^3, GW on
        dict(name="dopri 256^3", kind="dopri", nx=256, ny=256, nz=256,
             gw=True, filt=True, bins=64, steps=2, dt=0.02, t_out=0),
        # the right-hand side inside those steps with the FP32 GW source
        _rhs("rhs 256^3 fp32", 256, 256, 256, True, False, fp32=True),
        # the largest transform: r2c and c2r of one 512^3 field
        dict(name="fft 512^3", kind="fft", nx=512, ny=512, nz=512),
    ]


def draw(rng):
    def grid(lo, hi, cap):
        while True:
            s = [1 << rng.randint(lo, hi) for _ in range(3)]
            if rng.random() < 0.4:
                s = [s[0]] * 3
            if s[0] * s[1] * s[2] <= cap:
                return dict(nx=s[0], ny=s[1], nz=s[2])

    kind = rng.choice(["rhs", "rhs", "rhs", "rk4", "dopri", "gsl", "ens", "fft"])
    bins = rng.randint(8, 100)
    gw, filt = rng.random() < 0.6, rng.random() < 0.5
    if kind == "rhs":
        return dict(kind=kind, **grid(3, 8, 1 << 24), gw=gw, filt=filt,
                    output=rng.random() < 0.25, fp32=gw and rng.random() < 0.3,
                    bins=bins)
    if kind == "fft":
        return dict(kind=kind, **grid(4, 9, 1 << 26))
    if kind == "ens":
        ns = rng.sample([16, 32, 64, 128], rng.randint(1, 3)) + [0, 0]
        r = [rng.randint(1, max(1, (1 << 22) // n ** 3 // 4)) if n else 0 for n in ns]
        r = [min(v, 40) for v in r]
        graph = rng.random() < 0.7
        return dict(kind=kind, n1=ns[0], r1=r[0], n2=ns[1], r2=r[1], n3=ns[2],
                    r3=r[2], gw=gw, filt=filt, bins=bins,
                    steps=rng.randint(1, 8), dt=rng.uniform(0.002, 0.01),
                    graph=graph, grouped=rng.random() < 0.25)
    g = grid(4, 7, 1 << 21)
    dt = rng.uniform(0.005, 0.02)
    if kind == "rk4":
        return dict(kind=kind, **g, gw=gw, filt=filt, bins=bins,
                    steps=rng.randint(2, 30), dt=dt)
    if kind == "gsl":
        return dict(kind=kind, **g, gw=gw, filt=filt, bins=bins, dt=dt)
    return dict(kind=kind, **g, gw=gw, filt=filt, bins=bins,
                steps=rng.randint(1, 4), dt=dt, t_out=rng.randint(0, 2))


# ---------------------------------------------------------------------------
# inputs (torch alone)
# ---------------------------------------------------------------------------
def _bounds(shape):
    # k_min = 0.1 along the shortest axis; the spacing is the same on all
    n0 = min(shape)
    return tuple((0.0, 2 * math.pi / 0.1 * n / n0) for n in shape)


class _Grid:
    """Wave numbers of a grid: full (kf), Nyquist-zeroed (kd) and k^2."""

    def __init__(self, shape):
        self.shape = shape
        self.N = shape[0] * shape[1] * shape[2]
        self.M = shape[0] * shape[1] * (shape[2] // 2 + 1)
        self.kf, self.kd = [], []
        for ax, (n, b) in enumerate(zip(shape, _bounds(shape))):
            m = torch.arange(n if ax < 2 else n // 2 + 1, device="cuda",
                             dtype=torch.float64)
            if ax < 2:
                m = torch.where(m > n // 2, m - n, m)
            k = m * (2 * math.pi / (b[1] - b[0]))
            view = [1, 1, 1]
            view[ax] = -1
            self.kf.append(k.reshape(view))
            self.kd.append(torch.where(2 * m.abs() == n, torch.zeros_like(k), k).reshape(view))
        self.ksq = sum(k * k for k in self.kf)

    def window(self):
        x = None
        for n, b, k in zip(self.shape, _bounds(self.shape), self.kf):
            v = k.abs() / ((n // 2) * (2 * math.pi / (b[1] - b[0])))
            x = v if x is None else torch.maximum(x, v)
        return torch.exp(-36.0 * x ** 36)


def _rfft(x):
    return torch.fft.rfftn(x, dim=(-3, -2, -1))


def _irfft(X, shape):
    return torch.fft.irfftn(X, s=shape, dim=(-3, -2, -1))


def _state_into(y, shape, gw, seed, amplitude, a0=1.0):
    """Fill the state vector y (Ntot doubles on the GPU)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    g = _Grid(shape)
    N, M = g.N, g.M
    w = ((g.ksq > 0) & (g.ksq <= (min(shape) * 0.1 / 4) ** 2)).double()
    omega = torch.sqrt(g.ksq + MASS ** 2)
    cs = (shape[0], shape[1], shape[2] // 2 + 1)

    def noise():
        return torch.randn(cs, dtype=torch.complex128, device="cuda", generator=gen)

    def field(spec, rms):
        x = _irfft(noise() * (w * spec), shape)
        return x * (rms / x.std())

    y[0:N] = (PHI0 + field(omega ** -0.5, amplitude)).reshape(-1)
    y[N:2 * N] = (DPHI0 + field(omega ** 0.5, amplitude)).reshape(-1)
    y[2 * N:3 * N] = field(1.0 / omega, 0.1 * amplitude).reshape(-1)
    y[3 * N:4 * N] = field(1.0 / omega, 0.1 * amplitude).reshape(-1)
    h = y[4 * N:4 * N + 8 * M]
    if gw:
        for b in range(4):
            z = noise() * (w * (1e-3 * amplitude * math.sqrt(N)))
            h[2 * M * b:2 * M * (b + 1)] = torch.view_as_real(z).reshape(-1)
    else:
        h.zero_()
    y[4 * N + 8 * M] = a0


def _ntot(shape):
    return 4 * shape[0] * shape[1] * shape[2] + 8 * shape[0] * shape[1] * (shape[2] // 2 + 1) + 1


def _amplitude(seed):
    return 10.0 ** (-6.0 + 2.0 * ((seed * 2654435761) % 1000) / 1000.0)


def _shape(case):
    return (case["nx"], case["ny"], case["nz"])


def _ens_sizes(case):
    return [(case["n%d" % i], case["r%d" % i]) for i in (1, 2, 3) if case["n%d" % i]]


# ---------------------------------------------------------------------------
# the library's side
# ---------------------------------------------------------------------------
class _Pointer:
    """Device memory of the library for torch.as_tensor (no copy).  The
    tensor holds this object, and this object the owner of the memory, so the
    memory lives as long as any view of it."""

    def __init__(self, ptr, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8",
                                         "data": (ptr, False), "version": 2}


def _view(ptr, n, owner):
    return torch.as_tensor(_Pointer(ptr, n, owner), device="cuda")


def _wrap(gpu, t):
    return ih.DeviceArray(gpu, t.numel(), ptr=t.data_ptr(), owned=False)


def _split(y, N):
    """phi, dphi, psi, dpsi; the tensor blocks; the scale factor."""
    return {"fields": y[:4 * N], "tensors": y[4 * N:-1], "a": y[-1:]}


def _live(y, N, gw):
    out = _split(y, N)
    if not gw:
        del out["tensors"]
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "ens":
        s["ens"] = []
        for i, (n, r) in enumerate(_ens_sizes(case)):
            e = ensemble.Ensemble(n, r, gw=case["gw"], filt=case["filt"], bins=case["bins"])
            y = _view(ih.host_lib().ih_ens_state(e.h), r * e.stride, e)
            for k in range(r):
                _state_into(y[k * e.stride:k * e.stride + e.Ntot], (n, n, n),
                            case["gw"], seed + 1000 * i + k, _amplitude(seed + k))
            s["ens"].append(e)
        torch.cuda.synchronize()
        return s
    shape = _shape(case)
    if kind in ("rhs", "fft"):
        g = ih.Gpu(shape, bounds=_bounds(shape), mass=MASS,
                   gw=case.get("gw", False), filt=case.get("filt", False),
                   bins=case.get("bins", 16), gw_fp32=case.get("fp32", False))
        s["gpu"] = g
        if kind == "rhs":
            s["f"] = torch.empty(g.Ntot, dtype=torch.float64, device="cuda")
            s["result"] = torch.zeros(g.Ntot, dtype=torch.float64, device="cuda")
            _state_into(s["f"], shape, case["gw"], seed, _amplitude(seed))
            s["df"], s["dr"] = _wrap(g, s["f"]), _wrap(g, s["result"])
            s["flags"] = (ih.IHG_FILTER if case["filt"] else 0) | (ih.IHG_OUTPUT if case["output"] else 0)
        else:
            gen = torch.Generator(device="cuda").manual_seed(seed)
            s["x"] = torch.randn(g.N, dtype=torch.float64, device="cuda", generator=gen)
            s["X"] = torch.empty(2 * g.M, dtype=torch.float64, device="cuda")
            s["back"] = torch.empty(g.N, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        return s
    method = {"rk4": ih.IH_RK4, "dopri": ih.IH_DOPRI853, "gsl": ih.IH_DOPRI89}[kind]
    sim = ih.Sim(shape, bounds=_bounds(shape), mass=MASS, gw=case["gw"],
                 filt=case["filt"], bins=case["bins"], method=method, ti=0.0,
                 tf=case["dt"] * case.get("steps", 1), dt=case["dt"],
                 rtol=RTOL, atol=ATOL, skip=10 ** 9, log_bins=kind == "dopri")
    _state_into(_view(ih.host_lib().ih_field(sim.sim), sim.Ntot, sim), shape,
                case["gw"], seed, _amplitude(seed))
    torch.cuda.synchronize()
    s["sim"], s["snap"] = sim, sim.snapshot()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rhs":
        g = s["gpu"]
        g.mk_rhs(s["df"], s["dr"], flags=s["flags"])
        out = _live(s["result"], g.N, case["gw"])
        if case["filt"]:
            out["filtered"] = s["f"][:4 * g.N]
        if case["output"]:
            out["observables"] = g.observables()
        return out
    if kind == "fft":
        g, lib = s["gpu"], ih.lib()
        ih._check(lib.ihg_fft_r2c(g.ctx, s["x"].data_ptr(), s["X"].data_ptr()))
        ih._check(lib.ihg_fft_c2r(g.ctx, s["X"].data_ptr(), s["back"].data_ptr()))
        return {"spectrum": s["X"], "back": s["back"]}
    if kind == "ens":
        ensemble.run(s["ens"], case["steps"], case["dt"], use_graph=case["graph"],
                     grouped=case["grouped"])
        out = []
        for e in s["ens"]:
            y = _view(ih.host_lib().ih_ens_state(e.h), e.nreal * e.stride, e)
            y = y.reshape(e.nreal, e.stride)
            out.append({"fields": y[:, :4 * e.N], "a": y[:, e.Ntot - 1]})
            if case["gw"]:
                out[-1]["tensors"] = y[:, 4 * e.N:e.Ntot - 1]
        return out
    sim, saves = s["sim"], []
    sim.restore(s["snap"])
    if kind == "rk4":
        sim.run_rk4(saves=saves)
    elif kind == "gsl":
        sim.run_gsl(1, saves=saves)
    else:
        n, dt = case["steps"], case["dt"]
        t_out = [dt * n * (i + 0.5) / case["t_out"] for i in range(case["t_out"])]
        sim.run_dopri853(forced=[dt] * n, saves=saves, t_out=t_out or None)
    out = _live(_view(ih.host_lib().ih_field(sim.sim), sim.Ntot, sim), sim.N, case["gw"])
    out["saves"] = [o for _, _, o in saves]
    return out


# ---------------------------------------------------------------------------
# the same in torch, 64 bits
# ---------------------------------------------------------------------------
class _Exact:
    def __init__(self, shape, gw):
        self.g = _Grid(shape)
        self.shape, self.gw = shape, gw
        self.w = None

    def filter(self, y):
        if self.w is None:
            self.w = self.g.window()
        N = self.g.N
        for b in range(4):
            x = y[b * N:(b + 1) * N].reshape(self.shape)
            y[b * N:(b + 1) * N] = _irfft(_rfft(x) * self.w, self.shape).reshape(-1)

    def rhs(self, y):
        g, shape, N, M = self.g, self.shape, self.g.N, self.g.M
        phi, dphi, psi, dpsi = (y[b * N:(b + 1) * N].reshape(shape) for b in range(4))
        a = y[-1]
        a2 = a * a
        X = _rfft(phi)
        grad = [_irfft(1j * k * X, shape) for k in g.kd]
        lap = _irfft(-g.ksq * X, shape)
        del X
        g2 = grad[0] ** 2 + grad[1] ** 2 + grad[2] ** 2
        t1 = (0.5 - psi) * dphi * dphi
        t2 = (0.5 + psi) * g2 / a2
        V = MASS ** 2 * phi * phi / 2.0
        pressure = t1 - t2 / 3.0 - V
        H = torch.sqrt((t1 + t2 + V).mean() / 3.0)
        pm = pressure.mean()
        out = torch.zeros_like(y)
        out[0:N] = dphi.reshape(-1)
        out[N:2 * N] = ((1 + 4 * psi) * lap / a2 - (3 * H - 4 * dpsi) * dphi
                        - (1 + 2 * psi) * MASS ** 2 * phi).reshape(-1)
        out[2 * N:3 * N] = dpsi.reshape(-1)
        out[3 * N:4 * N] = (0.5 * pressure + (psi - 0.5) * pm - 4 * H * dpsi).reshape(-1)
        out[-1] = a * H
        if self.gw:
            del t1, t2, V, pressure, lap, g2
            S = {}
            for i in range(3):
                for j in range(i, 3):
                    S[i, j] = S[j, i] = _rfft(grad[i] * grad[j])
            k = g.kf
            inv = torch.where(g.ksq > 0, 1.0 / g.ksq, torch.zeros_like(g.ksq))
            row = [sum(k[j] * S[i, j] for j in range(3)) for i in range(3)]
            tr = S[0, 0] + S[1, 1] + S[2, 2]
            kk = sum(k[i] * row[i] for i in range(3)) * inv
            s1, s2 = kk + tr, kk - tr

            def pair(p, q):
                o0 = S[p, p] - 2 * k[p] * inv * row[p] + 0.5 * (k[p] * k[p] * inv * s1 + s2)
                o1 = (S[p, q] - k[p] * inv * row[q] - k[q] * inv * row[p]
                      + 0.5 * k[p] * inv * k[q] * s1)
                return o0, o1

            o0, o1 = pair(0, 1)
            on_z, on_y = k[2].abs() > 1e-15, k[1].abs() > 1e-15
            for p, q, mask in ((0, 2, ~on_z & on_y), (1, 2, ~on_z & ~on_y)):
                v0, v1 = pair(p, q)
                o0, o1 = torch.where(mask, v0, o0), torch.where(mask, v1, o1)
            for o in (o0, o1):
                o[0, 0, 0] = 0
            hb = y[4 * N:-1].reshape(4, -1, 2)
            ob = out[4 * N:-1].reshape(4, -1, 2)
            fac = -(2 * pm + g.ksq / a2).reshape(-1, 1)
            for b, o in ((0, o0), (1, o1)):
                ob[b] = hb[2 + b]
                ob[2 + b] = (fac * hb[b] - 3 * H * hb[2 + b]
                             + 2 * torch.view_as_real(o).reshape(-1, 2) / a2)
        return out

    def rk4(self, y, dt):
        k1 = self.rhs(y)
        k2 = self.rhs(y + dt / 2 * k1)
        k3 = self.rhs(y + dt / 2 * k2)
        k4 = self.rhs(y + dt * k3)
        return y + dt * (k1 + 2 * k2 + 2 * k3 + k4) / 6.0

    def flow(self, y, dt):
        """The solution a step later: Gragg's modified midpoint rule with 2,
        4, 6 and 8 substeps, extrapolated in the square of the substep."""
        ns, f0, T = (2, 4, 6, 8), self.rhs(y), []
        for n in ns:
            h = dt / n
            u, v = y, y + h * f0
            for _ in range(n - 1):
                u, v = v, u + 2 * h * self.rhs(v)
            row = [0.5 * (u + v + h * self.rhs(v))]
            for j, old in enumerate(T):
                row.append(row[j] + (row[j] - old) / ((n / ns[len(T) - 1 - j]) ** 2 - 1))
            T = row
        return T[-1]


def exact(case, seed):
    kind = case["kind"]
    if kind == "ens":
        out = []
        for i, (n, r) in enumerate(_ens_sizes(case)):
            E = _Exact((n, n, n), case["gw"])
            ys = []
            for k in range(r):
                y = torch.empty(_ntot((n, n, n)), dtype=torch.float64, device="cuda")
                _state_into(y, (n, n, n), case["gw"], seed + 1000 * i + k, _amplitude(seed + k))
                for _ in range(case["steps"]):
                    if case["filt"]:
                        E.filter(y)
                    y = E.rk4(y, case["dt"])
                ys.append(y)
            y, N = torch.stack(ys), n ** 3
            out.append({"fields": y[:, :4 * N], "a": y[:, -1]})
            if case["gw"]:
                out[-1]["tensors"] = y[:, 4 * N:-1]
        return out
    shape = _shape(case)
    if kind == "fft":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        N = shape[0] * shape[1] * shape[2]
        x = torch.randn(N, dtype=torch.float64, device="cuda", generator=gen)
        return {"spectrum": torch.view_as_real(_rfft(x.reshape(shape))).reshape(-1),
                "back": x * N}
    E = _Exact(shape, case["gw"])
    N = E.g.N
    y = torch.empty(_ntot(shape), dtype=torch.float64, device="cuda")
    _state_into(y, shape, case["gw"], seed, _amplitude(seed))
    if kind == "rhs":
        if case["filt"]:
            E.filter(y)
        out = _live(E.rhs(y), N, case["gw"])
        if case["filt"]:
            out["filtered"] = y[:4 * N]
        if case["output"]:
            out["observables"] = None
        return out

    def filt():
        if case["filt"]:
            E.filter(y)

    if kind == "rk4":
        for _ in range(case["steps"]):
            filt()
            y = E.rk4(y, case["dt"])
    else:
        filt()  # the save before the first step filters the state
        for _ in range(case.get("steps", 1)):
            y = E.flow(y, case["dt"])
            if kind == "dopri":
                filt()
    filt()  # and so does the last save
    out = _live(y, N, case["gw"])
    out["saves"] = None
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without: the live state read and its slope written
# per right-hand side; per stage sum and per update every operand once;
# transforms at 2.5 N log2 N and the pointwise arithmetic as operations
# ---------------------------------------------------------------------------
def _one_rhs(shape, gw, filt, output=False):
    N = shape[0] * shape[1] * shape[2]
    M = shape[0] * shape[1] * (shape[2] // 2 + 1)
    fft = 2.5 * N * math.log2(N)
    live = 8.0 * (4 * N + (8 * M if gw else 0))
    b, f = 2 * live, (11 if gw else 5) * fft + 60.0 * N + (200.0 * M if gw else 0)
    if filt:
        b, f = b + 32.0 * N, f + 8 * fft
    if output:
        f += 4 * fft + 100.0 * N
    return live, b, f


def work(case):
    kind = case["kind"]
    if kind == "fft":
        N = case["nx"] * case["ny"] * case["nz"]
        M = case["nx"] * case["ny"] * (case["nz"] // 2 + 1)
        return {"bytes": 2.0 * (8 * N + 16 * M), "flops": 5.0 * N * math.log2(N)}
    if kind == "ens":
        b = f = 0.0
        for n, r in _ens_sizes(case):
            live, rb, rf = _one_rhs((n, n, n), case["gw"], False)
            _, fb, ff = _one_rhs((n, n, n), case["gw"], case["filt"])
            b += r * case["steps"] * (3 * rb + fb + 15 * live)
            f += r * case["steps"] * (3 * rf + ff + live)
        return {"bytes": b, "flops": f}
    shape = _shape(case)
    live, rb, rf = _one_rhs(shape, case["gw"], False)
    _, fb, ff = _one_rhs(shape, case["gw"], case["filt"])
    if kind == "rhs":
        _, b, f = _one_rhs(shape, case["gw"], case["filt"], case["output"])
        return {"bytes": b, "flops": f}
    _, ob, of = _one_rhs(shape, case["gw"], case["filt"], True)
    n = case.get("steps", 1)
    if kind == "rk4":
        return {"bytes": n * (3 * rb + fb + 15 * live) + ob,
                "flops": n * (3 * rf + ff + live) + of}
    if kind == "dopri":
        # 11 stage right-hand sides and sums (73 state vectors through
        # memory), the error sums, and the filtered one of the new state
        return {"bytes": n * (11 * rb + fb + 83 * live) + 2 * ob,
                "flops": n * (11 * rf + ff + 20 * live) + 2 * of}
    return {"bytes": 13 * rb + 100 * live + 2 * ob, "flops": 13 * rf + 25 * live + 2 * of}
