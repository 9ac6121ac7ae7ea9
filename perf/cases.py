"""The workloads that this library's speed is judged by.

Every case is one piece of work as a program that solves Gross-Pitaevskii
problems has it done through the Python binding: a context (or a batch, or the
solve service) is set up once, and a pass advances it by one output interval and
hands back what such a program then reads: the wavefunction, the energies and,
in two dimensions, the vortices. Units are those of the harmonic oscillator
(hbar = m = 1).

listed()  the cases; draw() gives more of the same ranges
prepare() inputs from a seed and the handle a program keeps
run()     one pass
work()    bytes and operations a pass cannot do without
exact()   the same results by torch.fft in 64 bits
"""
import math

import numpy as np
import torch

import gpue_amd as G

LENGTHS = [16, 32, 48, 64, 96, 128, 192, 256, 384, 512, 1024, 2048, 4096]

# the time-dependent trap and the static one that the equation cases set
EQN_T = "0.5*(x*x+y*y)*(1+0.1*sin(2*t))"
EQN_S = "0.5*(x*x+y*y)+0.3*cos(x)*sin(y)"


def listed():
    base = dict(kind="solve", nx=1, ny=1, nz=1, prec=64, real=False, omega=0.0, fields="trap", steps=100,
                every=0, upload=False, vortices=0)

    def case(name, **kw):
        return dict(base, name=name, **kw)

    return [
        # the smallest call: a ground state on a line (dimnum = 1), one output interval
        case("line_1024_ground", dim=1, nx=1024, every=100),
        # an everyday 2D ground state (no rotation) with the energy cadence of the step loop
        case("plane_256_ground", dim=2, nx=256, ny=256, every=100),
        # the rotating condensate of the benchmark: relaxation in imaginary time ...
        case("plane_512_rotating_ground", dim=2, nx=512, ny=512, omega=0.9, vortices=12),
        # ... and its dynamics, with the vortices located after every output interval
        case("plane_512_rotating_dynamics", dim=2, nx=512, ny=512, omega=0.9, vortices=12, real=True),
        # a trap that an equation string modulates in time: every step evaluates it anew
        case("plane_256_modulated_trap", dim=2, nx=256, ny=256, fields="eqn_t", real=True),
        # fields read from files (V and both components of A as tables) on an uneven grid, started from
        # an uploaded state each time
        case("plane_384x192_field_tables", dim=2, nx=384, ny=192, fields="tables", omega=0.3, real=True, upload=True),
        # a large 2D state, uploaded, relaxed and read back
        case("plane_2048_ground", dim=2, nx=2048, ny=2048, steps=200, upload=True),
        # the 3D ground state of the benchmark in both precisions
        case("box_256_ground", dim=3, nx=256, ny=256, nz=256, steps=200, every=100),
        case("box_256_ground_fp32", dim=3, nx=256, ny=256, nz=256, prec=32, steps=200),
        # a 3D condensate rotating about z, in real time, on an uneven box
        case("box_128x128x96_rotating_dynamics", dim=3, nx=128, ny=128, nz=96, omega=0.6, real=True, steps=200),
        # a parameter scan: rotating FP32 instances of mixed sizes advanced together between two
        # convergence checks
        dict(name="scan_of_16", kind="batch", count=16, largest=512, prec=32, real=False, steps=200),
        # the solve service: a burst of mixed requests from submission to results
        dict(name="service_of_10", kind="serve", count=10, largest=512, steps=200),
    ]


def _pick(rng, lo, hi):
    """A supported axis length of [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo * 0.85), math.log(hi * 1.15)))
    return min((n for n in LENGTHS if lo <= n <= hi), key=lambda n: abs(math.log(n / v)))


def draw(rng):
    kind = rng.choice(["line", "plane", "plane", "plane", "fields", "fields", "box", "box", "batch", "serve"])
    c = dict(kind="solve", nx=1, ny=1, nz=1, prec=rng.choice([64, 64, 32]), real=rng.random() < 0.5, omega=0.0,
             fields="trap", steps=rng.randrange(40, 121), every=0, upload=rng.random() < 0.3, vortices=0)
    if kind == "line":
        c.update(dim=1, nx=_pick(rng, 64, 4096), every=rng.choice([0, 50]))
    elif kind == "plane":
        c.update(dim=2, nx=_pick(rng, 64, 2048), ny=_pick(rng, 64, 2048), every=rng.choice([0, 0, 50]))
        if rng.random() < 0.6:
            c["omega"] = round(rng.uniform(0.1, 0.95), 3)
    elif kind == "fields":
        f = rng.choice(["eqn_t", "eqn_s", "tables"])
        c.update(dim=2, nx=_pick(rng, 64, 512), ny=_pick(rng, 64, 512), fields=f)
        if f == "tables":
            c["omega"] = round(rng.uniform(0.1, 0.6), 3)
        if f == "eqn_t":
            c["prec"] = 64   # the library takes time-dependent fields in 64 bits only
    elif kind == "box":
        c.update(dim=3, nx=_pick(rng, 32, 192), ny=_pick(rng, 32, 192), nz=_pick(rng, 32, 192))
        if rng.random() < 0.5:
            c["omega"] = round(rng.uniform(0.1, 0.8), 3)
    elif kind == "batch":
        return dict(kind="batch", count=rng.randrange(3, 17), largest=rng.choice([192, 256, 384, 512]),
                    prec=rng.choice([32, 32, 64]), real=rng.random() < 0.3, steps=rng.randrange(40, 161))
    else:
        return dict(kind="serve", count=rng.randrange(3, 11), largest=rng.choice([192, 256, 384]),
                    steps=rng.randrange(40, 161))
    return c


# --- problems ----------------------------------------------------------------
def _params(c):
    """Keyword arguments of the context of a "solve" case."""
    half = {1: 12.0, 2: 10.0 if max(c["nx"], c["ny"]) <= 256 else 12.0, 3: 8.0}[c["dim"]]
    dt = (5e-4 if c["dim"] == 3 else 1e-3, 1e-3 if c["fields"] == "eqn_t" else 1e-4)
    kw = dict(dimnum=c["dim"], xDim=c["nx"], yDim=c["ny"], zDim=c["nz"], xMax=half, yMax=half, zMax=half,
              g={1: 50.0, 2: 1000.0, 3: 5000.0}[c["dim"]] if c["omega"] or c["dim"] != 2 else 500.0, gpe=1,
              gdt=dt[0], dt=dt[1], precision=c["prec"])
    if c["dim"] == 3:
        kw["omegaZ"] = 2.0
    if c["omega"]:
        kw.update(omega=c["omega"], corotating=1)
    return kw


def _axes(kw):
    """Coordinates and wave numbers per axis, and the spacings."""
    x, k, d = [], [], []
    for n, L in zip((kw["xDim"], kw["yDim"], kw["zDim"])[: kw["dimnum"]], (kw["xMax"], kw["yMax"], kw["zMax"])):
        i = torch.arange(n, dtype=torch.float64)
        h = L / (n // 2)
        x.append(torch.cat([-L + i[: n // 2] * h, i[: n // 2] * h]))
        k.append(torch.where(i < n // 2, i, i - n) * (math.pi / L))
        d.append(h)
    return x, k, d


def _along(v, a, dim):
    """A vector of axis a (0 = x) shaped to broadcast over a (z, y, x) field."""
    return v.reshape([-1 if dim - 1 - j == a else 1 for j in range(dim)])


def _start(kw, seed, vortices=0):
    """psi0: a Gaussian cloud with 1 % noise and, in 2D, vortices at random places of its core; normalised."""
    x, _, d = _axes(kw)
    dim = kw["dimnum"]
    g = torch.Generator().manual_seed(int(seed))
    psi = None
    for a in range(dim):
        e = _along(torch.exp(-x[a] ** 2 / (8.0 if dim < 3 else 4.0)), a, dim)
        psi = e if psi is None else psi * e
    psi = psi * (1 + 0.01 * (2 * torch.rand(psi.shape, generator=g, dtype=torch.float64) - 1))
    if vortices:
        z = torch.complex(_along(x[0], 0, 2).expand(psi.shape).contiguous(), _along(x[1], 1, 2).expand(psi.shape).contiguous())
        psi = psi.to(torch.complex128)
        for px, py in (7.0 * torch.rand((vortices, 2), generator=g, dtype=torch.float64) - 3.5).tolist():
            w = z - complex(px, py)
            psi = psi * (w / torch.sqrt(w.abs() ** 2 + 0.25))
    psi = psi.to(torch.complex128)
    return psi / torch.sqrt((psi.abs() ** 2).sum() * math.prod(d))


def _tables(c, kw):
    """V and A of the field-table cases: an uneven trap and a gauge field that fades with the radius."""
    x, _, _ = _axes(kw)
    X, Y = _along(x[0], 0, 2), _along(x[1], 1, 2)
    fade = torch.exp(-(X ** 2 + Y ** 2) / 50.0)
    V = 0.5 * (X ** 2 + 1.3 * Y ** 2) + 0.2 * torch.sin(X)
    return V, -c["omega"] * Y * fade, c["omega"] * X * fade


def _scan(c, seed):
    """(parameters, seed of psi0) of the instances of a batch."""
    rng = np.random.default_rng(seed)
    sizes = [n for n in (128, 192, 256, 384, 512) if n <= c["largest"]]
    got = []
    for i in range(c["count"]):
        n = sizes[(i * 7 + 3) % len(sizes)]
        half = 10.0 if n <= 256 else 12.0
        got.append((dict(dimnum=2, xDim=n, yDim=n, zDim=1, xMax=half, yMax=half, zMax=half,
                         g=float(rng.uniform(100, 2000)), gpe=1, omega=float(rng.uniform(0, 0.95)), corotating=1,
                         omegaY=float(rng.uniform(0.8, 1.2)), gdt=1e-3, dt=1e-4, precision=c["prec"]),
                    int(seed) * 1000 + i))
    return got


def _requests(c, seed):
    """(parameters, request options) of a burst: three 2D ground states to one 3D quench, half of them FP32."""
    rng = np.random.default_rng(seed)
    sizes = [n for n in (128, 192, 256, 384, 512) if n <= c["largest"]]
    got = []
    for i in range(c["count"]):
        prec = 64 if i % 2 else 32
        opt = dict(seed=int(seed) * 1000 + i, check_every=100, energy_tol=0.0)
        if i % 4 < 3:
            n = sizes[(i * 7 + 2) % len(sizes)]
            kw = dict(dimnum=2, xDim=n, yDim=n, zDim=1, xMax=10.0, yMax=10.0, zMax=10.0)
            opt.update(max_imag_steps=c["steps"])
        else:
            n = 64 if i % 8 < 4 else 96
            kw = dict(dimnum=3, xDim=n, yDim=n, zDim=n, xMax=8.0, yMax=8.0, zMax=8.0, omegaZ=2.0)
            opt.update(max_imag_steps=c["steps"] // 2, real_steps=c["steps"], quench_factor=float(rng.uniform(0.5, 2.0)))
        got.append((dict(kw, g=float(rng.uniform(100, 1000)), gpe=1, gdt=1e-3 if kw["dimnum"] == 2 else 5e-4, dt=1e-4,
                         precision=prec), opt))
    return got


# --- what a program keeps, and one pass ----------------------------------------
def prepare(case, seed):
    if case["kind"] == "batch":
        ctxs = []
        for kw, s in _scan(case, seed):
            c = G.Context(**kw)
            c.upload(_start(kw, s, vortices=4).numpy())
            ctxs.append(c)
        return dict(case=case, ctxs=ctxs, batch=G.Batch(ctxs))
    if case["kind"] == "serve":
        reqs = _requests(case, seed)
        total = sum(kw["xDim"] * kw["yDim"] * kw["zDim"] * 32 for kw, _ in reqs)
        return dict(case=case, reqs=[(G.make_params(**kw), opt) for kw, opt in reqs],
                    shapes=[(kw["zDim"], kw["yDim"], kw["xDim"])[3 - kw["dimnum"]:] for kw, _ in reqs],
                    server=G.Server(budget_bytes=4.0 * total + 1e9, max_slots=8))
    kw = _params(case)
    ctx = G.Context(**kw)
    if case["fields"] == "tables":
        for which, f in zip((G.FIELD_V, G.FIELD_AX, G.FIELD_AY), _tables(case, kw)):
            ctx.set_field(which, f.numpy())
    elif case["fields"] != "trap":
        ctx.set_field_eqn(G.FIELD_V, EQN_T if case["fields"] == "eqn_t" else EQN_S)
    psi0 = _start(kw, seed, case["vortices"]).numpy()
    ctx.upload(psi0)
    return dict(case=case, ctx=ctx, psi0=psi0, step=0)


def _held(a, prec):
    """Results in the precision that the solution is held in (FP32 contexts hand their values out as doubles)."""
    return torch.from_numpy(a).to(torch.complex64 if np.iscomplexobj(a) else torch.float32) if prec == 32 else a


def run(state):
    c = state["case"]
    if c["kind"] == "batch":
        b = state["batch"]
        b.evolve(c["steps"], 1 if c["real"] else 0)
        e, m = b.energy()
        return dict(energy=_held(e, c["prec"]), mu=_held(m, c["prec"]),
                    psi=[_held(x.download(), c["prec"]) for x in state["ctxs"]])
    if c["kind"] == "serve":
        sv = state["server"]
        out = [np.empty(s, np.complex128) for s in state["shapes"]]
        for i, (p, opt) in enumerate(state["reqs"]):
            sv.submit(i, p, psi_out=out[i], **opt)
        sv.drain(60.0)
        res = sorted(sv.poll(), key=lambda r: r["id"])
        prec = [p.precision for p, _ in state["reqs"]]
        return dict(psi=[_held(o, q) for o, q in zip(out, prec)],
                    energy=[_held(np.array([r["energy"], r["mu"]]), q) for r, q in zip(res, prec)],
                    steps=[[r["status"], r["imag_steps"], r["real_steps"]] for r in res])
    ctx, gstate = state["ctx"], 1 if c["real"] else 0
    if c["upload"]:
        ctx.upload(state["psi0"])
        state["step"] = 0
    _, energies = ctx.evolve(c["steps"], gstate, first_step=state["step"], energy_every=c["every"])
    state["step"] += c["steps"]
    got = {}
    if c["every"]:
        got["energy"] = _held(energies, c["prec"])
    else:
        got["energy"] = _held(np.array(ctx.energy()), c["prec"])
    if c["vortices"] and c["real"]:
        got["marker"], got["found"] = ctx.vortex_marker(4.0)
    got["psi"] = _held(ctx.download(), c["prec"])
    return got


# --- the least work of a pass ----------------------------------------------------
def _step_work(kw, steps, gauge):
    """Every step reads and writes the state once; transforms at 5 n log2 n, pointwise operators at 40 a point."""
    n = kw["xDim"] * kw["yDim"] * kw["zDim"]
    size = 8 if kw["precision"] == 32 else 16
    lg = sum(math.log2(d) for d in (kw["xDim"], kw["yDim"], kw["zDim"]) if d > 1)
    lg_gauge = sum(math.log2(d) for d in (kw["xDim"], kw["yDim"])) if gauge else 0.0
    return steps * 2.0 * size * n, steps * n * (10.0 * (lg + lg_gauge) + 40.0)


def work(case):
    if case["kind"] == "batch":
        w = [_step_work(kw, case["steps"], True) for kw, _ in _scan(case, 1)]
    elif case["kind"] == "serve":
        w = [_step_work(kw, o["max_imag_steps"] + o.get("real_steps", 0), False) for kw, o in _requests(case, 1)]
    else:
        w = [_step_work(_params(case), case["steps"], case["omega"] and case["dim"] > 1)]
    return dict(bytes=sum(b for b, _ in w), flops=sum(f for _, f in w))


# --- the same in 64 bits ---------------------------------------------------------
class _Solver:
    """The split-operator step and the energy by torch.fft in complex128."""

    def __init__(self, kw, psi, V=None, A=None):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dim, self.g, self.dt = kw["dimnum"], kw["g"], (kw["gdt"], kw["dt"])
        x, k, self.d = _axes(kw)
        w = (1.0, kw.get("omegaY", 1.0), kw.get("omegaZ", 1.0))
        om = kw.get("omega", 0.0)
        self.gauge = bool(kw.get("corotating")) and self.dim > 1
        ax = [_along(v, a, self.dim).to(self.dev) for a, v in enumerate(x)]
        self.k = [_along(v, a, self.dim).to(self.dev) for a, v in enumerate(k)]
        self.K = sum(0.5 * v * v for v in self.k)
        self.x = ax
        if A is None:   # the frame rotating about z
            A = [-om * ax[1] if self.dim > 1 else 0.0 * ax[0], om * w[1] * ax[0]]
        self.A = [a.to(self.dev) for a in A]
        if V is None:
            V = sum(0.5 * (w[a] * v) ** 2 for a, v in enumerate(ax)) + 0.5 * sum(a * a for a in self.A)
        self.V = V if callable(V) else V.to(self.dev)
        self.psi = psi.to(self.dev)

    def v_at(self, t):
        return self.V(self.x, t) if callable(self.V) else self.V

    def step(self, i, real):
        dt = self.dt[real]
        f = -1j * dt if real else -dt
        V, p, dims = self.v_at(dt * i), self.psi, tuple(range(self.dim))
        p = p * torch.exp(0.5 * f * (V + self.g * p.abs() ** 2))
        p = torch.fft.ifftn(torch.exp(f * self.K) * torch.fft.fftn(p, dim=dims), dim=dims)
        p = p * torch.exp(0.5 * f * (V + self.g * p.abs() ** 2))
        if self.gauge:
            for a in ((0, 1) if i % 2 else (1, 0)):
                ax = self.dim - 1 - a
                p = torch.fft.ifft(torch.exp(f * self.A[a] * self.k[a]) * torch.fft.fft(p, dim=ax), dim=ax)
        if not real:
            p = p / torch.sqrt((p.abs() ** 2).sum() * math.prod(self.d))
        self.psi = p

    def energy(self, t=0.0):
        p, dims = self.psi, tuple(range(self.dim))
        rho, dV = p.abs() ** 2, math.prod(self.d)
        e = (self.K * torch.fft.fftn(p, dim=dims).abs() ** 2).sum() / p.numel() + (self.v_at(t) * rho).sum()
        if self.gauge:   # forward differences on the flat array; past its end the neighbour counts as 2 psi
            flat, s = p.reshape(-1), 1
            grad = torch.zeros_like(p)
            for a in range(2):
                nxt = torch.cat([flat[s:], 2 * flat[-s:]])
                grad = grad + self.A[a] * ((nxt - flat) / self.d[a]).reshape(p.shape)
                s *= p.shape[self.dim - 1 - a]
            e = e + (p.conj() * 1j * grad).real.sum()
        four = self.g * (rho * rho).sum()
        return [float((e + 0.5 * four) * dV), float((e + four) * dV)]

    def evolve(self, steps, real, every=0, first=0):
        got = []
        for i in range(first, first + steps):
            self.step(i, real)
            if every and i % every == 0:
                got.append(self.energy(self.dt[real] * i)[0])
        return np.array(got)

    def out(self):
        return self.psi.cpu().numpy()


def _service_start(kw, seed):
    """psi0 of the solve service: exp(-r^2/2)(1 + 0.01 u), u from the splitmix64 finaliser of seed and index."""
    x, _, d = _axes(kw)
    dim = kw["dimnum"]
    r2 = sum(_along(v, a, dim) ** 2 for a, v in enumerate(x))
    m64 = (1 << 64) - 1
    with np.errstate(over="ignore"):
        z = np.arange(r2.numel(), dtype=np.uint64) * np.uint64(2)
        z += np.uint64((seed * 0x9E3779B97F4A7C15 + 0x632BE59BD9B4E019) & m64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = torch.from_numpy((z >> np.uint64(11)).astype(np.float64) * (2.0 / 9007199254740992.0) - 1.0)
    psi = torch.exp(-r2 / 2) * (1 + 0.01 * u.reshape(r2.shape))
    return (psi / torch.sqrt((psi ** 2).sum() * math.prod(d))).to(torch.complex128)


def exact(case, seed):
    if case["kind"] == "batch":
        e, m, psi = [], [], []
        for kw, s in _scan(case, seed):
            sol = _Solver(kw, _start(kw, s, vortices=4))
            sol.evolve(case["steps"], int(case["real"]))
            a, b = sol.energy()
            e.append(a)
            m.append(b)
            psi.append(sol.out())
        return dict(energy=np.array(e), mu=np.array(m), psi=psi)
    if case["kind"] == "serve":
        psi, energy = [], []
        for kw, o in _requests(case, seed):
            sol = _Solver(kw, _service_start(kw, o["seed"]))
            sol.evolve(o["max_imag_steps"], 0)
            if o.get("real_steps"):
                sol.g *= o["quench_factor"]
                sol.evolve(o["real_steps"], 1)
            psi.append(sol.out())
            energy.append(np.array(sol.energy()))
        return dict(psi=psi, energy=energy, steps=None)
    kw = _params(case)
    V = A = None
    if case["fields"] == "tables":
        V, *A = _tables(case, kw)
    elif case["fields"] == "eqn_s":
        def V(x, t):
            return 0.5 * (x[0] ** 2 + x[1] ** 2) + 0.3 * torch.cos(x[0]) * torch.sin(x[1])
    elif case["fields"] == "eqn_t":
        def V(x, t):
            return 0.5 * (x[0] ** 2 + x[1] ** 2) * (1 + 0.1 * math.sin(2 * t))
    sol = _Solver(kw, _start(kw, seed, case["vortices"]), V, A)
    real = int(case["real"])
    cadence = sol.evolve(case["steps"], real, case["every"])
    last = np.array(sol.energy(sol.dt[real] * (case["steps"] - 1)))
    got = dict(energy=cadence if case["every"] else last, psi=sol.out())
    if case["vortices"] and case["real"]:
        got.update(marker=None, found=None)
    return got
