"""Performance cases: the modeling and gradient calls a user of seiscl_amd
makes, through its public entry points.

Each case is a whole user-level call on a model that already lives on the GPU:
a forward shot (``Model.forward``), a misfit gradient (``Model.gradient`` +
``grad_read``, or ``autograd.seismic`` + ``backward``), or a set of modeling
requests (``serving.serve_batched``, which builds the models itself).

Grids, FD orders, absorbing widths and options are those of the benchmark
workloads (seiscl_amd/workloads.py), of the front end's defaults and of the
tests, with shorter records so that a pass stays short: a time step costs the
same at any step of a shot.  Ricker sources start at most a third of the record
before their peak, so that short records carry waves as well.

``exact`` integrates the same discrete equations with torch in float64 (or
returns what the same formulas give for the gradients); it uses nothing of
this repository.
"""
import math

import numpy as np
import torch

from seiscl_amd import Context, Model
from seiscl_amd.autograd import Propagator, seismic
from seiscl_amd.serving import make_requests, serve_batched

# Holberg coefficients (maximum relative error 0.1 %), FD order -> weights.
HOLBERG = {
    2: (1.0010,),
    4: (1.1382, -0.046414),
    6: (1.1965, -0.078804, 0.0081781),
    8: (1.2257, -0.099537, 0.018063, -0.0026274),
    10: (1.2415, -0.11231, 0.026191, -0.0064682, 0.001191),
    12: (1.2508, -0.12034, 0.032131, -0.010142, 0.0029857, -0.00066667),
}
# CPML and taper constants of the front end's defaults
VPPML, NPOWER, FPML, KMAX, ABPC = 3500.0, 2.0, 15.0, 2.0, 6.0
FL = {1: (15.0,), 2: (5.0, 25.0)}   # relaxation frequencies (Hz)
TAU = 0.04                           # attenuation level, Q about 50
VMIN, VMAX = 1800.0, 4300.0


def _case(kind, **kw):
    c = dict(kind=kind, ND=2, NZ=100, NY=1, NX=100, NT=200, FD=8, L=0, freesurf=0, FP16=0,
             abs_type=1, nab=16, seisout=1, src=100, nshots=1)
    c.update(kw)
    return c


def listed():
    return [
        # The smallest call: a test-sized 2D shot with the front end's default
        # constants (FD order 8, pressure records); launches and latency.
        _case("forward", name="fwd2d_small", NZ=100, NX=100, NT=500, FD=8, seisout=2),
        # The plain 2D elastic benchmark shot: 200 x 400, FD order 4, a
        # vertical force, velocity records.
        _case("forward", name="fwd2d_elastic", NZ=200, NX=400, NT=1500, FD=4, nab=20, src=2),
        # Land-style 2D modeling: attenuation, free surface, odd sizes, every
        # output.
        _case("forward", name="fwd2d_visco_surface", NZ=433, NX=1217, NT=1000, FD=6, L=1,
              freesurf=1, seisout=4),
        # Marine-style 2D acoustic modeling at the upper end of the serving
        # sizes.
        _case("forward", name="fwd2d_acoustic", ND=22, NZ=600, NX=1500, NT=1200, FD=8, seisout=2,
              src=3),
        # Serving: eight 2D requests of mixed size, order and physics, built,
        # stepped together and read back.
        _case("serve", name="serve2d", nshots=8, NZ=600, NX=1500, NT=2000),
        # A 2D elastic FWI gradient through torch.autograd on device tensors:
        # 300 x 800, FD order 8, two shots, forward and backward.
        _case("autograd", name="grad2d_elastic", NZ=300, NX=800, NT=1000, FD=8, nshots=2),
        # A 2D viscoelastic gradient with a free surface (odd sizes).
        _case("gradient", name="grad2d_visco", NZ=211, NX=397, NT=1000, FD=4, L=2, freesurf=1),
        # 3D elastic modeling on a ragged grid at the default FD order.
        _case("forward", name="fwd3d_elastic_odd", ND=3, NZ=161, NY=123, NX=147, NT=300, FD=8,
              nab=12),
        # The headline 3D viscoelastic workload: 256^3, L = 2, free surface.
        _case("forward", name="fwd3d_visco", ND=3, NZ=256, NY=256, NX=256, NT=300, FD=4, L=2,
              freesurf=1),
        # The same physics with half-precision storage of the wavefields.
        _case("forward", name="fwd3d_visco_half", ND=3, NZ=224, NY=192, NX=208, NT=300, FD=4, L=2,
              freesurf=1, FP16=2),
        # A 3D elastic gradient (boundary saving and backpropagation).
        _case("gradient", name="grad3d_elastic", ND=3, NZ=120, NY=128, NX=136, NT=250, FD=4),
        # The 3D viscoelastic gradient (checkpoints and recomputation) with
        # half-precision storage, as the large FWI batch runs it.
        _case("gradient", name="grad3d_visco_half", ND=3, NZ=150, NY=130, NX=144, NT=200, FD=4,
              L=2, freesurf=1, FP16=2, nab=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# Upper bounds on the cell-steps (cells x steps x shots) of drawn cases.
_CAP = {("forward", 2): 8e8, ("forward", 3): 1e9, ("autograd", 2): 4e8,
        ("gradient", 2): 8e7, ("gradient", 3): 4e8}


def draw(rng):
    kind = rng.choice(["forward2", "forward2", "acoustic", "forward3", "forward3", "serve",
                       "autograd", "gradient2", "gradient3"])
    if kind == "serve":
        return _case("serve", nshots=rng.randint(3, 8), NZ=_log_int(rng, 120, 600),
                     NX=_log_int(rng, 240, 1500), NT=rng.randint(500, 2000))
    fd = rng.choice([4, 4, 8, 8, 2, 6, 10, 12])
    nab = rng.randint(8, 20)
    lo = 2 * nab + fd + 10
    if kind in ("forward3", "gradient3"):
        c = _case("forward" if kind == "forward3" else "gradient", ND=3, FD=fd, nab=nab,
                  NZ=_log_int(rng, lo, 256), NY=_log_int(rng, lo, 200),
                  NX=_log_int(rng, lo, 200), NT=rng.randint(40, 300),
                  L=rng.choice([0, 0, 1, 2]), seisout=rng.choice([1, 2]))
        if kind == "forward3":
            c.update(freesurf=rng.randint(0, 1), FP16=rng.choice([0, 0, 0, 2, 64]))
        elif c["L"]:
            c.update(freesurf=rng.randint(0, 1), FP16=rng.choice([0, 2]))
    else:
        c = _case("gradient" if kind == "gradient2" else
                  "autograd" if kind == "autograd" else "forward",
                  ND=22 if kind == "acoustic" else 2, FD=fd, nab=nab,
                  NZ=_log_int(rng, lo, 600), NX=_log_int(rng, lo, 1500),
                  NT=_log_int(rng, 100, 1500))
        if kind == "acoustic":
            c.update(seisout=rng.choice([1, 2, 4]), src=3, abs_type=rng.choice([1, 1, 1, 2]))
        elif kind == "forward2":
            c.update(seisout=rng.choice([1, 2, 4]), src=rng.choice([100, 2]),
                     L=rng.choice([0, 0, 1, 2]), freesurf=rng.randint(0, 1),
                     abs_type=rng.choice([1, 1, 1, 2]), FP16=rng.choice([0, 0, 0, 0, 2, 64]))
        elif kind == "autograd":
            c.update(nshots=rng.randint(1, 3))
        else:
            c.update(L=rng.choice([1, 2]), freesurf=rng.randint(0, 1))
    cap = _CAP[(c["kind"], 3 if c["ND"] == 3 else 2)]
    c["NT"] = max(40, min(c["NT"], int(cap / (_cells(c) * c["nshots"]))))
    return c


def _cells(c):
    return c["NZ"] * c["NY"] * c["NX"]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _shape(c):
    return (c["NZ"], c["NY"], c["NX"]) if c["ND"] == 3 else (c["NZ"], c["NX"])


def _ricker(f0, NT, dt):
    t = np.arange(NT) * dt - min(1.5 / f0, NT * dt / 3)
    a = (math.pi * f0 * t) ** 2
    return ((1 - 2 * a) * np.exp(-a)).astype(np.float32)


def _model(c, rng, start=False):
    """Layered vp 1800-4300 m/s with smooth 3 % perturbations, vs = vp/1.8,
    rho 1800-2600; start: without the perturbations."""
    shape = _shape(c)
    nz = shape[0]
    cuts = np.sort(rng.integers(1, nz, size=5))
    v1 = np.linspace(VMIN * 1.03, VMAX / 1.04, 6)[np.searchsorted(cuts, np.arange(nz), "right")]
    coarse = tuple(max(2, n // 16) for n in shape)
    low = torch.from_numpy(rng.standard_normal(coarse).astype(np.float32))
    up = torch.nn.functional.interpolate(
        low[None, None], size=shape, align_corners=True,
        mode="trilinear" if len(shape) == 3 else "bilinear")[0, 0].clamp_(-3, 3)
    amp = 0.0 if start else 0.01
    vp = torch.from_numpy(v1.astype(np.float32)).reshape((nz,) + (1,) * (len(shape) - 1))
    vp = vp * (1 + amp * up)
    p = dict(vp=vp, rho=1800 + (800 / 2700) * (vp - 1800))
    if c["ND"] != 22:
        p["vs"] = vp / 1.8
    if c["L"]:
        p["taup"] = torch.full(shape, TAU)
        p["taus"] = torch.full(shape, TAU)
    return {k: np.ascontiguousarray(v.numpy()) for k, v in p.items()}


def _inputs(c, seed):
    """(constants, parameters, shots, observed data or None)."""
    rng = np.random.default_rng([seed, 7])
    three = c["ND"] == 3
    dh, dt = 10.0, 8e-4 if three else 1e-3
    NT, nab = c["NT"], c["nab"]
    f0 = float(rng.uniform(10.0, 20.0))
    csts = dict(N=np.array(_shape(c)), ND=c["ND"], dh=dh, dt=dt, NT=NT, FDORDER=c["FD"],
                MAXRELERROR=1, abs_type=c["abs_type"], nab=nab, freesurf=c["freesurf"],
                L=c["L"], f0=f0, seisout=c["seisout"], FP16=c["FP16"])
    if c["L"]:
        csts["FL"] = np.array(FL[c["L"]])
    params = _model(c, rng)
    zs = (2 if c["freesurf"] else nab + 3) * dh
    gx = np.arange(nab, c["NX"] - nab, 3 if three else 2) * dh
    gy = np.zeros(1)
    if three:
        gy = np.arange(nab, c["NY"] - nab, 3) * dh
    gx, gy = (a.ravel() for a in np.meshgrid(gx, gy, indexing="ij"))
    o = 0 * gx
    rec = np.stack([gx, gy, o + zs, o, np.arange(gx.size) + 1.0, o, o, o])
    src = _ricker(f0, NT, dt)[:, None] * np.float32(1 + rng.random())
    shots, data = [], []
    for k in range(c["nshots"]):
        x = (nab + (c["NX"] - 2 * nab) * (k + 0.3 + 0.4 * rng.random()) / c["nshots"]) // 1
        y = c["NY"] // 2 if three else 0
        pos = np.array([[x * dh], [y * dh], [zs + 2 * dh], [float(k)], [float(c["src"])]])
        shots.append((pos, src, rec))
    if c["kind"] in ("gradient", "autograd"):
        # observed data: white traces smoothed in time, of the records' order
        # of magnitude (a particle velocity of dt f / (rho dh), a pressure
        # of dt f after the source's first steps)
        nout = 1 if c["seisout"] == 2 else 3 if three else 2
        size = 0.03 * dt * (1.0 if c["seisout"] == 2 else 1 / (2000.0 * 3000.0))
        for _ in shots:
            w = rng.standard_normal((nout, NT + 16, gx.size)).astype(np.float32)
            w = np.cumsum(w, axis=1)
            data.append([np.ascontiguousarray((w[q, 16:] - w[q, :-16]) * np.float32(size))
                         for q in range(nout)])
    return csts, params, shots, data


def _requests(c, seed):
    """The serving case's requests as single forward cases; their sizes follow
    from the case, their models and shots from the seed."""
    rng = np.random.default_rng([c["NZ"], c["NX"], c["NT"]])
    jobs = []
    for k in range(c["nshots"]):
        acoustic = bool(k % 2)
        jobs.append((_case("forward", ND=22 if acoustic else 2, seisout=2 if acoustic else 1,
                           src=3 if acoustic else 100, FD=(4, 8)[(k // 2) % 2],
                           NZ=max(100, int(c["NZ"] * rng.uniform(0.2, 1.0))),
                           NX=max(200, int(c["NX"] * rng.uniform(0.2, 1.0))),
                           NT=int(c["NT"] * rng.uniform(0.5, 1.0))), seed * 64 + k))
    return jobs


# ---------------------------------------------------------------------------
# The calls
# ---------------------------------------------------------------------------
def prepare(case, seed):
    ctx = Context(0)
    if case["kind"] == "serve":
        work = []
        for c, s in _requests(case, seed):
            csts, params, shots, _ = _inputs(c, s)
            work.append((csts, params, shots[0]))
        return dict(case=case, ctx=ctx, work=work)
    csts, params, shots, data = _inputs(case, seed)
    if case["kind"] == "autograd":
        prop = Propagator(ctx, params, **csts)
        names = ("vp", "vs", "rho")
        par = [torch.from_numpy(params[n]).cuda().requires_grad_() for n in names]
        obs = [torch.from_numpy(d).cuda() for shot in data for d in shot]
        return dict(case=case, ctx=ctx, prop=prop, par=par, shots=shots, obs=obs)
    return dict(case=case, ctx=ctx, model=Model(ctx, params, **csts), shots=shots, data=data)


def run(state):
    kind = state["case"]["kind"]
    if kind == "serve":
        reqs = serve_batched(state["ctx"], make_requests(state["work"]))
        return [r.out for r in reqs]
    if kind == "autograd":
        for p in state["par"]:
            p.grad = None
        outs = seismic(state["prop"], state["shots"], *state["par"])
        loss = sum(0.5 * ((o - d) ** 2).sum() for o, d in zip(outs, state["obs"]))
        loss.backward()
        return dict(out=[o.detach() for o in outs], grad=[p.grad for p in state["par"]])
    m = state["model"]
    if kind == "forward":
        return m.forward(*state["shots"][0])
    m.grad_zero()
    out, _ = m.gradient(*state["shots"][0], din=state["data"][0])
    return dict(out=out, grad=m.grad_read())


# ---------------------------------------------------------------------------
# Work and tolerances
# ---------------------------------------------------------------------------
def work(case):
    """Per time step every state array (wavefields, memory variables) is read
    and written once and every coefficient read once; gradients add the
    adjoint state, the forward state each adjoint step needs and the double
    accumulators.  CPML strips are left out.  Seismograms are written once."""
    if case["kind"] == "serve":
        w = [work(c) for c, _ in _requests(case, 0)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    c, L, H, n3 = case, case["L"], case["FD"] // 2, case["ND"] == 3
    el = {0: 4, 2: 2, 64: 8}[c["FP16"]]     # bytes of a stored wavefield value
    co = 8 if c["FP16"] == 64 else 4        # bytes of a coefficient
    if c["ND"] == 22:
        nf, nm, nc, nd = 3, 0, 3, 4
    elif n3:
        nf, nm, nc, nd = 9, 6 * L, 13 if L else 8, 18
    else:
        nf, nm, nc, nd = 5, 3 * L, 8 if L else 5, 8
    fwd = 2 * (nf + nm) * el + nc * co
    flops = nd * 3 * H + 4 * nf + 12 * nm
    adj = 0
    if c["kind"] != "forward":
        acc = 5 if L else 3
        if L:       # the history written and read, adjoint state, moduli
            adj = 2 * nf * el + 2 * (nf + nm) * 4 + (nc + 2) * co + 2 * 8 * acc
        else:       # the forward state run backwards beside the adjoint one
            adj = 4 * nf * 4 + nc * co + 2 * 8 * acc
        flops = 3 * flops + 60
    nout = {1: 3 if n3 else 2, 2: 1, 4: 3 if c["ND"] == 22 else 6}[c["seisout"]]
    nrec = len(range(c["nab"], c["NX"] - c["nab"], 3 if n3 else 2))
    if n3:
        nrec *= len(range(c["nab"], c["NY"] - c["nab"], 3))
    steps = c["NT"] * c["nshots"]
    seis = 4 * nout * nrec * steps * (1 if c["kind"] == "forward" else 3)
    return dict(bytes=float(_cells(c) * steps * (fwd + adj) + seis),
                flops=float(_cells(c) * steps * flops))


def tolerance(case):
    # Measured against exact() over the listed and some drawn cases, and stated
    # at about four times what was seen: 32-bit sums over hundreds of steps
    # (up to 1.5e-6), wavefields stored in 16 bits (up to 1.4e-2), and the
    # rounding of the 32-bit records of runs in 64 bits (1e-7).
    if case["FP16"] == 2:
        return {"rel": 0.03, "max": 0.99}
    if case["FP16"] == 64:
        return {"rel": 5e-7, "max": 2e-5}
    return {"rel": 6e-6, "max": 6e-4}


# ---------------------------------------------------------------------------
# The same discrete equations in float64
# ---------------------------------------------------------------------------
class _Exact:
    """One shot in float64 with torch.  Fields are [X, (Y,) Z] tensors with H
    halo cells on every side; derivatives come back on the interior."""

    def __init__(self, c, csts, params):
        self.c, self.H = c, c["FD"] // 2
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.three = c["ND"] == 3
        self.ax = {"x": 0, "y": 1, "z": 2} if self.three else {"x": 0, "z": 1}
        self.n = tuple(_shape(c)[::-1])
        self.hc = [float(np.float32(h)) for h in HOLBERG[c["FD"]]]
        self.dt, self.dh = float(np.float32(csts["dt"])), float(csts["dh"])
        self.L, self.fs, self.nab = c["L"], c["freesurf"], c["nab"]
        self.p = {k: self._t(v.T) for k, v in params.items()}
        self._moduli(float(np.float32(csts["f0"])))
        self._absorb()

    def _t(self, a):
        return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to(self.dev)

    # ---- parameters -------------------------------------------------------
    def _at(self, a, axis, i):
        return a.narrow(axis, i % a.shape[axis], 1)

    def _avg2(self, a, axis):
        return torch.cat([0.5 * (a.narrow(axis, 0, a.shape[axis] - 1) +
                                 a.narrow(axis, 1, a.shape[axis] - 1)),
                          self._at(a, axis, -1)], axis)

    def _avg4(self, a, ax1, ax2, harmonic):
        """Average over the four cells around an edge; the last plane of the
        first axis is copied, that of the second axis stays zero."""
        n1, n2 = a.shape[ax1] - 1, a.shape[ax2] - 1
        q = [a.narrow(ax1, i, n1).narrow(ax2, j, n2) for i in (0, 1) for j in (0, 1)]
        out = a.new_zeros(a.shape)
        out.narrow(ax1, 0, n1).narrow(ax2, 0, n2).copy_(
            4 / sum(1 / v for v in q) if harmonic else 0.25 * sum(q))
        self._at(out, ax1, -1).copy_(self._at(a, ax1, -1))
        return out

    def _moduli(self, f0):
        p, k, ax = self.p, self.dt / self.dh, self.ax
        self.rho = p["rho"]
        b = k / self.rho
        self.rv = {"v" + s: self._avg2(b, ax[s]) for s in ax}
        self.M0 = self.M = p["vp"] ** 2 * self.rho * k
        if self.c["ND"] == 22:
            return
        self.mu0 = self.mu = p["vs"] ** 2 * self.rho * k
        pairs = [("x", "z"), ("x", "y"), ("y", "z")] if self.three else [("x", "z")]
        if not self.L:
            self.ms = {u + v: self._avg4(self.mu, ax[u], ax[v], True) for u, v in pairs}
            return
        w0 = 2 * math.pi * f0
        fl = [float(np.float32(f)) for f in FL[self.L]]
        self.s0 = sum((w0 / (2 * math.pi * f)) ** 2 / (1 + (w0 / (2 * math.pi * f)) ** 2)
                      for f in fl)
        eta = [2 * math.pi * f * self.dt for f in fl]
        self.rl = [(1 / (1 + e / 2), 1 - e / 2, e) for e in eta]
        tp, ts = p["taup"], p["taus"]
        self.M = self.M0 / (1 + self.s0 * tp)
        self.mu = self.mu0 / (1 + self.s0 * ts)
        self.g, self.e = self.M * (1 + self.L * tp), self.M * tp / self.dt
        self.f, self.d = 2 * self.mu * (1 + self.L * ts), 2 * self.mu * ts / self.dt
        self.ms, self.ds = {}, {}
        for u, v in pairs:
            m = self._avg4(self.mu, ax[u], ax[v], True)
            t = self._avg4(ts, ax[u], ax[v], False)
            self.ms[u + v], self.ds[u + v] = m * (1 + self.L * t), m * t / self.dt

    def _absorb(self):
        nab, dt, dh = self.nab, self.dt, self.dh
        self.pml, self.taper = {}, {}
        if self.c["abs_type"] == 2:
            amp = 1 - ABPC / 100
            a2 = -math.log(amp) / (nab - 1) ** 2
            t = [math.exp(-a2 * (nab - i) ** 2) for i in range(1, nab + 1)]
            for s, axis in self.ax.items():
                v = torch.ones(self.n[axis], dtype=torch.float64, device=self.dev)
                w = torch.tensor(t, dtype=torch.float64, device=self.dev)
                if not (s == "z" and self.fs and self.c["ND"] != 22):
                    v[:nab] *= w
                v[-nab:] *= w.flip(0)
                self.taper[s] = self._line(v, axis)
            return
        amax = math.pi * FPML
        d0 = -(NPOWER + 1) * VPPML * math.log(float(np.float32(0.0008))) / (2 * nab * dh)
        for s, axis in self.ax.items():
            n = self.n[axis]
            for half in (0, 1):
                K, a, b = np.ones(n), np.zeros(n), np.zeros(n)
                for i in range(n):
                    near = i < nab and not (s == "z" and self.fs)
                    if not near and i <= n - nab - 1:
                        continue
                    j = i if near else (n - 1 - i if half else n - i)
                    x = (nab - j - (0.5 if half else 0)) / nab
                    d = d0 * (0.25 * x + 0.75 * x ** NPOWER)
                    K[i] = 1 + (KMAX - 1) * x ** NPOWER
                    al = amax * (1 - x)
                    b[i] = math.exp(-(d / K[i] + al) * dt)
                    a[i] = d * (b[i] - 1) / (K[i] * (d + K[i] * al)) if abs(d) > 1e-6 else 0.0
                self.pml[s, half] = tuple(self._line(self._t(v), axis) for v in (K, a, b))

    def _line(self, v, axis):
        shape = [1] * len(self.n)
        shape[axis] = -1
        return v.reshape(shape)

    # ---- fields -----------------------------------------------------------
    def _zeros(self, full=True):
        n = tuple(k + 2 * self.H for k in self.n) if full else self.n
        return torch.zeros(n, dtype=torch.float64, device=self.dev)

    def state(self):
        f = {"v" + s: self._zeros() for s in self.ax}
        if self.c["ND"] == 22:
            f["p"] = self._zeros()
        else:
            for k in [s + s for s in self.ax] + list(self.ms):
                f["s" + k] = self._zeros()
                if self.L:
                    f["r" + k] = [self._zeros(False) for _ in range(self.L)]
        f["psi"] = {}
        return f

    def inner(self, a):
        for k in range(a.dim()):
            a = a.narrow(k, self.H, a.shape[k] - 2 * self.H)
        return a

    def diff(self, f, name, s, plus, psi=None):
        """Staggered derivative of field `name` along s, CPML-corrected with
        the memory psi when given."""
        a, H, axis = f[name], self.H, self.ax[s]
        for k in range(a.dim()):
            if k != axis:
                a = a.narrow(k, H, a.shape[k] - 2 * H)
        n = self.n[axis]
        out = None
        for k, h in enumerate(self.hc):
            hi, lo = (k + 1, -k) if plus else (k, -k - 1)
            t = a.narrow(axis, H + hi, n) - a.narrow(axis, H + lo, n)
            out = t.mul_(h) if out is None else out.add_(t, alpha=h)
        if psi is not None and self.pml:
            K, al, b = self.pml[s, 1 if plus else 0]
            key = name + s
            if key not in psi:
                psi[key] = self._zeros(False)
            q = psi[key].mul_(b).addcmul_(al, out)
            out = out.div_(K).add_(q)
        return out

    def dv(self, f, pml=True):
        """Velocity increments."""
        psi = f["psi"] if pml else None
        if self.c["ND"] == 22:
            return {"v" + s: self.diff(f, "p", s, True, psi) * self.rv["v" + s] for s in self.ax}
        out = {}
        for s in self.ax:
            d = None
            for t in self.ax:
                key = "s" + "".join(sorted(s + t))
                q = self.diff(f, key, t, s == t, psi)
                d = q if d is None else d.add_(q)
            out["v" + s] = d.mul_(self.rv["v" + s])
        return out

    def strains(self, f, pml=True):
        psi = f["psi"] if pml else None
        e = {s + s: self.diff(f, "v" + s, s, False, psi) for s in self.ax}
        if self.c["ND"] != 22:
            for k in self.ms:
                e[k] = (self.diff(f, "v" + k[0], k[1], True, psi)
                        .add_(self.diff(f, "v" + k[1], k[0], True, psi)))
        return e

    def elastic_ds(self, e, M, f2, ms):
        th = sum(e[s + s] for s in self.ax)
        out = {s + s: M * th - f2 * (th - e[s + s]) for s in self.ax}
        out.update({k: ms[k] * e[k] for k in ms})
        return out

    def taper_(self, a):
        for w in self.taper.values():
            a.mul_(w)

    def update_v(self, f):
        for k, d in self.dv(f).items():
            a = self.inner(f[k])
            a.add_(d)
            self.taper_(a)

    def update_s(self, f):
        """Stress update; returns (strains, partial increments, memory
        terms old, new) for the gradients."""
        e = self.strains(f)
        if self.c["ND"] == 22:
            a = self.inner(f["p"])
            a.add_(self.M * sum(e.values()))
            self.taper_(a)
            return None
        old, new = {}, {}
        if not self.L:
            inc = self.elastic_ds(e, self.M, 2 * self.mu, self.ms)
        else:
            inc = self.elastic_ds(e, self.g, self.f, self.ms)
            drive = self.elastic_ds(e, self.e, self.d, self.ds)
            for k in inc:
                r = f["r" + k]
                old[k] = self.dt / 2 * sum(r)
                for q, (b, c, et) in zip(r, self.rl):
                    q.mul_(c).add_(drive[k], alpha=-et).mul_(b)
                new[k] = self.dt / 2 * sum(r)
                inc[k] = inc[k] + old[k]
        for k in inc:
            a = self.inner(f["s" + k])
            a.add_(inc[k])
            if self.L:
                a.add_(new[k])
            self.taper_(a)
        return e, inc, old, new

    def surface(self, f, e):
        """Image-method free surface after update_s, with its strains."""
        if not self.fs:
            return
        H = self.H
        top = lambda a: a[..., 0]
        self.inner(f["szz"])[..., 0] = 0
        for m in range(1, H + 1):
            f["szz"][..., H - m] = -f["szz"][..., H + m]
            for k in ("sxz", "syz"):
                if k in f:
                    f[k][..., H - m] = -f[k][..., H + m - 1]
        hor = [s for s in self.ax if s != "z"]
        eh = sum(top(e[s + s]) for s in hor)
        ez = top(e["zz"])
        g, f2 = (self.g, self.f) if self.L else (self.M, 2 * self.mu)
        g, f2 = top(g), top(f2)
        h = -((g - f2) ** 2 * eh / g) - (g - f2) * ez
        for s in hor:
            a = top(self.inner(f["s" + s + s]))
            a.add_(h)
            if self.L:
                d, ee = top(self.d), top(self.e)
                r = [top(q) for q in f["r" + s + s]]
                a.sub_(self.dt / 2 * sum(r))
                for q, (b, _, et) in zip(r, self.rl):
                    q.add_(b * et * ((d - ee) * (f2 / g - 1) * eh - (d - ee) * ez))
                a.add_(self.dt / 2 * sum(r))
        if self.L:
            for q in f["rzz"]:
                q[..., 0] = 0

    # ---- shots ------------------------------------------------------------
    def bind(self, shot):
        pos, src, rec = shot
        cell = lambda v: np.trunc(np.float32(v) / np.float32(self.dh)).astype(np.int64)
        keys = ("x", "y", "z") if self.three else ("x", "z")
        row = {"x": 0, "y": 1, "z": 2}
        self.sc = tuple(int(cell(pos[row[s]])[0]) for s in keys)
        self.rc = tuple(torch.from_numpy(cell(rec[row[s]])).to(self.dev) for s in keys)
        self.stype = int(pos[4, 0])
        self.src = [float(np.float32(v)) for v in src[:, 0]]
        so, nd = self.c["seisout"], self.c["ND"]
        v = ["vx", "vy", "vz"] if nd == 3 else ["vx", "vz"]
        s = [] if nd == 22 else ["sxx", "szz", "sxz"]
        self.outs = {1: v, 2: ["p"], 4: v + s + ["p"]}[so]

    def normals(self):
        return ["s" + s + s for s in self.ax]

    def inject(self, f, t, sign=1):
        amp = sign * self.dt * self.src[t]
        if self.stype == 100:
            for k in self.normals():
                self.inner(f[k])[self.sc] += amp / len(self.ax)
        else:
            self.inner(f["vz" if self.stype == 2 else "p"])[self.sc] += amp

    def record(self, f):
        out = []
        for k in self.outs:
            if k == "p" and self.c["ND"] != 22:
                out.append(sum(self.inner(f[q])[self.rc] for q in self.normals()) / len(self.ax))
            else:
                out.append(self.inner(f[k])[self.rc])
        return torch.stack(out)

    def forward(self, shot, keep=None):
        """Seismograms [nout][NT, nrec]; keep(f, t, when) sees the state after
        the sources ("src") and after the stress update ("end")."""
        self.bind(shot)
        f, rec = self.state(), []
        for t in range(self.c["NT"]):
            self.inject(f, t)
            if keep:
                keep(f, t, "src")
            self.update_v(f)
            r = self.update_s(f)
            if keep:
                keep(f, t, "end")
            self.surface(f, r[0] if r else None)
            rec.append(self.record(f))
        return f, list(torch.stack(rec, 1))

    # ---- gradients --------------------------------------------------------
    def shell(self):
        """Mask of the FDOH-thick shell on the inner face of the layers."""
        m = torch.zeros(self.n, dtype=torch.bool, device=self.dev)
        a, H = self.nab, self.H
        m[tuple(slice(a, n - a) for n in self.n)] = True
        m[tuple(slice(a + H, n - a - H) for n in self.n)] = False
        return m

    def fields(self):
        return ["v" + s for s in self.ax] + self.normals() + ["s" + k for k in self.ms]

    def scaled(self, res):
        """Adjoint sources: the residuals in the units of the updates."""
        out = []
        for k, r in zip(self.outs, res):
            if k == "p":
                w = -2 * (self.M - self.mu)[self.rc] * self.dh
            else:
                w = self.rv[k][self.rc] * self.dt * self.dt / self.dh
            out.append(r * w)
        return out

    def add_sources(self, f, res, t):
        for k, r in zip(self.outs, res):
            names, v = ([k], r[t]) if k != "p" else (self.normals(), r[t] / len(self.ax))
            for q in names:
                self.inner(f[q])[self.rc] += v

    def surface_adj(self, f):
        nd = len(self.ax)
        top = lambda a: a[..., 0]
        M, mu = top(self.M), top(self.mu)
        lam = M - 2 * mu
        s = {k: top(self.inner(f["s" + k + k])) for k in self.ax}
        a = {k: -v.clone() for k, v in s.items()}
        if nd == 2:
            q = 1 / (4 * M * mu - 4 * mu * mu)
            n = {"x": q * (M * a["x"] - lam * a["z"]), "z": torch.zeros_like(M)}
        else:
            q = 1 / (6 * M * mu - 8 * mu * mu)
            n = {k: q * (2 * (M - mu) * a[k] - lam * (a["x"] + a["y"] + a["z"] - a[k]))
                 for k in self.ax}
            n["z"] = torch.zeros_like(M)
        tot = sum(n.values())
        for k in self.ax:
            s[k].copy_(-(M * n[k] + lam * (tot - n[k])))
        h, hz, ts = -lam ** 2 / M, -lam, tot - n["z"]
        w = h * ts
        for k in self.ax:
            if k == "z":
                continue
            axis, n_ = self.ax[k], self.n[self.ax[k]]
            v = top(self.inner(f["v" + k]))
            r = top(self.rv["v" + k])
            for j, c in enumerate(self.hc):
                # the column's own strain takes +c at offset -j, -c at j + 1
                v.narrow(axis, j, n_ - j).add_(
                    c * w.narrow(axis, 0, n_ - j) * r.narrow(axis, j, n_ - j))
                v.narrow(axis, 0, n_ - j - 1).sub_(
                    c * w.narrow(axis, j + 1, n_ - j - 1) * r.narrow(axis, 0, n_ - j - 1))
        vz = self.inner(f["vz"])
        for j, c in enumerate(self.hc):
            vz[..., j].add_(c * hz * ts * self.rv["vz"][..., j])

    def gradient(self, shot, res_of):
        """(seismograms, gradients): res_of(seismograms) gives the residuals."""
        nt, names = self.c["NT"], None
        hist, mask = [], None if self.L else None

        def keep(f, t, when):
            if self.L and when == "src":
                hist.append([self.inner(f[k]).clone() for k in self.fields()])
            if not self.L and when == "end":
                hist.append([self.inner(f[k])[mask] for k in self.fields()])
        if not self.L:
            mask = self.shell()
        f, out = self.forward(shot, keep)
        names = self.fields()
        res = self.scaled(res_of(out))
        a = self.state()
        gM, gmu, gr = (torch.zeros(self.n, dtype=torch.float64, device=self.dev)
                       for _ in range(3))
        gtp, gts = torch.zeros_like(gM), torch.zeros_like(gM)
        M, mu = self.M0, self.mu0
        nd = len(self.ax)
        bulk = 3 * M - 4 * mu if nd == 3 else 2 * M - 2 * mu
        c1, c3 = 1 / bulk ** 2, 1 / mu ** 2
        for t in range(nt - 1, 0, -1):
            if self.fs:
                self.surface_adj(a)
            self.add_sources(a, res, t)
            if self.L:
                h = dict(zip(names, hist.pop()))
            else:
                hist.pop()
                e = self.strains(f, False)
                for k, d in self.elastic_ds(e, self.M, 2 * self.mu, self.ms).items():
                    self.inner(f["s" + k]).sub_(d)
                for k, v in zip(names, hist[-1]):
                    if k[0] == "s":
                        self.inner(f[k])[mask] = v
                h = {k: self.inner(f[k]) for k in names}
            e, ls, old, new = self.update_s(a)
            s = {k: h["s" + k] for k in ls}
            sd = sum(s[q + q] for q in self.ax)
            dM = c1 * sd * sum(ls[q + q] for q in self.ax)
            if nd == 3:
                dev = c3 / 6 * sum(ls[q + q] * (3 * s[q + q] - sd) for q in self.ax)
                dmu = 4 / 3 * dM - dev
            else:
                dmu = dM - c3 / 4 * (s["xx"] - s["zz"]) * (ls["xx"] - ls["zz"])
            gmu += dmu - c3 * sum(s[k] * ls[k] for k in self.ms)
            gM -= dM
            if self.L:
                self.tau_terms(e, s, ls, old, new, bulk, gtp, gts)
            else:
                dv = self.dv(f, False)
                for k, d in dv.items():
                    self.inner(f[k]).sub_(d)
                for k, v in zip(names, hist[-1]):
                    if k[0] == "v":
                        self.inner(f[k])[mask] = v
            d = self.dv(a)
            for k in d:
                self.inner(a[k]).add_(d[k])
                gr -= h[k] * d[k]
            if not self.L:
                self.inject(f, t, -1)
        return out, self.transform(gM, gmu, gr, gtp, gts)

    def tau_terms(self, e, s, ls, old, new, bulk, gtp, gts):
        nd, L, dt, s0 = len(self.ax), self.L, self.dt, self.s0
        tp, ts = self.p["taup"], self.p["taus"]
        th = sum(e[q + q] for q in self.ax)
        Rm = {k: old[k] + new[k] for k in ls}
        F = sum(Rm[q + q] for q in self.ax) / (nd * self.e - (nd - 1) * self.d)
        kp, ks = s0 / (1 + s0 * tp), s0 / (1 + s0 * ts)
        Xp = (self.M * L - kp * self.g) * th + (self.M / dt - kp * self.e) * F
        lam = self.M0 - 2 * self.mu0
        sth = sum(s[q + q] for q in self.ax) / bulk
        gtp -= sth * Xp
        tot = 0
        for q in self.ax:
            k = q + q
            dev, m = th - e[k], self.e * F - Rm[k]
            X = -(2 * self.mu * L * dev) - m / ts - ks * (-(self.f * dev) - m)
            tot = tot + (s[k] - lam * sth) / (2 * self.mu0) * X
        for k in self.ms:
            mu = self.ms[k] - L * self.ds[k] * dt
            tk = torch.where(mu != 0, self.ds[k] * dt / mu, torch.zeros_like(mu))
            X = mu * L * e[k] - s0 / (1 + s0 * tk) * (ls[k] + new[k])
            X = X + torch.where(tk > 0, Rm[k] / tk, torch.zeros_like(mu))
            tot = tot + s[k] / self.mu0 * X
        gts -= tot

    def transform(self, gM, gmu, gr, gtp, gts):
        dt, dh, rho = self.dt, self.dh, self.rho
        M, mu = self.M0 * dh / dt, self.mu0 * dh / dt
        gM, gmu = gM / dt, gmu / dt
        gr = gr / dt * dh * dh / (dt * dt) + M / rho * gM + mu / rho * gmu
        g = dict(vp=2 * torch.sqrt(rho * M) * gM, vs=2 * torch.sqrt(rho * mu) * gmu, rho=gr)
        if self.L:
            g.update(taup=gtp * dh / dt ** 2, taus=gts * dh / dt ** 2)
        return {k: v.permute(*reversed(range(v.dim()))).contiguous() for k, v in g.items()}


def exact(case, seed):
    if case["kind"] == "serve":
        return [exact(c, s) for c, s in _requests(case, seed)]
    csts, params, shots, data = _inputs(case, seed)
    x = _Exact(case, csts, params)
    if case["kind"] == "forward":
        return x.forward(shots[0])[1]
    outs, grad = [], None
    for shot, din in zip(shots, data):
        d = [x._t(v) for v in din]
        out, g = x.gradient(shot, lambda o: [u - v for u, v in zip(o, d)])
        outs += out
        grad = g if grad is None else {k: grad[k] + g[k] for k in g}
    if case["kind"] == "autograd":
        grad = [grad[k] for k in ("vp", "vs", "rho")]
    return dict(out=outs, grad=grad)
