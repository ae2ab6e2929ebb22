"""The work that users of this stepper have it do, as measurable cases.

A case is one program's use of the public entry points (HipStepper, its meter and downloads, TDGLGPU's
upload / steps / download cycle of tdglgpu, HipBatch): its way of driving the stepper, its material, its
grid and its scheme options.  `listed` holds the cases that stand for the configurations the repository
quotes and for the odd sizes between them; `draw` gives more of the same ranges.

`exact` steps the same inputs in plain 64-bit torch: the scheme's formulas on whole arrays, with the field
solved by conjugate gradients to the rounding.  It takes the Stepper's coefficients, masks and boundary
profiles as inputs, as the device does, and none of the repository's stepping code.
"""
import math

import numpy as np
import torch

from juliatdgl_amd import configs
from juliatdgl_amd.hip import HipBatch, HipStepper
from juliatdgl_amd.meter import Voltmeter
from juliatdgl_amd.scheme import Grid, catalogue_masks, hole_masks, make_stepper, notch_masks, two_band, wedge_masks
from juliatdgl_amd.state import State, seeded_state
from juliatdgl_amd.sweep import RunSpec, state_of, stepper_of
from juliatdgl_amd.tdglgpu import GPUStepper, device_state, device_state_, gpu_steps, host_state

LMAX = 40  # time steps of a ladder cycle


# ------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # The smallest call: one time step of the CPU-runnable case and a look at the state, as a script that
        # follows a transient does.  Launches, copies and waits are all there is.
        dict(name="single_step_12x8x4", way="transfer", model="two", field="sep", nx=12, ny=8, nz=4, buf=1, steps=1),
        # TDGLGPU's ladder cycle (upload, lMax steps, download) with the PCG history carried in and out, on a small
        # sample with an insulating buffer and odd extents: the drop-in hook without a resident state.
        dict(name="hook_pcg_53x27x9", way="transfer", model="mgb2", field="pcg", nx=53, ny=27, nz=9, buf=2, steps=LMAX),
        # The reference's validation run plain96.toml as a resident ladder: ten cycles with their records, then
        # the state for a checkpoint.  The separable implicit field.
        dict(name="plain_96x48x24", way="ladder", model="mgb2", field="sep", nx=96, ny=48, nz=24, buf=1, cycles=10),
        # The reference's validation run pcg96.toml: the insulating PCG.
        dict(name="pcg_96x48x24", way="ladder", model="mgb2", field="pcg", nx=96, ny=48, nz=24, buf=2, cycles=6, tune=True),
        # Two KWT bands on staged steps with the rotating frame and the PCG at 1e-10, the bench's second workload.
        dict(name="kwt_pcg_128x64x16", way="ladder", model="kwt", field="pcg", nx=128, ny=64, nz=16, buf=2, cycles=5,
             tune=True),
        # The bench's default: three anisotropic bands, a wide insulating buffer, the open boundary; the largest run
        # the repository quotes.
        dict(name="open_3band_256x128x32", way="ladder", model="three", field="pcg", nx=256, ny=128, nz=32, buf=8,
             bc="open", cycles=2, tune=True),
        # The same physics on a small odd grid, untuned: what a user's first trial of the open boundary looks like.
        dict(name="open_3band_75x41x13", way="ladder", model="three", field="pcg", nx=75, ny=41, nz=13, buf=4, bc="open",
             cycles=4),
        # The upper end of the served range without noise: three bands, the separable field, planes too wide for
        # the full-length transforms.
        dict(name="plain_3band_256x128x32", way="ladder", model="three_dt", field="sep", nx=256, ny=128, nz=32, buf=1,
             cycles=3),
        # A served run with thermal noise from the device's generator, ten steps a call as crossing_times takes
        # them, on a ragged grid.
        dict(name="noise_148x60x10", way="ladder", model="three_dt", field="sep", nx=148, ny=60, nz=10, buf=1, cycles=30,
             lmax=10, noise=1e-3),
        # Two normal fluids: the Helmholtz solve for their potential beside the field solve.
        dict(name="fluids_60x36x12", way="ladder", model="mgb2", field="sep", nx=60, ny=36, nz=12, buf=1, cycles=5, qp=1.0),
        # The mode that keeps every inner vector of the solve in Float32 under FP64 refinement.
        dict(name="refine_97x64x16", way="ladder", model="three", field="pcg", nx=97, ny=64, nz=16, buf=4, cycles=2,
             refine=True),
        # A current sweep advanced by batched kernels: twelve runs of uneven grids in the sweep's range.
        dict(name="batch_12_runs", way="batch", model="two", field="sep", nx=160, ny=96, nz=24, buf=1, runs=12, cycles=4),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["plain", "pcg", "kwt", "open", "noise", "hook", "batch", "exact_pcg"])
    if kind == "batch":
        return dict(way="batch", model="two", field="sep", nx=4 * log(16, 40), ny=4 * log(8, 24), nz=4 * log(2, 6), buf=1,
                    runs=rng.randint(3, 12), cycles=rng.randint(1, 4))
    nx, ny, nz = log(24, 200), log(16, 100), log(4, 32)
    if kind == "plain":
        return dict(way="ladder", model=rng.choice(["mgb2", "three_dt"]), field="sep", nx=nx, ny=ny, nz=nz, buf=1,
                    cycles=rng.randint(1, 5))
    if kind == "noise":
        return dict(way="ladder", model=rng.choice(["two", "three_dt"]), field="sep", nx=nx, ny=ny, nz=nz, buf=1,
                    cycles=rng.randint(4, 20), lmax=10, noise=1e-3)
    if kind == "hook":
        return dict(way="transfer", model="mgb2", field=rng.choice(["sep", "pcg"]), nx=nx, ny=ny, nz=nz, buf=2,
                    steps=rng.choice([1, 10, LMAX]))
    if kind == "exact_pcg":  # every part of the solve in FP64
        return dict(way="ladder", model="mgb2", field="pcg", nx=min(nx, 96), ny=min(ny, 64), nz=min(nz, 20), buf=2, cycles=1,
                    pcg32=False)
    if kind == "kwt":
        return dict(way="ladder", model="kwt", field="pcg", nx=min(nx, 128), ny=min(ny, 64), nz=min(nz, 16), buf=2,
                    cycles=rng.randint(1, 3))
    if kind == "open":
        return dict(way="ladder", model="three", field="pcg", nx=min(nx, 128), ny=min(ny, 64), nz=min(nz, 16),
                    buf=rng.randint(2, 8), bc="open", cycles=rng.randint(1, 2))
    return dict(way="ladder", model="mgb2", field="pcg", nx=nx, ny=ny, nz=nz, buf=rng.randint(2, 4), cycles=rng.randint(1, 3),
                tune=rng.random() < 0.5)


# ------------------------------------------------------------------------------------------- the inputs
def _stepper(c):
    """The Stepper of a case and its (H, J)."""
    nx, ny, nz, buf = c["nx"], c["ny"], c["nz"], c["buf"]
    kw = {}
    if c["field"] == "pcg":
        kw.update(sigma_vac=0.01)
        if c.get("pcg32") is False:
            kw.update(pcg_fast=False, pcg_f32=False, pcg_tol=1e-12)
        if c.get("refine"):
            kw.update(pcg_refine=True)
    if c.get("bc") == "open":
        kw.update(selffield_bc="open")
    if c.get("qp"):
        kw.update(qp_exchange=c["qp"])
    if c["model"] == "kwt":
        st, p = configs.kwt_pcg_128x64x16(nx=nx, ny=ny, nz=nz)
        return st, p["H"], p["J"]
    gr = Grid.make(nx, ny, nz, dx=0.5, buf=buf)
    if c["model"] == "three":
        mk = notch_masks(gr, (nx // 2 - 4, nx // 2 + 4), (0, ny // 4))
        return make_stepper(configs.three_band_aniso_model(), gr, mk, **kw), 0.2, 0.1
    if c["model"] == "mgb2":
        return make_stepper(two_band(xi_ratio=4.0, kappa=2.0), gr, wedge_masks(gr), **kw), 0.03, 0.3
    if c.get("noise"):
        kw.update(noise=c["noise"], noise_seed=11)
    if c["model"] == "three_dt":
        mk = hole_masks(gr, (nx / 2, ny / 2), 0.2 * min(nx, ny))
        return make_stepper(configs.three_band_aniso_model(), gr, mk, dt=0.01, **kw), 0.3, 0.4
    mk = catalogue_masks(gr, "WEDGE", wedge_depth=0.25)
    return make_stepper(configs.two_band_model(), gr, mk, dt=0.01, **kw), 0.3, 0.3


def _sizes(c):
    """The uneven grids of a batch: multiples of four from a fifth of the largest up to it."""
    r = np.random.default_rng(c["runs"])
    out = []
    for q in range(c["runs"]):
        s = r.uniform(0.25, 1.0, 3) if q else np.ones(3)
        out.append(tuple(max(lo, 4 * int(round(n * x / 4))) for n, x, lo in zip((c["nx"], c["ny"], c["nz"]), s, (32, 16, 4))))
    return out


def _specs(c, seed):
    return [RunSpec(q, nx, ny, nz, (0.05 + 0.03 * q) * (1 if q % 2 else -1), depth=0.1 + 0.02 * q, seed=1000 * seed + q)
            for q, (nx, ny, nz) in enumerate(_sizes(c))]


def _meter(st):
    return Voltmeter.of_ladder(st, min(8, (st.grid.x2 - st.grid.x1) // 4))


def prepare(case, seed):
    c = case
    if c["way"] == "batch":
        devs, runs = [], []
        for spec in _specs(c, seed):
            st = stepper_of(spec)
            dev = HipStepper(st)
            s0 = state_of(spec, st)
            dev.upload(s0)
            dev.meter_begin(_meter(st))
            devs.append(dev)
            runs.append((st, spec.H, st.selffield(spec.J), s0))
        return dict(case=c, devs=devs, batch=HipBatch(devs), H=[r[1] for r in runs], HJ=[r[2] for r in runs], m=0,
                    out=[r[3].empty_like() for r in runs])
    st, H, J = _stepper(c)
    s0 = seeded_state(st.model, st.grid, st.masks, H, seed=seed)
    HJ = st.selffield(J)
    if c["way"] == "transfer":
        gs = GPUStepper(st)
        return dict(case=c, gs=gs, g=device_state(gs, s0), s=s0, H=H, HJ=HJ, pcg=None)
    dev = HipStepper(st)
    dev.upload(s0)
    if c.get("tune"):
        dev.autotune(H, HJ)
    dev.meter_begin(_meter(st))
    return dict(case=c, dev=dev, H=H, HJ=HJ, m=0, out=s0.empty_like())


def _fields(s: State):
    return dict(s.arrays())


def _record(r):
    return [r["V"], r["TA"], r["Tf1"], *r["T"], *r["Tabs"], r["It"], r["Is"], *r["dif"], r["amax"], r["diffh"]]


def run(state):
    c = state["case"]
    H, HJ = state["H"], state["HJ"]
    if c["way"] == "transfer":
        # _gpu_cycle!: the state (and the PCG history) up, the steps, both down
        s, gs, g = state["s"], state["gs"], state["g"]
        device_state_(g, s)
        if state["pcg"] is not None:
            gs.dev.set_pcg(state["pcg"])
        gpu_steps(g, gs, c["steps"], H=H, HJ=HJ)
        if c["field"] == "pcg":
            state["pcg"] = gs.dev.get_pcg()
        return _fields(host_state(s, g))
    recs = []
    if c["way"] == "batch":
        for _ in range(c["cycles"]):
            state["batch"].step(LMAX, H, HJ)
            recs.append([x for r in state["batch"].meter_cycle(state["m"] == 0) for x in _record(r)])
            state["m"] += 1
        out = {}
        for q, (dev, into) in enumerate(zip(state["devs"], state["out"])):
            dev.download(into)
            out[f"run{q}"] = {k: v for k, v in zip(("G1", "G2", "thx", "thy", "thz"), (*into.G, into.thx, into.thy, into.thz))}
        return dict(out, records=np.array(recs))
    dev = state["dev"]
    for _ in range(c["cycles"]):
        dev.step(c.get("lmax", LMAX), H, HJ)
        recs.append(_record(dev.meter_cycle(state["m"] == 0)))
        state["m"] += 1
    return dict(_fields(dev.download(state["out"])), records=np.array(recs))


# ------------------------------------------------------------------------------------------- what it needs
def _grids(c):
    if c["way"] == "batch":
        return [(2, nx + 2, ny + 2, nz + 2) for nx, ny, nz in _sizes(c)]
    b = 2 if c["model"] == "kwt" else c["buf"]
    bands = 3 if c["model"].startswith("three") else 2
    return [(bands, c["nx"] + 2 * b, c["ny"] + 2 * b, c["nz"] + 2 * b)]


def work(case):
    """Per step: the bands, links, field, current and masks read once and what the step changes written once; the
    band update, the currents, the curl with its sines, and the field's solve with its one pair of transforms (dense
    half-size products along each axis).  Per pass: the state once more for each direction it travels."""
    c = case
    steps = c["steps"] if c["way"] == "transfer" else c["cycles"] * c.get("lmax", LMAX)
    by = fl = 0.0
    for bands, Nx, Ny, Nz in _grids(c):
        n = (Nx + 1) * (Ny + 1) * (Nz + 1)
        state = n * (32 * bands + 3 * (8 + 8 + 16 + 16 + 8 + 8))
        by += steps * n * (32 * bands + 3 * (16 + 16) + 3 * 8 + 3 * (8 + 8) + 3 * (8 + 8) + 4 * 8)
        by += state * (2 if c["way"] == "transfer" else 1)
        fl += steps * n * (bands * 200 + 400 + 3 * 2 * (Nx + Ny + Nz))
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """Relative 2-norm of each output array.  The separable solve is direct: its transforms in another grouping of
    their sums (parity-folded or full length) differ by up to 2.3e-12 and 8.4e-11 (the largest value's, hx, which is
    small against the fields it is the difference of).  The PCG stops at its tolerance (1e-8, 1e-10 with KWT, 1e-12 all
    in FP64), and where inside it depends on the order of its sums: two preconditioner paths differ by up to 8.4e-8 and
    7.1e-7 on the listed cases (the z links' phases, which carry little) and by more on some smaller ones."""
    if case["field"] == "sep":
        return {"rel": 1e-11, "max": 4e-10}
    return {"rel": 1e-6, "max": 1e-5}


# ------------------------------------------------------------------------------------------- in 64 bits
def _i(z):
    return 1j * z


class _Plain:
    """The release-2.0 step of one run on whole torch arrays (complex128 / float64), index i of the reference at
    i - 1."""

    def __init__(self, st, s, dev):
        self.st, self.gr = st, st.grid
        self.dev = dev
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
        self.G = [t(g) for g in s.G]
        self.th = [t(s.thx), t(s.thy), t(s.thz)]
        self.ph = [t(s.phx), t(s.phy), t(s.phz)]
        self.V = [t(s.Vx), t(s.Vy), t(s.Vz)]
        self.U = [t(s.Ux), t(s.Uy), t(s.Uz)]
        self.J = [t(s.Jx), t(s.Jy), t(s.Jz)]
        self.h = [t(s.hx), t(s.hy), t(s.hz)]
        mk = st.masks
        self.f = t(mk.f)
        self.tau = [t(mk.tx), t(mk.ty), t(mk.tz)]
        gr = self.gr
        self.sl = (slice(gr.x1, gr.x2), slice(gr.y1, gr.y2), slice(gr.z1, gr.z2))  # interior nodes of the block
        self.D = [t(d) for d in st.D] if st.D is not None else None
        self.x = None
        self.bar = {k: t(v) for k, v in st.bar.items()} if st.bar is not None else None
        n = (gr.Nx - 1, gr.Ny - 1, gr.Nz - 1)
        self.basis = [self._bases(m) for m in n]
        self.count, self.old, self.new = -1, None, None
        if st.open is not None:
            self._green()

    # ---- the bands
    def _bases(self, n):
        k = torch.arange(n, dtype=torch.float64, device=self.dev)
        s = 2 * torch.sin(math.pi * k / (2 * n))
        V = math.sqrt(2 / n) * torch.cos(math.pi * k[None, :] * (k[:, None] + 0.5) / n)
        V[:, 0] = 1 / math.sqrt(n)
        U = -math.sqrt(2 / n) * torch.sin(math.pi * k[None, 1:] * (k[:-1, None] + 1) / n)
        return V, U, s

    def _om_pad(self, om):
        """The frame's rate on every block node: the faces copy the nearest interior node."""
        return torch.nn.functional.pad(om[None, None], (1, 1, 1, 1, 1, 1), mode="replicate")[0, 0]

    def _links(self, mode, c, om):
        """The links of a stage over the interior and its faces: per axis the link towards +e of every node from the
        one before the interior on."""
        gr, out = self.gr, []
        for ax in range(3):
            sl = list(self.sl)
            sl[ax] = slice(sl[ax].start - 1, sl[ax].stop)
            v = self.V[ax][tuple(sl)]
            if mode == "direct":
                out.append(v)
                continue
            q = v * self.U[ax][tuple(sl)].conj()
            sf = -q.imag
            small = (q.real > 0) & (sf.abs() <= 0.05)
            if mode == "frac":
                t = (sf + sf ** 3 / 6) * c
                short = torch.complex(1 - t * t / 2, -t * (1 - t * t / 6))
                out.append(v * torch.where(small, short, torch.polar(torch.ones_like(sf), q.angle() * c)))
            else:  # the rotating frame: V e^{i R c}, R the links' own turn and the frame's along them
                p = self._om_pad(om)
                n = p.shape[ax] - 1
                inner = [slice(1, -1)] * 3
                inner[ax] = slice(0, n + 1)
                p = p[tuple(inner)]
                dom = p.narrow(ax, 1, n) - p.narrow(ax, 0, n)
                a = (torch.where(small, -(sf + sf ** 3 / 6), q.angle()) + dom * self.st.dt) * c
                short = torch.complex(1 - a * a / 2, a * (1 - a * a / 6))
                out.append(v * torch.where(a.abs() <= 0.05, short, torch.polar(torch.ones_like(a), a)))
        return out

    def _stage(self, mu, cf, S, L, fly):
        """One pass of band mu on the interior from the node array S with the links L."""
        gr, sl = self.gr, self.sl
        g = S[sl]
        acc = g
        for ax, k in enumerate((cf.kx, cf.ky, cf.kz)):
            n = g.shape[ax]
            lp, lm = L[ax].narrow(ax, 1, n), L[ax].narrow(ax, 0, n)
            up, dn = list(sl), list(sl)
            up[ax] = slice(sl[ax].start + 1, sl[ax].stop + 1)
            dn[ax] = slice(sl[ax].start - 1, sl[ax].stop - 1)
            sp, sm = S[tuple(up)], S[tuple(dn)]
            if fly:  # the covariant Neumann ghosts of S
                sp, sm = sp.clone(), sm.clone()
                sp.select(ax, n - 1).copy_((lp.conj() * g).select(ax, n - 1))
                sm.select(ax, 0).copy_((lm * g).select(ax, 0))
            acc = acc + k * (lp * sp - 2 * g + lm.conj() * sm)
        acc = acc + (self.f[sl] * cf.eps - cf.beta * (g.abs() ** 2)) * (cf.c * g)
        for nu in range(self.st.N):
            if nu != mu:
                acc = acc + cf.cpl[nu] * self.G[nu][sl]
        if cf.g2 > 0:
            q = 1 + cf.g2 * g.abs() ** 2
            dp = torch.sqrt(q) * (acc - g)
            acc = g + dp - ((g.conj() * dp).real / q) * (cf.g2 * g)
        return acc

    def _band(self, mu):
        st, sl = self.st, self.sl
        ns = st.rkl[mu]
        kc = st.rkc[mu] if (ns > 0 and st.rkc is not None) else None
        cf = st.bcs[mu] if ns > 0 else st.bc[mu]
        h = st.dt / st.divisor[mu] if ns > 0 else st.dt
        A = B = self.G[mu]
        om = None
        for j in range(1, max(ns, 1) + 1):
            mode, c = "direct", 0.0
            if j >= 2 and st.extrap:
                mode = "rot" if st.rotframe else "frac"
                c = kc.c[j - 2] if kc is not None else (j - 1) * j / (ns * (ns + 1))
            g = B[sl]
            p = self._stage(mu, cf, B, self._links(mode, c, om), j >= 2)
            if st.rotframe:
                if j == 1:
                    a2 = g.abs() ** 2
                    w = ((g.conj() * (p - g)).imag / (a2 * h)).clamp(-0.5 / st.dt, 0.5 / st.dt)
                    om = torch.where(a2 > 1e-3, w, torch.zeros_like(w))
                p = p - _i(om * h) * g
            if j >= 2:
                m, n = (kc.mu[j - 1], kc.nu[j - 1]) if kc is not None else ((2 * j - 1) / j, (1 - j) / j)
                p = m * p + n * A[sl]
            if st.rotframe and j == max(ns, 1):
                p = p * torch.polar(torch.ones_like(om), om * st.dt)
            C = self.G[mu].clone()
            C[sl] = p
            A, B = B, C
        return B

    # ---- the field
    def _diff(self, a, ax):
        n = a.shape[ax] - 1
        return a.narrow(ax, 1, n) - a.narrow(ax, 0, n)

    def _back(self, a, ax):
        """a(i) - a(i - 1) with zeros outside: the adjoint of -_diff."""
        z = list(a.shape)
        z[ax] = 1
        z = torch.zeros(z, dtype=a.dtype, device=a.device)
        return self._diff(torch.cat([z, a, z], ax), ax)

    def _curl(self, p):
        px, py, pz = p
        d = self._diff
        return d(pz, 1) - d(py, 2), d(px, 2) - d(pz, 0), d(py, 0) - d(px, 1)

    def _matvec(self, p, D):
        hx, hy, hz = self._curl(p)
        b, a = self._back, self.st.fc.a
        q = (b(hz, 1) - b(hy, 2), b(hx, 2) - b(hz, 0), b(hy, 0) - b(hx, 1))
        return [d * x + a * y for d, x, y in zip(D, p, q)]

    def _transform(self, x, ax, M):
        return torch.movedim(torch.tensordot(x, M, dims=([ax], [0])), -1, ax)

    def _direct(self, b):
        """(I + aK)^{-1} b by the cosine and sine bases of the three axes."""
        X = []
        for c in range(3):
            x = b[c]
            for ax in range(3):
                V, U, _ = self.basis[ax]
                x = self._transform(x, ax, U if ax == c else V)
            X.append(torch.nn.functional.pad(x, tuple(v for ax in (2, 1, 0) for v in ((1, 0) if ax == c else (0, 0)))))
        kx, ky, kz = (self.basis[ax][2].view([-1 if a == ax else 1 for a in range(3)]) for ax in range(3))
        k2 = kx * kx + ky * ky + kz * kz
        d = (kx * X[0] + ky * X[1] + kz * X[2]) / k2.clamp_min(1e-300)
        f = 1 / (1 + self.st.fc.a * k2)
        out = []
        for c, k in enumerate((kx, ky, kz)):
            x = k * d + f * (X[c] - k * d)
            x = x.narrow(c, 1, x.shape[c] - 1)
            for ax in range(3):
                V, U, _ = self.basis[ax]
                x = self._transform(x, ax, (U if ax == c else V).T)
            out.append(x)
        return out

    def _solve(self, b, D):
        """(D + aK) x = b by conjugate gradients under the direct solve with D = 1, from the last solution."""
        dot = lambda u, v: sum((p * q).sum() for p, q in zip(u, v))  # noqa: E731
        nb = dot(b, b).sqrt()
        if float(nb) == 0:
            self.x = [torch.zeros_like(v) for v in b]
            return self.x
        x = self.x if self.x is not None else self._direct(b)
        r = [u - v for u, v in zip(b, self._matvec(x, D))]
        z = self._direct(r)
        p, rz = z, dot(r, z)
        for q in range(300):
            if q % 4 == 0 and float(dot(r, r).sqrt() / nb) < 1e-13:
                break
            w = self._matvec(p, D)
            al = rz / dot(p, w)
            x = [u + al * v for u, v in zip(x, p)]
            r = [u - al * v for u, v in zip(r, w)]
            z = self._direct(r)
            rz, old = dot(r, z), rz
            p = [u + (rz / old) * v for u, v in zip(z, p)]
        self.x = x
        return x

    def _ranges(self):
        i = slice(1, -1)
        return [(i, i, i)] * 3  # per component: links 2..N-1 along its own axis, nodes 2..N along the others

    def _field(self):
        st, gr = self.st, self.gr
        fc, out = st.fc, []
        hx, hy, hz = self.h
        s = slice(1, -1)
        d = self._diff
        cur = ((fc.sxy, d(hz, 1)[:, :, s], fc.sxz, d(hy, 2)[:, s, :]), (fc.syz, d(hx, 2)[s, :, :], fc.syx, d(hz, 0)[:, :, s]),
               (fc.szx, d(hy, 0)[:, s, :], fc.szy, d(hx, 1)[s, :, :]))
        for ax in range(3):
            inr = tuple(slice(None) if a == ax else s for a in range(3))
            node, nxt = list(inr), list(inr)
            node[ax], nxt[ax] = slice(0, -1), slice(1, None)
            V = self.V[ax][inr]
            J = sum(st.wa[ax][mu] * (self.G[mu][tuple(node)].conj() * V * self.G[mu][tuple(nxt)]).imag for mu in range(st.N))
            self.J[ax] = torch.zeros_like(self.J[ax])
            self.J[ax][inr] = J
            c1, d1, c2, d2 = cur[ax]
            inc = (fc.d1 * self.tau[ax][tuple(node)]) * J - c1 * d1 + c2 * d2
            ph = self.ph[ax].clone()
            ph[inr] = self.th[ax][inr] + inc
            out.append(ph)
        b = [(o - t)[r].contiguous() for o, t, r in zip(out, self.th, self._ranges())]
        if self.D is not None:
            out = [t + (o - t) / dd for o, t, dd in zip(out, self.th, self.D)]
            D = [dd[r] for dd, r in zip(self.D, self._ranges())]
        else:
            D = [1.0, 1.0, 1.0]
        if st.field_mode in (1, 2):
            x = self._solve(b, D)
            for o, t, v, r in zip(out, self.th, x, self._ranges()):
                o[r] = t[r] + v
        return out

    # ---- the open boundary
    def _green(self):
        o = self.st.open
        self.M, self.ghat = [], []
        for c in range(3):
            n = [s + (0 if a == c else 1) for a, s in enumerate((self.gr.Nx, self.gr.Ny, self.gr.Nz))]
            M = [2 * v for v in n]
            ax = [torch.minimum(torch.arange(m), m - torch.arange(m)).double() for m in M]
            i, j, k = ax[0].view(-1, 1, 1), ax[1].view(1, -1, 1), ax[2].view(1, 1, -1)
            r2 = i * i + j * j + k * k
            far = (1 + (5 * (i ** 4 + j ** 4 + k ** 4) / r2 ** 2 - 3) / (8 * r2)) / (4 * math.pi * r2.sqrt())
            R = o.R
            t = torch.from_numpy(np.ascontiguousarray(o.lgf))
            near = t[i.long().clamp_max(R), j.long().clamp_max(R), k.long().clamp_max(R)]
            g = torch.where((i <= R) & (j <= R) & (k <= R), near, far)
            self.M.append(M)
            self.ghat.append(torch.fft.rfftn((o.fac * g).to(self.dev)))

    def _open(self, HJ):
        o, gr = self.st.open, self.gr
        first = self.count < 0
        self.count += 1
        if not (self.count >= o.every or first):
            return
        hx, hy, hz = self.h
        d, s = self._diff, slice(1, -1)
        jb = torch.from_numpy(np.ascontiguousarray(o.Jbar)).to(self.dev)
        dj = [torch.zeros_like(t) for t in self.th]
        dj[0][s, s, s] = (o.kappa2 * (d(hz, 1)[:, :, s] / gr.dy - d(hy, 2)[:, s, :] / gr.dz) - HJ * jb[None, s, s])[s]
        dj[1][s, s, s] = (o.kappa2 * (d(hx, 2)[s, :, :] / gr.dz - d(hz, 0)[:, :, s] / gr.dx))[:, s]
        dj[2][s, s, s] = (o.kappa2 * (d(hy, 0)[:, s, :] / gr.dx - d(hx, 1)[s, :, :] / gr.dy))[:, :, s]
        t = []
        for c in range(3):
            f = torch.fft.irfftn(torch.fft.rfftn(dj[c], s=self.M[c]) * self.ghat[c], s=self.M[c])
            n = dj[c].shape
            t.append(f[:n[0], :n[1], :n[2]])
        new = [v / (gr.dx * gr.dx) for v in self._curl(t)]
        self.old = new if first else self.new
        self.new = new
        self.count = 0

    def _boundary(self, h, H, HJ):
        st = self.st
        hx, hy, hz = h
        for a in (0, -1):
            hz[:, :, a] = hz[a] = hz[:, a] = H
            hx[a] = hx[:, a] = 0.0
            hy[:, a] = 0.0
        if st.selffield_bc == "slab":
            hy[:, :, 0], hy[:, :, -1] = -HJ, HJ
            return
        b = self.bar
        for c, a in enumerate((0, -1)):
            hy[:, :, a] = HJ * b["hy_z"][None, :, c]
        for c, a in enumerate((0, -1)):
            hy[:, a, :] = HJ * b["hy_y"][c][None]
        for c, a in enumerate((0, -1)):
            hz[:, :, a] = H + HJ * b["hz_z"][None, :, c]
        for c, a in enumerate((0, -1)):
            hz[:, a, :] = H + HJ * b["hz_y"][c][None]
        for a in (0, -1):
            hz[a] = H + HJ * b["hz_x"]
            hy[a] = HJ * b["hy_x"]
        if st.open is None:
            return
        f = min((self.count + 1) / st.open.every, 1.0)
        rx, ry, rz = (o + f * (n - o) for o, n in zip(self.old, self.new))
        s = slice(1, -1)
        for a in (0, -1):
            hz[s, a] += rz[s, a]
            hx[s, a] = rx[s, a]
            hy[s, :, a] += ry[s, :, a]
            hx[s, :, a] = rx[s, :, a]
            hz[a] += rz[a]
            hy[a] += ry[a]

    def step(self, H, HJ):
        st, gr = self.st, self.gr
        if st.open is not None:
            self._open(HJ)
        F = [self._band(mu) for mu in range(st.N)]
        ph = self._field()
        s = slice(1, -1)
        U = []
        for ax in range(3):
            inr = tuple(slice(None) if a == ax else s for a in range(3))
            u = self.U[ax].clone()
            u[inr] = torch.polar(torch.ones_like(ph[ax][inr]), -ph[ax][inr])
            U.append(u)
        d2 = gr.dx * gr.dx
        cx, cy, cz = (v / d2 for v in self._curl(ph))
        hx, hy, hz = (v.clone() for v in self.h)
        hx[s, s, s], hy[s, s, s], hz[s, s, s] = cx[s, s, s], cy[s, s, s], cz[s, s, s]
        self._boundary((hx, hy, hz), H, HJ)
        # covariant Neumann ghosts, x then y then z
        lo, hi = (gr.x1 - 1, gr.y1 - 1, gr.z1 - 1), (gr.x2, gr.y2, gr.z2)
        for f in F:
            for ax in range(3):
                rng = [slice(l, h + 1) if a < ax else slice(l + 1, h) for a, (l, h) in enumerate(zip(lo, hi))]

                def at(n):
                    q = list(rng)
                    q[ax] = n
                    return tuple(q)
                f[at(lo[ax])] = U[ax][at(lo[ax])] * f[at(lo[ax] + 1)]
                f[at(hi[ax])] = U[ax][at(hi[ax] - 1)].conj() * f[at(hi[ax] - 1)]
        self.G = F
        self.th, self.ph = ph, self.th
        self.V, self.U = U, self.V
        self.h = [hx, hy, hz]

    def fields(self):
        out = {f"G{mu + 1}": g for mu, g in enumerate(self.G)}
        out.update({f"F{mu + 1}": g for mu, g in enumerate(self.G)})
        for k, v in (("th", self.th), ("ph", self.ph), ("U", self.U), ("V", self.V), ("J", self.J), ("h", self.h)):
            out.update({k + a: x for a, x in zip("xyz", v)})
        return {k: v.cpu().numpy() for k, v in out.items()}


def exact(case, seed):
    c = case
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if c["way"] == "batch":
        out = {}
        for q, spec in enumerate(_specs(c, seed)):
            st = stepper_of(spec)
            p = _Plain(st, state_of(spec, st), dev)
            for _ in range(c["cycles"] * LMAX):
                p.step(spec.H, st.selffield(spec.J))
            f = p.fields()
            out[f"run{q}"] = {k: f[k] for k in ("G1", "G2", "thx", "thy", "thz")}
        return dict(out, records=None)
    steps = c["steps"] if c["way"] == "transfer" else c["cycles"] * c.get("lmax", LMAX)
    cells = c["nx"] * c["ny"] * c["nz"]
    if c.get("noise") or c.get("qp") or (c["field"] == "pcg" and steps * cells > 5e7):
        return None
    st, H, J = _stepper(c)
    if any(r == 0 and n != 1 for r, n in zip(st.rkl, st.nsub)):
        return None
    p = _Plain(st, seeded_state(st.model, st.grid, st.masks, H, seed=seed), dev)
    for _ in range(steps):
        p.step(H, st.selffield(J))
    f = p.fields()
    return f if c["way"] == "transfer" else dict(f, records=None)
