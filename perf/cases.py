"""The work a user of this framework has it do, as cases that can be timed and compared.

Every case advances domains by one RK3 time step through the public entry points
(wrf_amd.runtime): the whole step, its graph replay, the per-routine calls a solve_em-shaped
host makes, and batched ensembles.  The state lives in HBM, as a running model keeps it; one
pass is one time step.  The sizes are those of the presets in wrf_amd/grid.py, of the tests
and of bench.py, or generic ones, odd and ragged among them.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from wrf_amd import grid, runtime
from wrf_amd.fields import FIELDS_1D, FIELDS_2D, FIELDS_3D

#: points of a domain that is built on the host as it is; larger ones repeat a smaller tile
HOST_POINTS = 1_500_000
DEVICE = "cuda:0"


# ------------------------------------------------------------------------------- the cases
def _case(name, nx, ny, nz, bc="periodic", passive=0, route="step", pd=0, mixing=0, precision=0, pad=32, members=1):
    """bc: periodic, open, specified, or terrain (hills on hybrid levels, open in x and
    periodic in y); passive: scalars after water vapour; route: step, graph, phases (one call
    per routine, as a solve_em host makes them) or ensemble (nx, ny: the widest member; the
    graph of a batched step); pd: positive-definite transport; mixing: 1 the sixth-order filter and the
    Rayleigh damper, 2 constant-coefficient diffusion, the filter and the implicit w damper;
    pad: rows padded to a multiple of so many points (1: a Fortran host's own rows)."""
    return dict(name=name, nx=nx, ny=ny, nz=nz, bc=bc, passive=passive, route=route, pd=pd, mixing=mixing,
                precision=precision, pad=pad, members=members)


def listed():
    return [
        # the reference's idealised supercell: the smallest domain, where launches and latency count
        _case("supercell_41", 41, 41, 40, bc="open"),
        # a small domain in a tight loop, replayed as a graph (the tests' re-entrancy size)
        _case("small_graph", 48, 40, 20, passive=3, route="graph"),
        # a Fortran host keeps its own unpadded rows and calls routine by routine
        _case("fortran_host", 121, 97, 45, passive=2, route="phases", pad=1),
        # the middle of the range: an ordinary periodic run with water vapour and six scalars
        _case("ordinary_160", 160, 128, 80, passive=6),
        # bench.py's headline workload
        _case("large_400", 400, 400, 80, passive=6),
        # positive-definite transport, the usual choice for moist runs
        _case("positive_definite", 256, 256, 60, passive=3, pd=1),
        # filters and dampers, on ragged sizes
        _case("mixing", 253, 201, 64, passive=1, mixing=2),
        # a nested-forecast style domain with boundary arrays on all four sides
        _case("specified", 200, 150, 50, bc="specified", passive=1),
        # the FP64 column solve (precision mode 1), ragged sizes, a tall column
        _case("precise_tall", 131, 119, 137, passive=1, precision=1),
        # the ensemble preset: 64 uneven open members in one batched graph
        _case("ensemble_64", 256, 256, 50, bc="open", route="ensemble", members=64),
        # the largest: terrain_c4, hills on hybrid levels, open in x, ten scalars
        _case("terrain_1200", 1200, 1200, 80, bc="terrain", passive=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["periodic", "periodic", "open", "graph", "phases", "pd", "mixing", "specified", "precise",
                       "ensemble", "terrain"])
    nz = rng.randint(20, 140)
    points = math.exp(rng.uniform(math.log(20_000), math.log(16_000_000)))
    aspect = math.exp(rng.uniform(math.log(0.4), math.log(2.5)))
    side = math.sqrt(points / nz)
    nx = min(1200, max(17, int(round(side * aspect))))
    ny = min(1200, max(17, int(round(side / aspect))))
    c = _case("", nx, ny, nz, passive=rng.randint(0, 7))
    if kind == "open":
        c["bc"] = "open"
    elif kind == "graph":
        c["route"] = "graph"
    elif kind == "phases":
        c.update(route="phases", pad=rng.choice([1, 4, 32]), bc=rng.choice(["periodic", "open"]))
    elif kind == "pd":
        c.update(pd=1, bc=rng.choice(["periodic", "periodic", "open"]))
    elif kind == "mixing":
        c.update(mixing=rng.randint(1, 2), bc=rng.choice(["periodic", "open"]))
    elif kind == "specified":
        # built on the host, boundary arrays and all
        f = math.sqrt(min(1.0, HOST_POINTS / float(nx * ny * nz)))
        c.update(bc="specified", nx=max(17, int(nx * f)), ny=max(17, int(ny * f)))
    elif kind == "precise":
        c["precision"] = 1
    elif kind == "ensemble":
        c.update(route="ensemble", bc=rng.choice(["open", "periodic"]), members=rng.randint(3, 24), nx=_log_int(rng, 64, 256),
                 ny=_log_int(rng, 64, 256), nz=rng.randint(30, 60), passive=rng.randint(0, 2))
    elif kind == "terrain":
        # a whole number of hills in the periodic direction
        n = max(1, ny // 100)
        c.update(bc="terrain", ny=n * max(40, min(120, ny // n)))
    del c["name"]
    return c


# ------------------------------------------------------------------------------- the states
def _spec(case, nx, ny, seed):
    passive = case["passive"]
    if case["bc"] == "terrain":
        return grid.terrain_c4(nx=nx, ny=ny, nz=case["nz"], n_passive=passive, n_ridges=2, ridge_a=(4000.0, 8000.0), seed=seed,
                               precision_mode=case["precision"], pad_i=case["pad"])
    bc = case["bc"]
    # dx = 1 km, dt = 6 s as large_c1; the ensemble and the smallest domains as supercell_c0
    coarse = nx * ny <= 256 * 256 and bc == "open"
    return grid.DomainSpec(nx=nx, ny=ny, nz=case["nz"], dx=2000.0 if coarse else 1000.0, dy=2000.0 if coarse else 1000.0,
                           dt=12.0 if coarse else 6.0, bc=bc, n_passive=passive, n_bubbles=2, bubble_amp=2.0, seed=seed,
                           precision_mode=case["precision"], pad_i=case["pad"])


def _options(case, cfg):
    if case["pd"]:
        cfg.moist_adv_opt = cfg.scalar_adv_opt = 1
    if case["mixing"] == 1:
        cfg.diff_6th_opt, cfg.damp_opt = 2, 2
    elif case["mixing"] == 2:
        cfg.diff_6th_opt, cfg.damp_opt = 1, 3
        cfg.diff_opt, cfg.km_opt, cfg.khdif, cfg.kvdif = 1, 1, 200.0, 20.0


def _tile(n):
    """The side of the tile that a direction of n points repeats."""
    return n if n <= 120 else -(-n // -(-n // 120))


def _source(n_dom, n_tile, lo, hi, halo, wraps, stag):
    """For each memory index lo..hi of a direction (1-based points), the tile's interior
    point it is a copy of: periodic images, or the edge's own value beyond an open edge."""
    at = np.arange(lo, hi + 1)
    at = (at - 1) % n_dom if wraps else np.clip(at - 1, 0, n_dom - 1 + stag)
    return torch.from_numpy(np.ascontiguousarray(at % n_tile + halo)).to(DEVICE)


_STAG = {"u": (1, 0), "v": (0, 1)}


def _repeat(dom, spec, small):
    """The domain `dom` (on the dims of `small`) grown to the dims of `spec` by repeating its
    interior, on the device; the struct's pointers follow."""
    d, ds = grid.make_dims(spec), dom.dims
    px, py = spec.bcx == "periodic", spec.bcy == "periodic"
    index = {}
    for stag in ((0, 0), (1, 0), (0, 1)):
        index[stag] = (_source(spec.ny, small.ny, d.jms, d.jme, ds.jds - ds.jms, py, stag[1]),
                       _source(spec.nx, small.nx, d.ims, d.ime, ds.ids - ds.ims, px, stag[0]))
    for name, t in dom.t.items():
        if t.dim() == 1:
            continue
        stag = _STAG.get(name[0], (0, 0)) if name in ("u_1", "u_2", "v_1", "v_2") else (0, 0)
        jj, ii = index[stag]
        dom.t[name] = t.index_select(0, jj).index_select(t.dim() - 1, ii)
    _point(dom)
    dom.dims = d


def _point(dom):
    """The struct's pointers at the tensors of dom.t."""
    P = ctypes.POINTER(ctypes.c_float)
    for n in FIELDS_3D + FIELDS_2D + FIELDS_1D:
        setattr(dom.state, n, ctypes.cast(dom.t[n].data_ptr(), P))
    dom.state.a, dom.state.alpha, dom.state.gamma = (dom.t[n].data_ptr() for n in ("a", "alpha", "gamma"))
    for m in range(dom.n_species):
        dom.state.q[m] = ctypes.cast(dom.t["q%d" % m].data_ptr(), P)
        dom.state.q_old[m] = ctypes.cast(dom.t["q_old%d" % m].data_ptr(), P)
        dom.state.q_tend[m] = ctypes.cast(dom.t["q_tend%d" % m].data_ptr(), P)


def _stir(dom, spec, seed):
    """Up- and downdraughts of a few m/s, as a running model has them (the initial states are
    at rest in the vertical), in both time levels, halo included."""
    d = dom.dims
    rng = np.random.Generator(np.random.Philox(seed))
    x = torch.arange(spec.nx, device=DEVICE) / spec.nx * 2.0 * math.pi
    y = torch.arange(spec.ny, device=DEVICE) / spec.ny * 2.0 * math.pi
    z = torch.arange(spec.nz + 1, device=DEVICE) / spec.nz * math.pi
    w = torch.zeros(spec.ny, spec.nz + 1, spec.nx, device=DEVICE)
    for m in range(1, 4):
        a, b = (torch.sin(m * r + rng.uniform(0.0, 2.0 * math.pi)) for r in (x, y))
        w += 2.0 * b[:, None, None] * torch.sin(z)[None, :, None] * a[None, None, :]
    w[:, 0] = w[:, -1] = 0.0
    jj = _source(spec.ny, spec.ny, d.jms, d.jme, 0, spec.bcy == "periodic", 0)
    ii = _source(spec.nx, spec.nx, d.ims, d.ime, 0, spec.bcx == "periodic", 0)
    for n in ("w_1", "w_2"):
        dom.t[n].copy_(w.index_select(0, jj).index_select(2, ii))


def _domain(case, nx, ny, seed):
    spec = _spec(case, nx, ny, seed)
    if nx * ny * spec.nz <= HOST_POINTS or spec.bc == "specified":
        hs = grid.build_initial_state(spec)
        if spec.bc == "specified":
            grid.build_lbc(hs, seed=seed, value_noise=0.0, tend_scale=1e-8)
        _options(case, hs.cfg)
        dom = runtime.DeviceDomain(hs, device=DEVICE)
        if spec.sounding == "wk":
            _stir(dom, spec, seed)
        return dom
    small = _spec(case, _tile(nx), _tile(ny), seed)
    # the tile itself is doubly periodic, so that its copies fit together
    small.bc = small.bc_x = small.bc_y = "periodic"
    dom = runtime.DeviceDomain(grid.build_initial_state(small), device=DEVICE)
    if spec.sounding == "wk":
        _stir(dom, small, seed)
    _repeat(dom, spec, small)
    dom.cfg = grid.make_config(spec)
    _options(case, dom.cfg)
    return dom


def _member_sizes(case):
    """Uneven members: the widest first, then sizes spread between a quarter of it and all."""
    rng = np.random.Generator(np.random.Philox(1004))
    part = (0.25, 0.375, 0.5, 0.75, 1.0)
    out = [(case["nx"], case["ny"])]
    while len(out) < case["members"]:
        a, b = rng.choice(part, size=2)
        out.append((max(17, int(case["nx"] * a)), max(17, int(case["ny"] * b))))
    return out


_NAMES = ("u_2", "v_2", "w_2", "t_2", "ph_2", "mu_2", "p", "al")


def _window(dom, name):
    """The domain's own points of a field: no halo, no padding."""
    d, t = dom.dims, dom.t[name]
    nj = d.jde - d.jds + (1 if name == "v_2" else 0)
    ni = d.ide - d.ids + (1 if name == "u_2" else 0)
    j, i = slice(d.jds - d.jms, d.jds - d.jms + nj), slice(d.ids - d.ims, d.ids - d.ims + ni)
    if t.dim() == 2:
        return t[j, i]
    return t[j, :d.kde if name in ("w_2", "ph_2") else d.kde - 1, i]


class Model:
    """What a user's program holds between steps: the domain (or the ensemble's members), the
    calls of one step, and views of the fields it looks at."""

    def __init__(self, case, seed):
        self.case, self.ensemble = case, None
        if case["route"] == "ensemble":
            self.domains = [_domain(case, nx, ny, seed + 7919 * m) for m, (nx, ny) in enumerate(_member_sizes(case))]
            names = _NAMES + tuple("q%d" % m for m in range(1 + case["passive"]))
            self.out = [self._together(n) for n in names]
            for dom in self.domains:
                _point(dom)
            self.ensemble = runtime.DeviceEnsemble(self.domains)
        else:
            self.domains = [_domain(case, case["nx"], case["ny"], seed)]
            dom = self.domains[0]
            self.out = [_window(dom, n) for n in _NAMES] + [_window(dom, "q%d" % m) for m in range(dom.n_species)]
            self.phases = runtime.step_phases(dom.cfg, dom.scal, dom.n_species, dom.n_moist)

    def _together(self, name):
        """One field of all members in one buffer (each member's part on a 256-byte start)."""
        sizes = [-(-d.t[name].numel() // 64) * 64 for d in self.domains]
        flat = torch.zeros(sum(sizes), dtype=torch.float32, device=DEVICE)
        at = 0
        for dom, n in zip(self.domains, sizes):
            t = dom.t[name]
            dom.t[name] = flat[at:at + t.numel()].view(t.shape).copy_(t)
            at += n
        return flat

    def __del__(self):
        try:
            if self.ensemble is not None:
                self.ensemble.close()
            else:
                self.domains[0].release()
        except Exception:
            pass


def prepare(case, seed):
    return Model(case, seed % (1 << 31))


def run(state):
    route = state.case["route"]
    if route == "ensemble":
        state.ensemble.step(1, graph=True, sync=False)
    elif route == "phases":
        dom = state.domains[0]
        for name, args in state.phases:
            dom.phase(name, *args)
    else:
        state.domains[0].step(1, graph=route == "graph", sync=False)
    return state.out


def _points(case):
    sizes = _member_sizes(case) if case["route"] == "ensemble" else [(case["nx"], case["ny"])]
    return sum(nx * ny for nx, ny in sizes) * case["nz"]


def work(case):
    """Per mass point and step, each field once: read u, v, w, theta, ph, p, al, the base state
    phb, pb, alb, the forcings of u, v, w, ph, theta and the diabatic heating; write both time
    levels of u, v, w, theta, ph, and p, al; per species read q and its tendency, write both
    time levels.  Operations: about 900 per Runge-Kutta substep (fluxes, pressure gradients, the equation
    of state), 180 per acoustic substep (ten of them), 110 per species and Runge-Kutta substep."""
    n, ns = _points(case), 1 + case["passive"]
    return {"bytes": 4.0 * n * (28 + 4 * ns), "flops": float(n) * (3 * 900 + 10 * 180 + 3 * 110 * ns)}


def tolerance(case):
    """Every kernel evaluates the reference's expressions in its order, each rounded once
    (IEEE FP32, no contraction), and the tests compare whole steps with the oracle bit for
    bit: a correct change leaves every bit as it is.  (Another FP32 evaluation of LOG and **
    alone moves w by 6e-3 after one step of the supercell, so a tolerance between two
    roundings would hide almost any mistake.)"""
    return "exact"


# ------------------------------------------------------------------------------- the same step in 64 bits
def _w(x):
    return torch.roll(x, 1, -1)


def _e(x):
    return torch.roll(x, -1, -1)


def _s(x):
    return torch.roll(x, 1, 0)


def _n(x):
    return torch.roll(x, -1, 0)


def _upwind5(q, vel, axis):
    """5th-order upwind face value left of each point along `axis`, times the face velocity."""
    qm3, qm2, qm1, qp1, qp2 = (torch.roll(q, r, axis) for r in (3, 2, 1, -1, -2))
    centred = (37.0 * (q + qm1) - 8.0 * (qp1 + qm2) + (qp2 + qm3)) / 60.0
    return vel * (centred - torch.sign(vel) * ((qp2 - qm3) - 5.0 * (qp1 - qm2) + 10.0 * (q - qm1)) / 60.0)


def _upwind3(qm2, qm1, q0, qp1, vel):
    """3rd-order upwind value at a face below q0, times the velocity (positive toward smaller
    eta, so the upwind side follows -vel)."""
    centred = (7.0 * (q0 + qm1) - (qp1 + qm2)) / 12.0
    return vel * (centred + torch.sign(-vel) * ((qp1 - qm2) - 3.0 * (q0 - qm1)) / 12.0)


class _Exact:
    """One RK3 step of a flat, doubly periodic domain (map factors 1, no rotation, no forcing)
    in float64: arrays (ny, levels, nx) without halo; u at west faces, v at south faces."""

    def __init__(self, dom):
        d, t = dom.dims, dom.t
        nj, ni, nz = d.jde - d.jds, d.ide - d.ids, d.kde - 1
        j, i = slice(d.jds - d.jms, d.jds - d.jms + nj), slice(d.ids - d.ims, d.ids - d.ims + ni)
        wide = lambda n: t[n][j, :nz + 1, i].double()  # noqa: E731
        mass = lambda n: t[n][j, :nz, i].double()  # noqa: E731
        self.nz, self.cfg = nz, dom.cfg
        for n in ("u_2", "v_2", "t_2", "p", "al", "pb", "alb"):
            setattr(self, n, mass(n))
        for n in ("w_2", "ph_2", "phb"):
            setattr(self, n, wide(n))
        self.mu_2, self.mub = (t[n][j, i].double() for n in ("mu_2", "mub"))
        self.q = [mass("q%d" % m) for m in range(dom.n_species)]
        for n in FIELDS_1D:
            setattr(self, n, t[n].double()[:nz + 1])
        for n in ("dt", "dx", "dy", "rdx", "rdy", "cf1", "cf2", "cf3", "cfn", "cfn1", "p_top"):
            setattr(self, n, float(np.float32(dom.scal[n])))
        self.ns = runtime.num_sound_steps(dom.cfg, dom.scal["dt"], dom.scal["dx"], dom.scal["dy"])

    def h(self, mu):
        """c1h mu + c2h at the mass levels."""
        z = self.nz
        return self.c1h[None, :z, None] * mu[:, None, :] + self.c2h[None, :z, None]

    def f(self, mu):
        """c1f mu + c2f at the w levels."""
        return self.c1f[None, :, None] * mu[:, None, :] + self.c2f[None, :, None]

    def lev(self, v, a=0, b=None):
        return v[a:b][None, :, None]

    def scalar(self, q, fx, fy, fz):
        """-div of the face fluxes of q: fx, fy at west and south faces, fz at w levels."""
        z = self.nz
        tend = -self.rdy * (_n(_upwind5(q, fy, 0)) - _upwind5(q, fy, 0))
        tend = tend - self.rdx * (_e(_upwind5(q, fx, 2)) - _upwind5(q, fx, 2))
        vf = torch.zeros_like(fz)
        for k in (1, z - 1):
            vf[:, k] = fz[:, k] * (self.fnm[k] * q[:, k] + self.fnp[k] * q[:, k - 1])
        vf[:, 2:z - 1] = _upwind3(q[:, :z - 3], q[:, 1:z - 2], q[:, 2:z - 1], q[:, 3:z], fz[:, 2:z - 1])
        return tend - self.lev(self.rdnw, 0, z) * (vf[:, 1:] - vf[:, :-1])

    def adv_w(self, w, ru, rv, ww):
        z = self.nz
        to_w = lambda r: torch.cat([torch.zeros_like(r[:, :1]),  # noqa: E731
                                    self.lev(self.fnm, 1, z) * r[:, 1:] + self.lev(self.fnp, 1, z) * r[:, :-1],
                                    (2.0 - self.fnm[z - 1]) * r[:, z - 1:] - self.fnp[z - 1] * r[:, z - 2:z - 1]], 1)
        fx, fy = to_w(ru), to_w(rv)
        tend = -self.rdy * (_n(_upwind5(w, fy, 0)) - _upwind5(w, fy, 0))
        tend = tend - self.rdx * (_e(_upwind5(w, fx, 2)) - _upwind5(w, fx, 2))
        vel = 0.5 * (ww[:, 1:] + ww[:, :-1])              # at the mass level below w level k, k = 1..nz
        vf = 0.5 * vel * (w[:, 1:] + w[:, :-1])
        vf[:, 1:z - 1] = _upwind3(w[:, :z - 2], w[:, 1:z - 1], w[:, 2:z], w[:, 3:], vel[:, 1:z - 1])
        tend[:, 1:z] -= self.lev(self.rdn, 1, z) * (vf[:, 1:] - vf[:, :-1])
        tend[:, z] += 2.0 * self.rdn[z - 1] * vf[:, z - 1]
        tend[:, 0] = 0.0
        return tend

    def pressure_force(self, p, ph, al, alt, mu, muf, cq, php, shift, rd):
        """The four-term pressure gradient at the faces `shift` points to, times cq."""
        z = self.nz
        both = p + shift(p)
        dpn = torch.zeros_like(ph)
        dpn[:, 0] = 0.5 * (self.cf1 * both[:, 0] + self.cf2 * both[:, 1] + self.cf3 * both[:, 2])
        dpn[:, 1:z] = 0.5 * (self.lev(self.fnm, 1, z) * both[:, 1:] + self.lev(self.fnp, 1, z) * both[:, :-1])
        d = lambda x: x - shift(x)  # noqa: E731
        dph = d(ph)
        dp = 0.5 * rd * self.h(muf) * (dph[:, 1:] + dph[:, :-1] + (alt + shift(alt)) * d(p) + (al + shift(al)) * d(self.pb))
        dp = dp + rd * d(php) * (self.lev(self.rdnw, 0, z) * (dpn[:, 1:] - dpn[:, :-1])
                                 - 0.5 * self.lev(self.c1h, 0, z) * (mu + shift(mu))[:, None, :])
        return cq * dp

    def substep(self, rk, dt_rk, dts, nsmall):
        z, g, t0 = self.nz, 9.81, 300.0
        rd, cp = 287.0, 3.5 * 287.0
        lev, rdnw, c1h = self.lev, self.lev(self.rdnw, 0, z), self.lev(self.c1h, 0, z)
        fnm, fnp = self.lev(self.fnm, 1, z), self.lev(self.fnp, 1, z)
        u, v, w, t, ph, mu = self.u_2, self.v_2, self.w_2, self.t_2, self.ph_2, self.mu_2
        mut = self.mub + mu
        muu, muv = 0.5 * (mut + _w(mut)), 0.5 * (mut + _s(mut))
        ru, rv, rw = u * self.h(muu), v * self.h(muv), w * self.f(mut)
        dnw = lev(self.dnw, 0, z)
        div = dnw * (self.rdx * (_e(ru) - ru) + self.rdy * (_n(rv) - rv))
        ww = torch.zeros_like(w)
        ww[:, 1:z] = -torch.cumsum(dnw * c1h * div.sum(1, keepdim=True) + div, 1)[:, :-1]
        qv = self.q[0]
        cqu, cqv = 1.0 / (1.0 + 0.5 * (qv + _w(qv))), 1.0 / (1.0 + 0.5 * (qv + _s(qv)))
        cqw = 0.5 * (qv[:, 1:] + qv[:, :-1])              # w levels 1..nz-1
        alt = self.al + self.alb
        tot = self.phb + ph
        php = 0.5 * (tot[:, 1:] + tot[:, :-1])
        # tendencies
        ru_t = self.scalar(u, 0.5 * (ru + _w(ru)), 0.5 * (rv + _w(rv)), 0.5 * (ww + _w(ww)))
        rv_t = self.scalar(v, 0.5 * (ru + _s(ru)), 0.5 * (rv + _s(rv)), 0.5 * (ww + _s(ww)))
        rw_t = self.adv_w(w, ru, rv, ww)
        t_t = self.scalar(t, ru, rv, ww)
        ru_t = ru_t - self.pressure_force(self.p, ph, self.al, alt, mu, muu, cqu, php, _w, self.rdx)
        rv_t = rv_t - self.pressure_force(self.p, ph, self.al, alt, mu, muv, cqv, php, _s, self.rdy)
        earth = 1.0 / 6370.0e3
        rws = rw[:, 1:] + rw[:, :-1]
        ru_t = ru_t - u * earth * 0.25 * (rws + _w(rws))
        rv_t = rv_t - v * earth * 0.25 * (rws + _s(rws))
        cq1 = 1.0 / (1.0 + cqw)
        top = cqw[:, -1]
        rw_t[:, z] += g * (cq1[:, -1] * 2.0 * self.rdnw[z - 1] * (-self.p[:, z - 1]) - self.c1f[z] * mu
                           - top * cq1[:, -1] * (self.c1f[z] * self.mub + self.c2f[z]))
        rw_t[:, 1:z] += g * (cq1 * lev(self.rdn, 1, z) * (self.p[:, 1:] - self.p[:, :-1]) - lev(self.c1f, 1, z) * mu[:, None, :]
                             - cqw * cq1 * self.f(self.mub)[:, 1:z])
        at_w = lambda x: fnm * x[:, 1:] + fnp * x[:, :-1]  # noqa: E731
        rw_t[:, 1:z] += earth * 0.25 * (at_w(ru + _e(ru)) * at_w(u + _e(u)) + at_w(rv + _n(rv)) * at_w(v + _n(v)))
        # geopotential tendency
        ph_t = torch.zeros_like(ph)
        wd = 0.5 * (ww[:, 1:] + ww[:, :-1]) * rdnw * (tot[:, 1:] - tot[:, :-1])
        ph_t[:, 1:z] -= fnm * wd[:, 1:] + fnp * wd[:, :-1]
        ph_t[:, 1:] += (self.f(mut) * g * w)[:, 1:]
        for vel, muf, shift, rdl, axis in ((v, muv, _n, self.rdy, 0), (u, muu, _e, self.rdx, 2)):
            face = torch.zeros_like(ph)
            face[:, 1:z] = 0.5 * (vel[:, 1:] + vel[:, :-1])
            face[:, z] = self.cfn * vel[:, z - 1] + self.cfn1 * vel[:, z - 2]
            face = face * self.f(muf)
            d1, d2, d3 = (torch.roll(tot, -r, axis) - torch.roll(tot, r, axis) for r in (1, 2, 3))
            ph_t[:, 1:] -= (0.5 * rdl * (shift(face) + face) * (45.0 * d1 - 9.0 * d2 + d3) / 60.0)[:, 1:]
        # to the small step's perturbations
        if rk == 1:
            self.u_1, self.v_1, self.w_1, self.t_1, self.ph_1, self.mu_1 = u, v, w, t, ph, mu
        full1 = self.mub + self.mu_1
        muus, muvs = 0.5 * (full1 + _w(full1)), 0.5 * (full1 + _s(full1))
        us, vs, ws, ts, phs, mus = u, v, w, t, ph, mu
        u = self.h(muus) * self.u_1 - self.h(muu) * us
        v = self.h(muvs) * self.v_1 - self.h(muv) * vs
        t = self.h(full1) * self.t_1 - self.h(mut) * ts
        w = self.f(full1) * self.w_1 - self.f(mut) * ws
        ph, mu, muts, ww1 = self.ph_1 - phs, self.mu_1 - mus, full1, ww
        c2a = cp / (cp - rd) * (self.pb + self.p) / alt
        eps, smdiv, emdiv = (float(np.float32(getattr(self.cfg, n))) for n in ("epssm", "smdiv", "emdiv"))

        def density():
            al = -1.0 / self.h(muts) * (alt * c1h * mu[:, None, :] + rdnw * (ph[:, 1:] - ph[:, :-1]))
            return al, c2a * (alt * (t - c1h * mu[:, None, :] * ts) / (self.h(muts) * (t0 + ts)) - al)

        al, p = density()
        pm1, mudf = p, torch.zeros_like(mu)
        if rk > 1:
            mudf = self.mudf
        ru_m, rv_m, ww_m = torch.zeros_like(u), torch.zeros_like(v), torch.zeros_like(w)
        mass_h, mass_f = self.h(mut), self.f(mut)
        for _ in range(nsmall):
            gx = self.pressure_force(p, ph, al, alt, mu, muu, cqu, php, _w, self.rdx)
            gy = self.pressure_force(p, ph, al, alt, mu, muv, cqv, php, _s, self.rdy)
            u = u + dts * ru_t - dts * gx - c1h * (emdiv * self.dx * (mudf - _w(mudf)))[:, None, :]
            v = v + dts * rv_t - dts * gy - c1h * (emdiv * self.dy * (mudf - _s(mudf)))[:, None, :]
            uf, vf = u + self.h(muu) * us, v + self.h(muv) * vs
            dv = self.rdy * (_n(vf) - vf) + self.rdx * (_e(uf) - uf)
            mudf = (dnw * dv).sum(1)
            old, mu = mu, mu + dts * mudf
            muts, muave = mut + mu, 0.5 * ((1.0 + eps) * mu + (1.0 - eps) * old)
            ww = torch.zeros_like(w)
            ww[:, 1:z] = -torch.cumsum(dnw * (c1h * mudf[:, None, :] + dv), 1)[:, :-1] - ww1[:, 1:z]
            t_old = t
            flux = torch.zeros_like(w)
            flux[:, 1:z] = ww[:, 1:z] * at_w(ts)
            fx, fy = 0.5 * u * (ts + _w(ts)), 0.5 * v * (ts + _s(ts))
            t = t + dts * t_t - dts * (self.rdy * (_n(fy) - fy) + self.rdx * (_e(fx) - fx) + rdnw * (flux[:, 1:] - flux[:, :-1]))
            ave = 0.5 * ((1.0 + eps) * t + (1.0 - eps) * t_old)
            ave = (ave + c1h * muave[:, None, :] * t0) / (self.h(muts) * (t0 + ts))
            # the implicit w and geopotential
            tot = phs + self.phb
            wd = 0.5 * (ww[:, 1:] + ww[:, :-1]) * rdnw * (tot[:, 1:] - tot[:, :-1])
            r = dts * (ph_t + 0.5 * g * (1.0 - eps) * w)
            r[:, 1:z] -= dts * (fnm * wd[:, 1:] + fnp * wd[:, :-1])
            r = ph + r / mass_f
            r[:, 0] = 0.0
            both = (1.0 + eps) * (r[:, 1:] - r[:, :-1]) + (1.0 - eps) * (ph[:, 1:] - ph[:, :-1])
            stiff = c2a * rdnw / mass_h
            buoy = c2a * alt * ave
            new = w + dts * rw_t
            rdn = lev(self.rdn, 1, z)
            new[:, 0] = 0.0
            new[:, 1:z] += cq1 * 0.5 * dts * g * rdn * (stiff[:, 1:] * both[:, 1:] - stiff[:, :-1] * both[:, :-1])
            new[:, 1:z] += dts * g * (rdn * (buoy[:, 1:] - buoy[:, :-1]) - lev(self.c1f, 1, z) * muave[:, None, :])
            new[:, z] += -0.5 * dts * g * stiff[:, -1] * self.rdnw[z - 1] * 2.0 * both[:, -1]
            new[:, z] -= dts * g * (2.0 * self.rdnw[z - 1] * buoy[:, -1] + self.c1f[z] * muave)
            cof = (0.5 * dts * g * (1.0 + eps)) ** 2
            wf, gam = [new[:, 0]], torch.zeros_like(mu)
            gams = [gam]
            for k in range(1, z + 1):
                if k < z:
                    cw = cq1[:, k - 1] * cof * self.rdn[k]
                    a = -cw * stiff[:, k - 1] / mass_f[:, k - 1] if k > 1 else torch.zeros_like(mu)
                    b = 1.0 + cw * (stiff[:, k] + stiff[:, k - 1]) / mass_f[:, k]
                    c = -cw * stiff[:, k] / mass_f[:, k + 1]
                else:
                    a = -2.0 * cof * self.rdnw[z - 1] * stiff[:, z - 1] / mass_f[:, z - 1]
                    b = 1.0 + 2.0 * cof * self.rdnw[z - 1] * stiff[:, z - 1] / mass_f[:, z]
                    c = torch.zeros_like(mu)
                alpha = 1.0 / (b - a * gam)
                wf.append((new[:, k] - a * wf[-1]) * alpha)
                gam = c * alpha
                gams.append(gam)
            for k in range(z - 1, 0, -1):
                wf[k] = wf[k] - gams[k] * wf[k + 1]
            w = torch.stack(wf, 1)
            ph = torch.cat([ph[:, :1], (r + 0.5 * dts * g * (1.0 + eps) * w / self.f(muts))[:, 1:]], 1)
            ru_m, rv_m, ww_m = ru_m + u, rv_m + v, ww_m + ww
            al, p = density()
            p, pm1 = p + smdiv * (p - pm1), p
        ru_m = ru_m / nsmall + self.h(muu) * us
        rv_m = rv_m / nsmall + self.h(muv) * vs
        ww_m = ww_m / nsmall + ww1
        self.mudf = mudf
        muus, muvs = 0.5 * (muts + _w(muts)), 0.5 * (muts + _s(muts))
        self.u_2 = (u + us * self.h(muu)) / self.h(muus)
        self.v_2 = (v + vs * self.h(muv)) / self.h(muvs)
        self.w_2 = (w + ws * mass_f) / self.f(muts)
        self.t_2 = (t + ts * mass_h) / self.h(muts)
        self.ph_2, self.mu_2 = ph + phs, mu + mus
        if rk == 1:
            self.q_1 = list(self.q)
        old, now = self.h(self.mu_1 + self.mub), self.h(self.mu_2 + self.mub)
        self.q = [(old * q1 + dt_rk * self.scalar(q, ru_m, rv_m, ww_m)) / now for q, q1 in zip(self.q, self.q_1)]
        # the equation of state
        pf = self.c3f[None, :, None] * muts[:, None, :] + self.c4f[None, :, None] + self.p_top
        pm = lev(self.c3h, 0, z) * muts[:, None, :] + lev(self.c4h, 0, z) + self.p_top
        tot = self.ph_2 + self.phb
        alt = (tot[:, 1:] - tot[:, :-1]) / pm / torch.log(pf[:, :-1] / pf[:, 1:])
        self.al = alt - self.alb
        self.p = 1.0e5 * (rd * (t0 + self.t_2) / (1.0e5 * alt)) ** (cp / (cp - rd)) - self.pb

    def step(self):
        dts = self.dt / self.ns
        self.substep(1, self.dt / 3.0, self.dt / 3.0, 1)
        self.substep(2, 0.5 * self.dt, dts, self.ns // 2)
        self.substep(3, self.dt, dts, self.ns)
        self.w_2 = self.w_2.clone()
        self.w_2[:, 0] = 0.0




def exact(case, seed):
    """The step in float64 for flat doubly periodic domains without filters (the limiter of
    positive-definite transport is left out: its species have no value here).  The boundary
    rows of open and specified domains, hills and the filters have no second restatement."""
    if case["bc"] != "periodic" or case["mixing"] or case["route"] == "ensemble":
        return None
    dom = _domain(case, case["nx"], case["ny"], seed % (1 << 31))
    x = _Exact(dom)
    x.step()
    u = torch.cat([x.u_2, x.u_2[:, :, :1]], 2)
    v = torch.cat([x.v_2, x.v_2[:1]], 0)
    q = [None if case["pd"] else a for a in x.q]
    return [u, v, x.w_2, x.t_2, x.ph_2, x.mu_2, x.p, x.al] + q
