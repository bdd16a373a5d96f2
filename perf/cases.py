"""Timed cases of the channel-flow layer, through its public Python entry points.

Every case starts from a seeded flow a run meets in earnest: the laminar
profile plus a few dozen solenoidal modes of about a tenth of the bulk
velocity, made with plain torch.  Kinds of case:

* ``step``      SLChannelFlow.step_sl_bdf2 in its BDF2 steady state (the
                bootstrap step is taken in prepare): what a run does all day.
* ``imex``      SLChannelFlow.step_imex, the Eulerian scheme.
* ``advect``    SLAdvector.advect of the three components.
* ``plugin``    HipSL.departure and gather per component, the calls a solver
                with its own step makes.
* ``stats``     TurbulenceStats.accumulate_statistics of one snapshot.
* ``ensemble``  a few Ensemble.step calls over small uneven members, then
                every member's fields.

``exact`` evaluates the same operations with plain torch in float64.
"""

import math

import torch

from slchannel_amd import HipSL, SLAdvector, SLChannelFlow, TurbulenceStats
from slchannel_amd.ensemble import Ensemble

DEVICE = "cuda"
F64 = torch.float64
EXACT_MOST = 17_000_000  # grid points exact() is evaluated for
COST = {"step": 9.0, "imex": 2.5, "advect": 3.0, "plugin": 5.0, "stats": 0.4}


def _case(kind, nx, ny, nz, **kw):
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "order": 6, "storage": 64, "wall": "channel",
         "cfl": 2.0}
    c.update(kw)
    return c


def listed():
    def named(name, *a, **kw):
        return {"name": name, **_case(*a, **kw)}

    return [
        # the smallest member a serving loop steps: latency and launches
        named("step_32x24x32_o4", "step", 32, 24, 32, order=4),
        # the validation channel: launches and kernels weigh alike
        named("step_64x64x64_o6", "step", 64, 64, 64, cfl=3.0),
        # a half channel with a free-slip top, every length odd
        named("step_135x75x99_o4_open", "step", 135, 75, 99, order=4, wall="open"),
        # the production grid, triquintic interpolation
        named("step_256x256x256_o6", "step", 256, 256, 256, cfl=1.0),
        # tricubic with the fields stored in single precision for the gathers
        named("step_256x192x160_o4_fp32", "step", 256, 192, 160, order=4, storage=32, cfl=1.2),
        # a large box
        named("step_512x512x256_o6", "step", 512, 512, 256, cfl=1.5),
        # the Eulerian scheme on a production grid, at its own small CFL
        named("imex_256x192x192", "imex", 256, 192, 192, cfl=0.25),
        # the reference's advection benchmark grid, tricubic
        named("advect_768x768x180_o4", "advect", 768, 768, 180, order=4),
        # a host solver's departure + gather calls, odd lengths
        named("plugin_161x128x97_o6", "plugin", 161, 128, 97, cfl=3.0),
        # on-the-fly statistics with three extra spectra planes
        named("stats_256x256x256", "stats", 256, 256, 256),
        # a batch of small uneven members, eight steps between read-outs
        named("ensemble_12_small_o6", "ensemble", 48, 32, 48, members=12, steps=8),
    ]


def _cost(c):
    return COST[c["kind"]] * c["nx"] * c["ny"] * c["nz"] * (1.0 if c["order"] == 6 else 0.75)


def draw(rng):
    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        # grids of a production run have many small factors; a third do not
        return n if rng.random() < 0.35 else max(lo, n - n % 4)

    kind = rng.choice(("step", "step", "step", "imex", "advect", "plugin", "stats", "ensemble"))
    order = rng.choice((4, 6))
    # the free-slip top is run with tricubic interpolation (triquintic is unstable there)
    wall = rng.choice(("channel", "open")) if order == 4 else "channel"
    if kind == "ensemble":
        return _case(kind, size(24, 64), size(16, 48), size(24, 64), order=order, cfl=2.0,
                     members=rng.randint(4, 15), steps=rng.choice((4, 8)))
    storage = 32 if kind in ("step", "advect") and rng.random() < 0.25 else 64
    most = _cost(_case("step", 512, 512, 256))
    while True:
        nx = size(24, 768)
        # a fine grid's time step is held by accuracy, not by the CFL number
        cfl = 0.25 if kind == "imex" else round(rng.uniform(1.0, min(3.0, max(1.2, 600.0 / nx))), 2)
        # the box is twice as long as wide: cells at most a few times longer than wide
        c = _case(kind, nx, size(max(16, int(0.4 * nx)), int(1.1 * nx)), size(24, 256),
                  order=order, wall=wall, cfl=cfl, storage=storage)
        if _cost(c) <= most:
            return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _box(c):
    """(Lx, Ly, Lz, gamma, Re, stretching, top wall)"""
    if c["wall"] == "open":
        return 4 * math.pi, 2 * math.pi, 1.0, 1.8, 5600.0, "bottom", "neumann"
    return 4 * math.pi, 2 * math.pi, 2.0, 1.5, 2800.0, "symmetric", "dirichlet"


def _z_tables(c):
    Lx, Ly, Lz, gamma, Re, stretch, top = _box(c)
    nz = c["nz"]
    k = torch.linspace(0, nz, nz + 1, dtype=F64)
    tg = torch.tanh(torch.tensor(gamma, dtype=F64))
    if stretch == "bottom":
        z_f = Lz * (1.0 - torch.tanh(gamma * (1.0 - k / nz)) / tg)
    else:
        z_f = 0.5 * Lz * (1 + torch.tanh(gamma * (2 * k / nz - 1)) / tg)
    zi = 0.5 * (z_f[:-1] + z_f[1:])
    z_c = torch.cat([-zi[:1], zi, (2 * z_f[-1] - zi[-1]).reshape(1)])
    return z_f, z_c


def _dt(c):
    return c["cfl"] * (4 * math.pi / c["nx"]) / 1.6


def _fields(c, seed):
    """Ghost-shaped u, v, w on the GPU: the laminar profile plus solenoidal
    modes, curl of A = sum a cos(kx x + ky y + phase) G_l(z), with G and G'
    zero at the walls."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    Lx, Ly, Lz = _box(c)[:3]
    z_f, z_c = _z_tables(c)
    r = torch.Generator().manual_seed(1000 + int(seed))
    B = 32
    kx = torch.randint(-6, 7, (B,), generator=r).to(F64) * (2 * math.pi / Lx)
    ky = torch.randint(1, 7, (B,), generator=r).to(F64) * (2 * math.pi / Ly)
    lz = torch.randint(1, 5, (B,), generator=r).to(F64) * (math.pi / Lz)
    a = torch.randn(3, B, generator=r, dtype=F64) * (0.25 / math.sqrt(B))
    a = a / torch.sqrt(kx * kx + ky * ky + lz * lz)
    ph = 2 * math.pi * torch.rand(3, B, generator=r, dtype=F64)

    def G(z):
        s, q = math.pi / Lz, z[:, None] * lz
        env = torch.sin(s * z)[:, None] ** 2
        denv = s * torch.sin(2 * s * z)[:, None]
        return env * torch.cos(q), denv * torch.cos(q) - env * lz * torch.sin(q)

    def field(xs, ys, z, terms):
        # terms: (component of A, coefficient per mode, cosine or sine, G or G')
        g, dg = (t.to(DEVICE) for t in G(z))
        ex, ey = (xs[:, None] * kx).to(DEVICE), (ys[:, None] * ky).to(DEVICE)
        out = torch.zeros(len(xs) * len(ys), len(z), dtype=F64, device=DEVICE)
        for comp, coef, fn, deriv in terms:
            t = ex[:, None, :] + ey[None, :, :] + ph[comp].to(DEVICE)
            m = fn(t).reshape(-1, B) * coef.to(DEVICE)
            out.addmm_(m, (dg if deriv else g).t().contiguous())
        return out.reshape(len(xs), len(ys), len(z))

    i = torch.arange(nx + 2, dtype=F64)
    j = torch.arange(ny + 2, dtype=F64)
    xf, xc = i[:-1] * (Lx / nx), (i - 0.5) * (Lx / nx)
    yf, yc = j[:-1] * (Ly / ny), (j - 0.5) * (Ly / ny)
    u = field(xf, yc, z_c, [(2, -a[2] * ky, torch.sin, False), (1, -a[1], torch.cos, True)])
    v = field(xc, yf, z_c, [(0, a[0], torch.cos, True), (2, a[2] * kx, torch.sin, False)])
    w = field(xc, yc, z_f, [(1, -a[1] * kx, torch.sin, False), (0, a[0] * ky, torch.sin, False)])
    zeta = z_c / Lz
    base = 1.5 * zeta * (2 - zeta) if c["wall"] == "open" else 6.0 * zeta * (1 - zeta)
    u += base.to(DEVICE)
    if c["kind"] == "stats":  # plane means of v and w: a skewed profile, wall transpiration
        v += (0.02 * torch.sin(0.5 * math.pi * zeta)).to(DEVICE)
        w += (0.01 * torch.sin(math.pi * z_f / Lz) ** 2).to(DEVICE)
    _ghosts(c, u, v, w)
    return u, v, w


def _ghosts(c, u, v, w):
    """Periodic x and y, no-slip walls (free-slip top of the open channel)."""
    top = 1.0 if c["wall"] == "open" else -1.0
    u[0] = u[-1]
    u[:, 0] = u[:, -2]
    u[:, -1] = u[:, 1]
    v[0] = v[-2]
    v[-1] = v[1]
    v[:, 0] = v[:, -1]
    w[0] = w[-2]
    w[-1] = w[1]
    w[:, 0] = w[:, -2]
    w[:, -1] = w[:, 1]
    for f in (u, v):
        f[:, :, 0] = -f[:, :, 1]
        f[:, :, -1] = top * f[:, :, -2]
    w[:, :, 0] = 0.0
    w[:, :, -1] = 0.0


def _config(c):
    Lx, Ly, Lz, gamma, Re, stretch, top = _box(c)
    return {
        "grid": {"nx": c["nx"], "ny": c["ny"], "nz": c["nz"]},
        "domain": {"Lx": Lx, "Ly": Ly, "Lz": Lz, "stretching_type": stretch},
        "flow": {"Re": Re, "U_bulk": 1.0, "gamma": gamma},
        "boundary_conditions": {"top_wall": {"type": top}},
        "sl": {"interp_order": c["order"],
               "interp_dtype": "fp32_accum64" if c["storage"] == 32 else "fp64"},
    }


def _advector(c):
    Lx, Ly, Lz, gamma, Re, stretch, top = _box(c)
    z_f, z_c = _z_tables(c)
    return SLAdvector(c["nx"], c["ny"], c["nz"], Lx / c["nx"], Ly / c["ny"], Lx, Ly, Lz, z_f, z_c,
                      gamma, stretching_type=stretch, order=c["order"], top_wall_bc_type=top,
                      interp_dtype="fp32_accum64" if c["storage"] == 32 else "fp64", device=DEVICE)


def _members(c):
    """Sizes around the case's own, as a batch of served requests has them."""
    out = []
    for m in range(c["members"]):
        s = (1.0, 0.75, 1.25)[m % 3]
        out.append(dict(c, kind="step", nx=int(c["nx"] * s), ny=int(c["ny"] * s),
                        nz=max(12, int(c["nz"] * (1.0, 1.25, 0.75)[m // 3 % 3]))))
    return out


STAT_PROFILES = ("U_sum", "uu_sum", "vv_sum", "ww_sum", "uw_sum", "Vm_sum", "Wm_sum", "Um2_sum",
                 "Vm2_sum", "Wm2_sum", "UmWm_sum")
STAT_SPECTRA = ("uu", "vv", "ww", "uw")
STAT_PLANES = (5.0, 30.0, 60.0)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "ensemble":
        ens = Ensemble(order=c["order"], device=DEVICE)
        ids = []
        for m, mc in enumerate(_members(c)):
            f = _fields(mc, 100 * seed + m)
            ids.append(ens.add(_config(mc), _dt(mc), fields=f))
        ens.step()  # the members' bootstrap
        return {"kind": kind, "ens": ens, "ids": ids, "steps": c["steps"]}
    u, v, w = _fields(c, seed)
    if kind in ("step", "imex"):
        flow = SLChannelFlow(config=_config(c), device=DEVICE)
        flow.set_fields(u, v, w)
        flow.project_initial()
        step = flow.step_sl_bdf2 if kind == "step" else flow.step_imex
        step(_dt(c))
        return {"kind": kind, "flow": flow, "dt": _dt(c)}
    if kind == "advect":
        return {"kind": kind, "adv": _advector(c), "f": (u, v, w), "dt": _dt(c)}
    if kind == "plugin":
        hip = HipSL(_advector(c))
        hip.set_mid(u, v, w)
        return {"kind": kind, "hip": hip, "f": (u, v, w), "dt": _dt(c)}
    Lx, Ly, Lz, gamma, Re, stretch, top = _box(c)
    z_f, z_c = _z_tables(c)
    st = TurbulenceStats(c["nx"], c["ny"], c["nz"], Lx, Ly, Lz, z_c, z_f, z_c[1:] - z_c[:-1],
                         z_f[1:] - z_f[:-1], Lx / c["nx"], Ly / c["ny"], 1.0 / Re, 180.0,
                         device=DEVICE, top_wall_bc_type=top, spectra_z_planes=STAT_PLANES)
    # the running sums the pass adds to, held as a run's output writer does
    sums = [getattr(st, n) for n in STAT_PROFILES]
    sums += [getattr(st, f"E_{s}_2d_sum") for s in STAT_SPECTRA]
    sums += [p["sums"][s] for p in st.extra_planes for s in STAT_SPECTRA]
    return {"kind": kind, "st": st, "f": (u, v, w), "sums": sums}


def run(state):
    kind = state["kind"]
    if kind in ("step", "imex"):
        flow = state["flow"]
        step = flow.step_sl_bdf2 if kind == "step" else flow.step_imex
        u_bulk, forcing = step(state["dt"])
        return [flow.u, flow.v, flow.w, flow.p, u_bulk, forcing]
    if kind == "advect":
        adv, f = state["adv"], state["f"]
        return list(adv.advect(*f, *f, state["dt"])) + [adv.n_clamped_last]
    if kind == "plugin":
        hip, out = state["hip"], []
        hip.nclamp.zero_()
        for comp, f in zip("uvw", state["f"]):
            n = hip.departure(comp, state["dt"])
            out.append(hip.gather(comp, f, n))
        return out + [hip.nclamp]
    if kind == "stats":
        state["st"].accumulate_statistics(*state["f"])
        return state["sums"]
    ens = state["ens"]
    for _ in range(state["steps"]):
        ens.step()
    return [ens.get_fields(m) for m in state["ids"]]


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    c = case
    if c["kind"] == "ensemble":
        parts = [work(m) for m in _members(c)]
        return {k: c["steps"] * sum(p[k] for p in parts) for k in ("bytes", "flops")}
    N = c["nx"] * c["ny"] * c["nz"]
    P = c["order"]
    gather = 2 * (P ** 3 + P ** 2 + P) + 3 * P * (P + 2)
    sample = 3 * 35  # one trajectory point: three trilinear samples and its weights
    solve = 3 * 8  # three z-diffusion back-substitutions
    poisson = 2 * 2.5 * math.log2(c["nx"] * c["ny"]) + 14 + 8 + 12
    if c["kind"] == "step":  # V^n, V^{n-1} in; u, v, w, p out
        return {"bytes": 8.0 * N * 10, "flops": N * (3 * (2 * gather + 3 * sample + 40) + solve + poisson)}
    if c["kind"] == "imex":  # V, previous rhs in; u, v, w, p, rhs out
        return {"bytes": 8.0 * N * 13, "flops": N * (3 * 45 + 3 * 4 + 2 * solve + poisson)}
    if c["kind"] == "advect":  # the fields in, the advected ones out
        return {"bytes": 8.0 * N * 6, "flops": N * 3 * (gather + 2 * sample + 12)}
    if c["kind"] == "plugin":  # as advect, the feet handed over in memory
        return {"bytes": 8.0 * N * (6 + 3 * 6), "flops": N * 3 * (gather + 2 * sample + 12)}
    return {"bytes": 8.0 * N * 3, "flops": N * 25.0}


# ---------------------------------------------------------------------------
# the same operations with plain torch in float64
# ---------------------------------------------------------------------------


class _Grid:
    def __init__(self, c):
        self.c = c
        self.nx, self.ny, self.nz = c["nx"], c["ny"], c["nz"]
        self.Lx, self.Ly, self.Lz, _, Re, _, self.top = _box(c)
        self.nu = 1.0 / Re
        self.dx, self.dy = self.Lx / self.nx, self.Ly / self.ny
        z_f, z_c = (t.to(DEVICE) for t in _z_tables(c))
        self.z_f, self.z_c = z_f, z_c
        self.dzf, self.dzc = z_f[1:] - z_f[:-1], z_c[1:] - z_c[:-1]


def _nodes(g, comp, f):
    """The component's periodic node buffer, its shifts and z nodes."""
    ox, oy = {0: (0, 1), 1: (1, 0), 2: (1, 1)}[comp]
    sx, sy = {0: (0.0, -0.5), 1: (-0.5, 0.0), 2: (-0.5, -0.5)}[comp]
    return f[ox:ox + g.nx, oy:oy + g.ny].contiguous(), sx, sy, g.z_f if comp == 2 else g.z_c


def _interp(g, comp, f, x, y, z, P):
    """Order-P tensor-product Lagrange interpolation at (x, y, clamped z)."""
    F, sx, sy, zn = _nodes(g, comp, f)
    h, NZ = P // 2 - 1, len(zn)
    F = F.reshape(-1)

    def axis(q, shift, n):
        s = q + shift
        b = torch.floor(s)
        t = s - b
        base = b.to(torch.int64) - h
        idx = [torch.remainder(base + m, n) for m in range(P)]
        return idx, [math_prod([t - (q2 - h) for q2 in range(P) if q2 != m])
                     / math.prod(float(m - q2) for q2 in range(P) if q2 != m) for m in range(P)]

    def math_prod(ts):
        out = ts[0]
        for t in ts[1:]:
            out = out * t
        return out

    ix, wx = axis(x / g.dx, sx, g.nx)
    iy, wy = axis(y / g.dy, sy, g.ny)
    m0 = (torch.searchsorted(zn, z, right=True) - 1).clamp(0, NZ - 2)
    k0 = (m0 - h).clamp(0, NZ - P)
    d = [z - zn[k0 + m] for m in range(P)]
    wz = []
    for m in range(P):
        den = math_prod([zn[k0 + m] - zn[k0 + q] for q in range(P) if q != m])
        wz.append(math_prod([d[q] for q in range(P) if q != m]) / den)
    out = torch.zeros_like(x)
    for i in range(P):
        si = torch.zeros_like(x)
        for j in range(P):
            base = (ix[i] * g.ny + iy[j]) * NZ + k0
            sj = torch.zeros_like(x)
            for k in range(P):
                sj += wz[k] * F[base + k]
            si += wy[j] * sj
        out += wx[i] * si
    return out


def _advect(g, comp, F, mid, dt, P):
    """(values at the feet of depth dt, clamped feet) on the interior."""
    i = torch.arange(1, g.nx + 1, dtype=F64, device=DEVICE).reshape(-1, 1, 1)
    j = torch.arange(1, g.ny + 1, dtype=F64, device=DEVICE).reshape(1, -1, 1)
    sx, sy = {0: (0.0, 0.5), 1: (0.5, 0.0), 2: (0.5, 0.5)}[comp]
    za = (g.z_f[1:-1] if comp == 2 else g.z_c[1:-1]).reshape(1, 1, -1)
    shape = (g.nx, g.ny, za.shape[2])
    xa = ((i - sx) * g.dx).expand(shape).reshape(-1)
    ya = ((j - sy) * g.dy).expand(shape).reshape(-1)
    za = za.expand(shape).reshape(-1)
    lo, hi = float(g.z_f[0] + 1e-12 * g.Lz), float(g.z_f[-1] - 1e-12 * g.Lz)
    x, y, z = xa, ya, za
    for _ in range(2):
        zc = z.clamp(lo, hi)
        us, vs, ws = (_interp(g, q, mid[q], x, y, zc, 2) for q in range(3))
        x, y, z = xa - 0.5 * dt * us, ya - 0.5 * dt * vs, (za - 0.5 * dt * ws).clamp(lo, hi)
    x, y, z = 2 * x - xa, 2 * y - ya, 2 * z - za
    n = ((z < lo) | (z > hi)).sum()
    return _interp(g, comp, F, x, y, z.clamp(lo, hi), P).reshape(shape), n


def _inner(g, comp, f):
    return f[1:g.nx + 1, 1:g.ny + 1, 1:(g.nz if comp == 2 else g.nz + 1)]


def _lap_xy(g, comp, f):
    F, _, _, _ = _nodes(g, comp, f)
    # the interior's first node is node 1 of the buffer in a face direction, node 0 in a centre one
    rx, ry = (-1 if comp == 0 else 0), (-1 if comp == 1 else 0)
    F = torch.roll(F, (rx, ry), (0, 1))
    F = F[:, :, 1:(g.nz if comp == 2 else g.nz + 1)]
    d2x = (torch.roll(F, -1, 0) - 2 * F + torch.roll(F, 1, 0)) / g.dx ** 2
    d2y = (torch.roll(F, -1, 1) - 2 * F + torch.roll(F, 1, 1)) / g.dy ** 2
    return g.nu * (d2x + d2y)


def _thomas(a, b, c, d):
    """Tridiagonal systems along the first axis; a, b, c: (n,) or (n, systems)."""
    n = d.shape[0]
    cp, x = [None] * n, d.clone()
    cp[0], x[0] = c[0] / b[0], d[0] / b[0]
    for k in range(1, n):
        den = b[k] - a[k] * cp[k - 1]
        cp[k] = c[k] / den
        x[k] = (d[k] - a[k] * x[k - 1]) / den
    for k in range(n - 2, -1, -1):
        x[k] -= cp[k] * x[k + 1]
    return x


def _zsolve(g, comp, f, dt, theta):
    F = _inner(g, comp, f)
    n = F.shape[2]
    if comp == 2:
        dl, dr, dc = g.dzf[:n], g.dzf[1:n + 1], g.dzc[1:n + 1]
    else:
        dl, dr, dc = g.dzc[:n], g.dzc[1:n + 1], g.dzf
    al = theta * dt * g.nu
    a, c = -al / (dl * dc), -al / (dr * dc)
    b = 1.0 + al * (1.0 / dl + 1.0 / dr) / dc
    a, b, c = a.clone(), b.clone(), c.clone()
    if comp != 2:
        b[0] -= a[0]
        b[-1] += c[-1] if g.top == "neumann" else -c[-1]
    rhs = F
    if theta < 1.0:
        U = f[1:g.nx + 1, 1:g.ny + 1]
        if comp == 2:
            # the scheme's w stencil is centred one face below the unknown
            d2 = torch.empty_like(F)
            d2[:, :, 1:-1] = ((U[:, :, 2:n] - U[:, :, 1:n - 1]) / dr[1:n - 1]
                              - (U[:, :, 1:n - 1] - U[:, :, 0:n - 2]) / dl[1:n - 1]) / dc[1:n - 1]
            d2[:, :, 0] = ((U[:, :, 1] - U[:, :, 0]) / dr[0] - U[:, :, 0] / dl[0]) / dc[0]
            d2[:, :, -1] = (-U[:, :, n - 1] / dr[-1]
                            - (U[:, :, n - 1] - U[:, :, n - 2]) / dl[-1]) / dc[-1]
        else:
            d2 = ((U[:, :, 2:] - F) / dr - (F - U[:, :, :-2]) / dl) / dc
            d2[:, :, 0] = ((U[:, :, 2] - U[:, :, 1]) / dr[0] - 2 * U[:, :, 1] / dl[0]) / dc[0]
            wall = 0.0 if g.top == "neumann" else -2.0 * U[:, :, n] / dr[-1]
            d2[:, :, -1] = (wall - (U[:, :, n] - U[:, :, n - 1]) / dl[-1]) / dc[-1]
        rhs = F + (1.0 - theta) * dt * g.nu * d2
    a[0], c[-1] = 0.0, 0.0
    x = _thomas(a, b, c, rhs.reshape(-1, n).t().contiguous())
    F.copy_(x.t().reshape(F.shape))


def _poisson(g, div):
    nx, ny, nz = g.nx, g.ny, g.nz
    kx = 2 * math.pi * torch.fft.fftfreq(nx, d=g.dx, dtype=F64).to(DEVICE)
    ky = 2 * math.pi * torch.fft.rfftfreq(ny, d=g.dy, dtype=F64).to(DEVICE)
    k2 = (((2 / g.dx) * torch.sin(kx * g.dx / 2))[:, None] ** 2
          + ((2 / g.dy) * torch.sin(ky * g.dy / 2))[None, :] ** 2).reshape(-1)
    cl, cr = 1.0 / (g.dzc[:-1] * g.dzf), 1.0 / (g.dzc[1:] * g.dzf)
    cl, cr = cl.clone(), cr.clone()
    cl[0], cr[-1] = 0.0, 0.0  # Neumann ends
    b = -(cl[:, None] + cr[:, None] + k2[None, :])
    c = cr[:, None].repeat(1, len(k2))
    b[0, 0], c[0, 0] = 1.0, 0.0  # the mean's level
    h = torch.fft.rfft2(div.permute(2, 0, 1).contiguous())
    x = _thomas(cl, b, c, h.reshape(nz, -1))
    p = torch.fft.irfft2(x.reshape(nz, nx, -1), s=(nx, ny)).permute(1, 2, 0)
    full = torch.zeros(nx + 2, ny + 2, nz + 2, dtype=F64, device=DEVICE)
    full[1:-1, 1:-1, 1:-1] = p
    full[0], full[-1] = full[nx], full[1]
    full[:, 0], full[:, -1] = full[:, ny], full[:, 1]
    full[:, :, 0], full[:, :, -1] = full[:, :, 1], full[:, :, nz]
    return full


def _project(g, u, v, w, scale, dt):
    nx, ny, nz = g.nx, g.ny, g.nz
    I, J, K = slice(1, nx + 1), slice(1, ny + 1), slice(1, nz + 1)
    div = ((u[I, J, K] - u[:nx, J, K]) / g.dx + (v[I, J, K] - v[I, :ny, K]) / g.dy
           + (w[I, J, 1:] - w[I, J, :-1]) / g.dzf)
    p = _poisson(g, div / scale)
    u[I, J, K] -= dt * (p[2:, J, K] - p[I, J, K]) / g.dx
    v[I, J, K] -= dt * (p[I, 2:, K] - p[I, J, K]) / g.dy
    w[I, J, 1:nz] -= dt * (p[I, J, 2:nz + 1] - p[I, J, 1:nz]) / g.dzc[1:nz]
    _ghosts(g.c, u, v, w)
    return p


def _bulk(g, u):
    cv = g.dx * g.dy * g.dzf
    return (_inner(g, 0, u) * cv).sum() / (g.Lx * g.Ly * g.Lz)


def _force(g, u, v, w, dt):
    corr = 1.0 - _bulk(g, u)
    _inner(g, 0, u).add_(corr)
    _ghosts(g.c, u, v, w)
    return [_bulk(g, u), corr / dt]


def _finish(g, V, dt, theta, force_dt):
    """Implicit z-diffusion, projection and flux shift of a predictor."""
    _ghosts(g.c, *V)
    for q in range(3):
        _zsolve(g, q, V[q], dt, theta)
    _ghosts(g.c, *V)
    p = _project(g, *V, dt, dt)
    return p, _force(g, *V, force_dt)


def _bdf1(g, V, dt, P):
    new = [torch.zeros_like(f) for f in V]
    for q in range(3):
        _inner(g, q, new[q]).copy_(_advect(g, q, V[q], V, dt, P)[0] + dt * _lap_xy(g, q, V[q]))
    p, bulk = _finish(g, new, dt, 1.0, dt)
    return new, p, bulk


def _bdf2(g, V, Vm, dt, P):
    mid = [2.0 * a - b for a, b in zip(V, Vm)]
    new, dte = [torch.zeros_like(f) for f in V], 2.0 * dt / 3.0
    for q in range(3):
        near, far = _advect(g, q, V[q], mid, dt, P)[0], _advect(g, q, Vm[q], mid, 2 * dt, P)[0]
        rh = 2.0 * _lap_xy(g, q, V[q]) - _lap_xy(g, q, Vm[q])
        _inner(g, q, new[q]).copy_((4.0 * near - far) / 3.0 + dte * rh)
    p, bulk = _finish(g, new, dte, 1.0, dt)
    return new, p, bulk


def _imex_rhs(g, V):
    """nu (d2x + d2y) - div(f V) on the interiors, flux form on the MAC grid."""
    nx, ny, nz = g.nx, g.ny, g.nz
    u, v, w = V
    ue = torch.cat([u, u[1:2]], 0)
    ve = torch.cat([v, v[:, 1:2]], 1)
    I, J, K = slice(1, nx + 1), slice(1, ny + 1), slice(1, nz + 1)
    Ip, Im, Jp, Jm = slice(2, nx + 2), slice(0, nx), slice(2, ny + 2), slice(0, ny)
    Kp, Km = slice(2, nz + 2), slice(0, nz)

    def mean(a, b):
        return 0.5 * (a + b)

    def at(f, i, j, k):
        return f[i, j, k]

    z = 1.0 / g.dzf
    ru = ((mean(at(ue, I, J, K), at(ue, Ip, J, K)) ** 2 - mean(at(ue, Im, J, K), at(ue, I, J, K)) ** 2) / g.dx
          + (mean(at(v, I, J, K), at(v, Ip, J, K)) * mean(at(u, I, J, K), at(u, I, Jp, K))
             - mean(at(v, I, Jm, K), at(v, Ip, Jm, K)) * mean(at(u, I, Jm, K), at(u, I, J, K))) / g.dy
          + (mean(at(w, I, J, K), at(w, Ip, J, K)) * mean(at(u, I, J, K), at(u, I, J, Kp))
             - mean(at(w, I, J, Km), at(w, Ip, J, Km)) * mean(at(u, I, J, Km), at(u, I, J, K))) * z)
    rv = ((mean(at(u, I, J, K), at(u, I, Jp, K)) * mean(at(v, I, J, K), at(v, Ip, J, K))
           - mean(at(u, Im, J, K), at(u, Im, Jp, K)) * mean(at(v, Im, J, K), at(v, I, J, K))) / g.dx
          + (mean(at(ve, I, J, K), at(ve, I, Jp, K)) ** 2 - mean(at(ve, I, Jm, K), at(ve, I, J, K)) ** 2) / g.dy
          + (mean(at(w, I, J, K), at(w, I, Jp, K)) * mean(at(v, I, J, K), at(v, I, J, Kp))
             - mean(at(w, I, J, Km), at(w, I, Jp, Km)) * mean(at(v, I, J, Km), at(v, I, J, K))) * z)
    W, Wp, Wm = slice(1, nz), slice(2, nz + 1), slice(0, nz - 1)
    rw = ((mean(at(u, I, J, W), at(u, I, J, Wp)) * mean(at(w, I, J, W), at(w, Ip, J, W))
           - mean(at(u, Im, J, W), at(u, Im, J, Wp)) * mean(at(w, Im, J, W), at(w, I, J, W))) / g.dx
          + (mean(at(v, I, J, W), at(v, I, J, Wp)) * mean(at(w, I, J, W), at(w, I, Jp, W))
             - mean(at(v, I, Jm, W), at(v, I, Jm, Wp)) * mean(at(w, I, Jm, W), at(w, I, J, W))) / g.dy
          + (mean(at(w, I, J, W), at(w, I, J, Wp)) ** 2 - mean(at(w, I, J, Wm), at(w, I, J, W)) ** 2) / g.dzc[1:nz])
    return [_lap_xy(g, q, V[q]) - r for q, r in enumerate((ru, rv, rw))]


def _imex(g, V, prev, dt):
    rhs = _imex_rhs(g, V)
    for q in range(3):
        r = rhs[q] if prev is None else 1.5 * rhs[q] - 0.5 * prev[q]
        _inner(g, q, V[q]).add_(dt * r)
    p, bulk = _finish(g, V, dt, 0.5, dt)
    return rhs, p, bulk


def _exact_steps(c, seed, steps):
    """[u, v, w, p, u_bulk, forcing] after the bootstrap and `steps` steps."""
    g, V = _Grid(c), list(_fields(c, seed))
    dt, P = _dt(c), c["order"]
    if c["kind"] == "imex":
        _project(g, *V, 1.0, 1.0)
        prev, p, bulk = _imex(g, V, None, dt)
        for _ in range(steps):
            prev, p, bulk = _imex(g, V, prev, dt)
        return V + [p] + bulk
    if not c.get("unprojected"):
        _project(g, *V, 1.0, 1.0)
    Vm = V
    V, p, bulk = _bdf1(g, V, dt, P)
    for _ in range(steps):
        new, p, bulk = _bdf2(g, V, Vm, dt, P)
        V, Vm = new, V
    return V + [p] + bulk


def _exact_stats(c, seed):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    u, v, w = _fields(c, seed)
    ui, vi, wi = u[:, 1:-1, 1:-1], v[1:-1, :, 1:-1], w[1:-1, 1:-1]
    uc, vc, wc = 0.5 * (ui[:-1] + ui[1:]), 0.5 * (vi[:, :-1] + vi[:, 1:]), 0.5 * (wi[:, :, :-1] + wi[:, :, 1:])
    U, V, W = (f.mean((0, 1)) for f in (uc, vc, wc))
    uf, vf = ui[1:] - ui[1:].mean((0, 1)), vi[:, 1:] - vi[:, 1:].mean((0, 1))
    ww = ((wi - wi.mean((0, 1))) ** 2).mean((0, 1))
    wf = wc - W
    out = [U, (uf ** 2).mean((0, 1)), (vf ** 2).mean((0, 1)), 0.5 * (ww[:-1] + ww[1:]),
           ((uc - U) * wf).mean((0, 1)), V, W, U * U, V * V, W * W, U * W]
    Lz, Re = _box(c)[2], _box(c)[4]
    ut = 180.0 / Re / (Lz / 2)
    zc = _z_tables(c)[1][1:-1]

    def fold(E):
        a, b = nx // 2, ny // 2
        return E[1:a + 1, 1:b + 1] + E[nx - a:, 1:b + 1].flip(0)

    for zp in (15.0,) + STAT_PLANES:
        z = zp / Re / ut
        kb, kt = int((zc - z).abs().argmin()), int((zc - (Lz - z)).abs().argmin())
        parts = []
        for k, s in ((kb, 1.0), (kt, -1.0)):
            fu, fv, fw = (torch.fft.rfft2(f) for f in (uf[:, :, k], vf[:, :, k], s * wf[:, :, k]))
            parts.append([fold((x * y.conj()).real) for x, y in ((fu, fu), (fv, fv), (fw, fw), (fu, fw))])
        out += [0.5 * (a + b) / (nx * ny) ** 2 for a, b in zip(*parts)]
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if c["nx"] * c["ny"] * c["nz"] > EXACT_MOST:
        return None
    if kind in ("step", "imex"):
        return _exact_steps(c, seed, 1)
    if kind == "stats":
        return _exact_stats(c, seed)
    if kind == "ensemble":
        out = []
        for m, mc in enumerate(_members(c)):
            r = _exact_steps(dict(mc, unprojected=True), 100 * seed + m, c["steps"])
            out.append(dict(zip("uvwp", r)))
        return out
    g, V = _Grid(c), list(_fields(c, seed))
    vals = [_advect(g, q, V[q], V, _dt(c), c["order"]) for q in range(3)]
    if kind == "plugin":
        return [x for x, _ in vals] + [None]
    out = []
    for q, (x, _) in enumerate(vals):
        f = torch.zeros_like(V[q])
        _inner(g, q, f).copy_(x)
        out.append(f)
    return out + [None]
