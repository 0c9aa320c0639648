"""The workloads that the framework's speed is measured on.

listed() names them, draw() gives more of the same ranges, prepare() makes what a program
holds before the call, run() makes one pass through the public entry points and exact()
computes the same outputs with plain torch in 64 bits, without this package.

A pass that updates a field leaves it on the GPU, as a program does that goes on with it:
its links are among the outputs and come to the host when they are looked at.
"""
import math

import numpy as np
import torch

SWEEP_SEED = 11          # Philox seed of every field's own generator
RHO = 0.12               # stout parameter of the smearing and metadynamics configurations
LEVELS = 4               # stout levels of the collective variable
FLOW_EPS = 0.01
SIGMA = 0.36             # width of the links around pure gauge: plaquettes of about 0.59 (beta = 6)


# ---------------------------------------------------------------- the cases

def case(kind, shape, **more):
    t, x, y, z = shape
    return dict(kind=kind, t=t, x=x, y=y, z=z, **more)


def listed():
    return [
        # the correctness configuration: a colour launch has a few thousand links at most
        dict(case("update", (8, 8, 8, 8), schedule=4, beta=5.7), name="update_8_cb4"),
        # the local-update loop of a small production lattice, two colours
        dict(case("update", (16, 16, 16, 16), schedule=2, beta=6.0), name="update_16_cb2"),
        # the headline configuration: HB + 4 OR on 32^4
        dict(case("update", (32, 32, 32, 32), schedule=2, beta=6.0), name="update_32_cb2"),
        # extents with few factors of two, under the main program's four-colour schedule
        dict(case("update", (28, 20, 12, 36), schedule=4, beta=6.0), name="update_ragged_cb4"),
        # local updates with the Luescher-Weisz action
        dict(case("symanzik", (24, 24, 24, 24), beta=4.5), name="symanzik_24"),
        # scale setting: the RK3 Wilson flow of a large field
        dict(case("flow", (32, 32, 32, 32), integrator="rk3", steps=2), name="flow_32_rk3"),
        # cooling a small field of odd extents with Euler steps
        dict(case("flow", (18, 14, 22, 10), integrator="euler", steps=10), name="flow_ragged_euler"),
        # the smeared field that the observables of a measurement are taken on
        dict(case("stout", (48, 24, 24, 24), levels=4), name="stout_48x24"),
        # one call of the main program's Observables()
        dict(case("measure", (32, 32, 32, 32)), name="measure_32"),
        # the metadynamics force: smeared charge forward, its derivative backward
        dict(case("force", (16, 16, 16, 16)), name="force_16"),
        # one HMC trajectory of the thermalisation, without the Metropolis step
        dict(case("hmc", (16, 16, 16, 32), steps=10), name="hmc_16x32"),
        # one parallel-tempering metadynamics step: every replica's trajectory, then swaps
        dict(case("tempering", (8, 8, 8, 8), replicas=16, steps=5), name="tempering_16x8"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, unit, v_lo, v_hi, l_lo, l_hi):
    """Four extents, multiples of unit, of a volume between v_lo and v_hi."""
    want = math.exp(rng.uniform(math.log(v_lo), math.log(v_hi)))
    for _ in range(200):
        s = [unit * max(1, _log_int(rng, l_lo, l_hi) // unit) for _ in range(4)]
        v = math.prod(s)
        if 0.75 * want <= v <= 1.33 * want and v <= v_hi:
            return tuple(s)
    n = unit * max(1, int(want ** 0.25) // unit)
    return (n, n, n, n)


def draw(rng):
    kind = rng.choice(["update", "update", "symanzik", "flow", "stout", "measure", "force", "hmc", "tempering"])
    if kind == "update":
        schedule = rng.choice([2, 4])
        return case(kind, _shape(rng, schedule, 8 ** 4, 32 ** 4 if schedule == 2 else 24 ** 4, 4, 48), schedule=schedule,
                    beta=round(rng.uniform(5.7, 6.4), 3))
    if kind == "symanzik":
        return case(kind, _shape(rng, 4, 8 ** 4, 20 ** 4, 4, 40), beta=round(rng.uniform(4.0, 5.0), 3))
    if kind == "flow":
        return case(kind, _shape(rng, 2, 8 ** 4, 30 ** 4, 4, 48), integrator=rng.choice(["rk3", "rk3", "euler"]),
                    steps=rng.randint(1, 4))
    if kind == "stout":
        return case(kind, _shape(rng, 2, 8 ** 4, 24 ** 4, 4, 48), levels=rng.randint(1, 6))
    if kind == "measure":
        return case(kind, _shape(rng, 2, 10 ** 4, 30 ** 4, 8, 48))
    if kind == "force":
        return case(kind, _shape(rng, 2, 8 ** 4, 16 ** 4, 4, 24))
    if kind == "hmc":
        return case(kind, _shape(rng, 2, 8 ** 4, 18 ** 4, 4, 32), steps=rng.randint(8, 14))
    return case(kind, _shape(rng, 2, 6 ** 4, 8 ** 4, 4, 16), replicas=rng.randint(2, 16), steps=rng.randint(3, 6))


def shape_of(c):
    return (c["t"], c["x"], c["y"], c["z"])


# ---------------------------------------------------------------- what a pass cannot do without

ROWS2 = 132 + 42                 # two rows of a 3x3 product, the third as their cross product
LINK = 96                        # bytes of an SU(3) link in two rows
PLAQ_STAPLE = 12 * ROWS2         # six terms of two products
RECT_STAPLE = 72 * ROWS2         # eighteen terms of four products
SUBGROUPS = 3 * 160 + 120        # three SU(2) steps and the reunitarisation
EXPONENTIAL = 600                # traceless part, exponential, product, reunitarisation


def work(c):
    v = math.prod(shape_of(c))
    n = 4 * v
    k = c["kind"]
    field = n * LINK
    if k == "update":
        return {"bytes": 2 * field, "flops": 5 * n * (PLAQ_STAPLE + SUBGROUPS)}
    if k == "symanzik":
        return {"bytes": 2 * field, "flops": 5 * n * (PLAQ_STAPLE + RECT_STAPLE + SUBGROUPS)}
    if k == "flow":
        stages = c["steps"] * (3 if c["integrator"] == "rk3" else 1)
        return {"bytes": 2 * field, "flops": stages * n * (PLAQ_STAPLE + EXPONENTIAL)}
    if k == "stout":
        return {"bytes": 2 * field, "flops": c["levels"] * n * (PLAQ_STAPLE + EXPONENTIAL)}
    if k == "measure":
        loops = 6 * (4 * 3 * ROWS2 + 2 * 5 * ROWS2 + 3 * 2 * ROWS2)
        return {"bytes": field + n * 144, "flops": v * loops + 8 * n * 198}
    tape = 3 * PLAQ_STAPLE + 4 * EXPONENTIAL
    one_force = n * (LEVELS * (PLAQ_STAPLE + EXPONENTIAL) + LEVELS * tape + 3 * 16 * 198) + 6 * v * 12 * ROWS2
    if k == "force":
        return {"bytes": field + n * 144, "flops": one_force}
    if k == "hmc":
        return {"bytes": 2 * field, "flops": 2 * c["steps"] * n * (PLAQ_STAPLE + EXPONENTIAL)}
    return {"bytes": 2 * c["replicas"] * field, "flops": 2 * c["steps"] * c["replicas"] * one_force}


# ---------------------------------------------------------------- 3x3 matrices in torch

def device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def mul(a, b):
    return a[..., :, 0:1] * b[..., 0:1, :] + a[..., :, 1:2] * b[..., 1:2, :] + a[..., :, 2:3] * b[..., 2:3, :]


def dag(a):
    return a.transpose(-1, -2).conj().resolve_conj()


def trace(a):
    return a[..., 0, 0] + a[..., 1, 1] + a[..., 2, 2]


def unitary(rows):
    """The SU(3) matrix whose rows 0 and 1 come from the given ones by Gram-Schmidt."""
    r0, r1 = rows[..., 0, :], rows[..., 1, :]
    r0 = r0 / (r0.abs() ** 2).sum(-1, keepdim=True).sqrt()
    r1 = r1 - (r1 * r0.conj()).sum(-1, keepdim=True) * r0
    r1 = r1 / (r1.abs() ** 2).sum(-1, keepdim=True).sqrt()
    a, b = (r0[..., 0], r0[..., 1], r0[..., 2]), (r1[..., 0], r1[..., 1], r1[..., 2])
    r2 = torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]], -1).conj()
    return torch.stack([r0, r1, r2.resolve_conj()], -2)


def antihermitian(a):
    """The traceless anti-hermitian part."""
    b = 0.5 * (a - dag(a))
    return b - (trace(b) / 3.0)[..., None, None] * torch.eye(3, dtype=a.dtype, device=a.device)


def exponential(a):
    """exp(a) of a small matrix by its power series."""
    one = torch.eye(3, dtype=a.dtype, device=a.device)
    r = one + a / 24.0
    for k in range(23, 0, -1):
        r = one + mul(a, r) / k
    return r


def at(field, mu, n):
    """field at x + n e_mu; the lattice dimensions are the first four."""
    return torch.roll(field, -n, mu)


# ---------------------------------------------------------------- inputs

def links(c, seed):
    """Links around pure gauge: near-unit matrices of width SIGMA, rotated by a random gauge
    transformation, so that single links are spread over the group while plaquettes are
    those of an equilibrium configuration.  Shape (4, T, X, Y, Z, 3, 3)."""
    shape = shape_of(c)
    gen = torch.Generator(device=device())
    gen.manual_seed(int(seed))

    def gauss(*s):
        return torch.view_as_complex(torch.randn(*s, 2, generator=gen, device=device(), dtype=torch.float64))

    g = unitary(gauss(*shape, 2, 3))
    one = torch.eye(3, dtype=torch.complex128, device=device())
    out = torch.empty(4, *shape, 3, 3, dtype=torch.complex128, device=device())
    for mu in range(4):
        a = gauss(*shape, 3, 3)
        m = unitary((one + SIGMA * antihermitian(a))[..., :2, :])
        out[mu] = mul(mul(g, m), dag(at(g, mu, 1)))
    return out


def to_host(u):
    """The framework's host order: link (site, mu), 18 doubles."""
    return np.ascontiguousarray(torch.view_as_real(u.movedim(0, 4).contiguous()).reshape(-1, 4, 18).cpu().numpy())


# ---------------------------------------------------------------- passes through the framework

_context = []


def context():
    import lettuce_amd as la
    if not _context:
        _context.append(la.Context(0))
    return _context[0]


class Outputs(dict):
    """A pass's numbers and its fields.  The fields are the state's own and stay on the GPU;
    their links come to the host when they are looked at."""

    def __getitem__(self, key):
        v = super().__getitem__(key)
        return v.download() if hasattr(v, "download") else v

    def get(self, key, default=None):
        return self[key] if key in self else default

    def values(self):
        return [self[k] for k in self]

    def items(self):
        return [(k, self[k]) for k in self]


def gauge_field(la, c, seed):
    f = la.GaugeField(context(), shape_of(c))
    f.upload(to_host(links(c, seed)))
    f.set_rng(SWEEP_SEED + int(seed), 0)
    return f


def bias_potential(la):
    return la.MetaBiasPotential(-8.0, 8.0, 800, 0.05, 0.05, 10.0, 1000.0, well_tempered=False)


def prepare(c, seed):
    import lettuce_amd as la
    k, shape, ctx = c["kind"], shape_of(c), context()
    s = {"la": la, "case": c}
    if k == "tempering":
        b = la.ReplicaBatch(ctx, [shape] * c["replicas"], LEVELS, RHO)
        for r in range(c["replicas"]):
            b.field(r).upload(to_host(links(c, 1000 * int(seed) + r)))
            b.set_rng(r, SWEEP_SEED + r + 64 * int(seed), 0)
        b.set_ladder([r / (c["replicas"] - 1) for r in range(c["replicas"])], None, int(seed), 0)
        b.set_bias(bias_potential(la))
        b.use_graph(True)
        s["batch"] = b
        torch.cuda.empty_cache()
        return s
    s["U"] = gauge_field(la, c, seed)
    if k == "symanzik":
        action = la.LuescherWeiszAction(c["beta"])
        s["heatbath"] = la.HeatbathKernel(s["U"], c["beta"], action)
        s["overrelax"] = la.OverrelaxationSubgroupKernel(s["U"], action=action)
    elif k == "flow":
        s["V"] = la.GaugeField(ctx, shape)
        s["flow"] = la.GradientFlowKernel(s["U"], s["V"], c["integrator"], FLOW_EPS)
    elif k == "stout":
        s["V"] = la.GaugeField(ctx, shape)
    elif k == "measure":
        s["chain"] = la.MatrixField(ctx, shape)
        s["action"] = la.LuescherWeiszAction(6.0)
    elif k == "force":
        s["F"] = la.MatrixField(ctx, shape)
        s["cv"] = la.CollectiveVariable(ctx, shape, LEVELS, RHO)
    elif k == "hmc":
        s["P"] = la.MatrixField(ctx, shape)
        s["hmc"] = la.HMCKernel(s["U"], la.GaugeField(ctx, shape), s["P"], "omf2", 6.0, 1.0)
    torch.cuda.empty_cache()
    return s


def run(s):
    la, c = s["la"], s["case"]
    k = c["kind"]
    if k == "update":
        # the loop body: one heatbath and four overrelaxation sweeps, then the plaquette
        p = la.UpdateSweeps(s["U"], c["beta"], 1, 4, 1, c["schedule"])
        return Outputs(plaquette=p, links=s["U"])
    if k == "symanzik":
        la.Iterator.Checkerboard4(s["heatbath"], 1)
        la.Iterator.Checkerboard4(s["overrelax"], 4)
        return Outputs(links=s["U"])
    if k == "flow":
        s["flow"](c["steps"])
        return Outputs(links=s["V"])
    if k == "stout":
        la.StoutSmearingN(s["U"], s["V"], c["levels"], RHO)
        return Outputs(links=s["V"])
    if k == "measure":
        u = s["U"]
        o = la.Observables(u)
        o["symanzik"] = s["action"].ActionNormalized(u)
        o["Q_plaq"] = la.TopChargePlaquette(u)
        o["W2"] = la.WilsonLoop(0, 2, True, u, s["chain"])
        o["W4"] = la.WilsonLoop(2, 4, False, u, s["chain"])
        o["W8"] = la.WilsonLoop(4, 8, False, u, s["chain"])
        p = la.PolyakovLoop(u)
        return Outputs(o, polyakov=np.array([p.real, p.imag]), chain=s["chain"])
    if k == "force":
        q = s["cv"].forward(s["U"])
        s["cv"].backward(1.0, s["F"])
        return Outputs(Q=q, force=s["F"])
    if k == "hmc":
        s["hmc"](c["steps"], metropolis_step=False)
        return Outputs(links=s["U"], momenta=s["P"])
    b = s["batch"]
    b.metad_hmc(c["steps"], 6.0, "omf2", 1.0, update_bias=True, swap="alternate")
    r = b.results()
    out = Outputs(accepted=r["accepted"], cv=r["cv"], labels=r["labels"], samples=b.samples())
    for i in range(c["replicas"]):
        out["links%d" % i] = b.field(i)
    return out


# ---------------------------------------------------------------- the same in plain torch, 64 bits

PLANES = [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)]


def plaquette_staple(u, mu):
    s = 0
    for nu in range(4):
        if nu == mu:
            continue
        un = u[nu]
        s = s + mul(mul(un, at(u[mu], nu, 1)), dag(at(un, mu, 1)))
        s = s + at(mul(dag(un), mul(u[mu], at(un, mu, 1))), nu, -1)
    return s


def rectangle_staple(u, mu):
    s = 0
    um = u[mu]
    for nu in range(4):
        if nu == mu:
            continue
        un = u[nu]
        unm = at(un, mu, 1)
        two, two_m = mul(un, at(un, nu, 1)), mul(unm, at(unm, nu, 1))    # two steps along nu
        s = s + mul(mul(two, at(um, nu, 2)), dag(two_m))
        s = s + at(mul(mul(dag(two), um), two_m), nu, -2)
        long_ = mul(um, at(um, mu, 1))                                     # two steps along mu
        ahead = mul(mul(un, at(long_, nu, 1)), dag(at(un, mu, 2)))
        ahead = ahead + at(mul(mul(dag(un), long_), at(un, mu, 2)), nu, -1)
        s = s + mul(ahead, dag(at(um, mu, 1))) + at(mul(dag(um), ahead), mu, -1)
    return s


def philox(site, k, sub, mu, stream, seed, counter):
    """Two uniforms per site from Philox4x32-10, key = seed, counter words {site, stream and
    draw, counter low, counter high}."""
    m32 = 0xFFFFFFFF

    def high_low(a, c):
        hi = ((a >> 16) * c + (((a & 0xFFFF) * c) >> 16)) >> 16
        return hi, (a * c) & m32

    x0 = site
    x1 = torch.full_like(site, (stream << 24) | (k << 4) | (sub << 2) | mu)
    x2 = torch.full_like(site, counter & m32)
    x3 = torch.full_like(site, counter >> 32)
    k0, k1 = seed & m32, (seed >> 32) & m32
    for r in range(10):
        h0, l0 = high_low(0xD2511F53, x0)
        h1, l1 = high_low(0xCD9E8D57, x2)
        x0, x1, x2, x3 = h1 ^ x1 ^ k0, l1, h0 ^ x3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32

    def u01(a, b):
        return ((a >> 5).double() * 67108864.0 + (b >> 6).double()) / 9007199254740992.0

    return u01(x0, x1), u01(x2, x3)


def su2_mul(a, b):
    return a[0] * b[0] - a[1] * b[1].conj(), a[0] * b[1] + a[1] * b[0].conj()


def heatbath_su2(v, norm, prefactor, site, sub, mu, seed, counter):
    """Kennedy-Pendleton draws of the sites given, the first accepted of eleven attempts."""
    n = site.numel()
    lam = torch.zeros(n, dtype=torch.float64, device=site.device)
    open_ = torch.arange(n, device=site.device)
    coef = -0.25 * prefactor * norm
    for k in range(11):
        s = site[open_]
        a0, a1 = philox(s, 2 * k, sub, mu, 0, seed, counter)
        b0, b1 = philox(s, 2 * k + 1, sub, mu, 0, seed, counter)
        x2 = torch.cos(2.0 * math.pi * (1.0 - a1))
        l = coef[open_] * (torch.log(1.0 - a0) + x2 * x2 * torch.log(1.0 - b0))
        good = b1 * b1 + l < 1.0
        lam[open_[good]] = l[good]
        open_ = open_[~good]
        if not open_.numel():
            break
    x0 = 1.0 - 2.0 * lam
    size = torch.sqrt(1.0 - x0 * x0)
    phi, ct = philox(site, 0xFFFFF, sub, mu, 0, seed, counter)
    ct = 1.0 - 2.0 * ct
    flat = size * torch.sqrt(1.0 - ct * ct)
    x = torch.complex(x0, flat * torch.cos(2.0 * math.pi * phi)), torch.complex(flat * torch.sin(2.0 * math.pi * phi), size * ct)
    e11, e12 = su2_mul(x, (v[0].conj(), -v[1]))
    e11[open_], e12[open_] = 1.0, 0.0
    return e11, e12


def colours(c, schedule, mu):
    """Colour of every site's link of direction mu."""
    x = [torch.arange(n, device=device()) for n in shape_of(c)]
    s = x[0][:, None, None, None] + x[1][:, None, None] + x[2][:, None] + x[3]
    if schedule == 2:
        return s % 2
    own = [1, 1, 1, 1]
    own[mu] = -1
    return (s + x[mu].reshape(own)) % 4


def sweep(u, c, schedule, staple, heat=None):
    """One sweep in place: overrelaxation, or with heat = (prefactor, seed, counter) heatbath."""
    sites = torch.arange(math.prod(shape_of(c)), device=device())
    for mu in range(4):
        col = colours(c, schedule, mu)
        for k in range(schedule):
            at_k = col == k
            st = staple(u, mu)[at_k]
            link = u[mu][at_k]
            site = sites[at_k.reshape(-1)]
            for sub, (i, j) in enumerate(((0, 1), (0, 2), (1, 2))):
                def w(a, b):
                    return (link[:, a] * st[:, b].conj()).sum(-1)
                a11 = 0.5 * (w(i, i) + w(j, j).conj())
                a12 = 0.5 * (w(i, j) - w(j, i).conj())
                norm = 1.0 / torch.sqrt(a11.abs() ** 2 + a12.abs() ** 2)
                v = norm * a11, norm * a12
                if heat is None:
                    sq = su2_mul(v, v)
                    e11, e12 = sq[0].conj(), -sq[1]
                else:
                    e11, e12 = heatbath_su2(v, norm, heat[0], site, sub, mu, heat[1], heat[2])
                ri = e11[:, None] * link[:, i] + e12[:, None] * link[:, j]
                rj = e11.conj()[:, None] * link[:, j] - e12.conj()[:, None] * link[:, i]
                link = link.clone()
                link[:, i], link[:, j] = ri, rj
            u[mu][at_k] = unitary(link[:, :2])


def plaquette_sum(u):
    return sum(trace(mul(mul(u[m], at(u[n], m, 1)), dag(mul(u[n], at(u[m], n, 1))))).real.sum().item() for m, n in PLANES)


def smear_step(u, coef, z=None, z_coef=0.0, scale=1.0):
    """exp(scale Z) U with Z = coef algebra(staple U^+) + z_coef z; returns U', Z."""
    new = [coef * antihermitian(mul(plaquette_staple(u, mu), dag(u[mu]))) for mu in range(4)]
    if z is not None:
        new = [new[mu] + z_coef * z[mu] for mu in range(4)]
    return [mul(exponential(scale * new[mu]), u[mu]) for mu in range(4)], new


def clover(u, m, n):
    """Sum of the four leaves around every site, minus its adjoint."""
    um, un = u[m], u[n]
    p = mul(mul(um, at(un, m, 1)), dag(mul(un, at(um, n, 1))))            # leaf at x, counted from x
    a = mul(mul(at(un, m, 1), dag(at(um, n, 1))), mul(dag(un), um))         # the same loop from x + m
    b = mul(mul(dag(at(um, n, 1)), dag(un)), mul(um, at(un, m, 1)))         # from x + m + n
    d = mul(mul(dag(un), um), mul(at(un, m, 1), dag(at(um, n, 1))))         # from x + n
    s = p + at(a, m, -1) + at(at(b, m, -1), n, -1) + at(d, n, -1)
    return s - dag(s)


def charge_density(u):
    f = {p: clover(u, *p) for p in PLANES}
    q = 0
    for sign, a, b in ((1, (0, 1), (2, 3)), (-1, (0, 2), (1, 3)), (1, (0, 3), (1, 2))):
        q = q + sign * trace(mul(f[a], f[b])).real
    return q * (-1.0 / (256.0 * math.pi ** 2)), f


def exact_measure(u, c):
    v = math.prod(shape_of(c))
    q, f = charge_density(u)
    e = 0
    for p in PLANES:
        h = -0.125j * f.pop(p)
        h = h - (trace(h) / 3.0)[..., None, None] * torch.eye(3, dtype=h.dtype, device=h.device)
        e = e + trace(mul(h, h)).real
    qt, et = q.sum((1, 2, 3)), e.sum((1, 2, 3)) / v
    plaq = plaquette_sum(u)
    rect, charge, single = 0.0, 0, {}
    for m, n in PLANES:
        um, un = u[m], u[n]
        p = mul(mul(um, at(un, m, 1)), dag(mul(un, at(um, n, 1))))
        single[(m, n)] = -1j * (p - dag(p))
        two_m, two_n = mul(um, at(um, m, 1)), mul(un, at(un, n, 1))
        rect += trace(mul(mul(um, at(two_n, m, 1)), dag(mul(two_n, at(um, n, 2))))).real.sum().item()
        rect += trace(mul(mul(two_m, at(un, m, 2)), dag(mul(un, at(two_m, n, 1))))).real.sum().item()
    for sign, a, b in ((1, (0, 1), (2, 3)), (-1, (0, 2), (1, 3)), (1, (0, 3), (1, 2))):
        charge = charge + sign * trace(mul(single[a], single[b])).real.sum().item()
    out = {"plaquette_sum": plaq, "Q": qt.sum().item(), "E_plaq": 2.0 * (18.0 - plaq / v), "E_clov": et.sum().item(),
           "Q_t": qt.cpu().numpy(), "E_t": et.cpu().numpy(), "Q_plaq": charge / (16.0 * math.pi ** 2)}
    c_rect = -1.0 / 12.0
    out["symanzik"] = ((1.0 - 8.0 * c_rect) * (6.0 * v - plaq / 3.0) + c_rect * (12.0 * v - rect / 3.0)) / (6.0 * v)
    chain = [u[mu] for mu in range(4)]
    have = 1
    for side in (2, 4, 8):
        while have < side:
            chain = [mul(chain[mu], at(u[mu], mu, have)) for mu in range(4)]
            have += 1
        w = sum(trace(mul(mul(chain[m], at(chain[n], m, side)), dag(mul(chain[n], at(chain[m], n, side))))).real.sum().item()
                for m, n in PLANES)
        out["W%d" % side] = 1.0 - w / (18.0 * v)
    out["chain"] = to_host(torch.stack(chain))
    p = u[0][0]
    for t in range(1, c["t"]):
        p = mul(p, u[0][t])
    p = trace(p).mean()
    out["polyakov"] = np.array([p.real.item(), p.imag.item()])
    return out


def exact_force(u):
    u = u.clone().requires_grad_(True)
    w = [u[mu] for mu in range(4)]
    for _ in range(LEVELS):
        w, _z = smear_step(w, RHO)
    q = charge_density(w)[0].sum()
    q.backward()
    force = 0.5 * antihermitian(mul(u.detach(), dag(u.grad)))
    return {"Q": q.item(), "force": to_host(force)}


def momenta(c, seed, counter):
    site = torch.arange(math.prod(shape_of(c)), device=device())
    out = []
    for mu in range(4):
        phi = []
        for k in range(4):
            u0, u1 = philox(site, k, 0, mu, 1, seed, counter)
            r = torch.sqrt(-2.0 * torch.log(1.0 - u0))
            phi += [r * torch.cos(2.0 * math.pi * u1), r * torch.sin(2.0 * math.pi * u1)]
        p1, p2, p3, p4, p5, p6, p7, p8 = phi
        p8 = p8 / math.sqrt(3.0)
        z = torch.zeros_like(p1)
        rows = [z, p3 + p8, p2, p1, p5, p4, -p2, p1, z, p8 - p3, p7, p6, -p5, p4, -p7, p6, z, -2.0 * p8]
        out.append(0.5 * torch.view_as_complex(torch.stack(rows, -1).reshape(*shape_of(c), 3, 3, 2)))
    return out


def exact_hmc(u, c, seed):
    beta, n = 6.0, c["steps"]
    u, p = [u[mu] for mu in range(4)], momenta(c, SWEEP_SEED + int(seed), 0)

    def kick(e):
        for mu in range(4):
            p[mu] = p[mu] + (e * beta / 6.0) * antihermitian(mul(plaquette_staple(u, mu), dag(u[mu])))

    def drift(e):
        for mu in range(4):
            u[mu] = unitary(mul(exponential(e * p[mu]), u[mu])[..., :2, :])

    eps, lam = 1.0 / n, 0.1931833275037836
    kick(lam * eps)
    for i in range(n):
        drift(0.5 * eps)
        kick((1.0 - 2.0 * lam) * eps)
        drift(0.5 * eps)
        kick(lam * eps * (2.0 if i < n - 1 else 1.0))
    return {"links": to_host(torch.stack(u)), "momenta": to_host(torch.stack(p))}


def exact(c, seed):
    k = c["kind"]
    if k == "tempering":
        return None     # every replica's whole trajectory with its smeared force: minutes
    u = links(c, seed)
    if k in ("update", "symanzik"):
        schedule = c.get("schedule", 4)
        if k == "symanzik":
            def staple(w, mu):
                return (1.0 + 8.0 / 12.0) * plaquette_staple(w, mu) - rectangle_staple(w, mu) / 12.0
        else:
            staple = plaquette_staple
        sweep(u, c, schedule, staple, (3.0 / c["beta"], SWEEP_SEED + int(seed), 0))
        for _ in range(4):
            sweep(u, c, schedule, staple)
        out = {"links": to_host(u)}
        if k == "update":
            out["plaquette"] = np.array([plaquette_sum(u)])
        return out
    if k == "flow":
        w = [u[mu] for mu in range(4)]
        for _ in range(c["steps"]):
            if c["integrator"] == "euler":
                w, _z = smear_step(w, FLOW_EPS)
                continue
            w, z = smear_step(w, FLOW_EPS, scale=0.25)
            w, z = smear_step(w, 8.0 / 9.0 * FLOW_EPS, z, -17.0 / 36.0)
            w, z = smear_step(w, 0.75 * FLOW_EPS, z, -1.0)
        return {"links": to_host(torch.stack(w))}
    if k == "stout":
        w = [u[mu] for mu in range(4)]
        for _ in range(c["levels"]):
            w, _z = smear_step(w, RHO)
        return {"links": to_host(torch.stack(w))}
    if k == "measure":
        return exact_measure(u, c)
    if k == "force":
        return exact_force(u)
    return exact_hmc(u, c, seed)
