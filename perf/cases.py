"""Performance cases: what programs on this library spend their time in.

Each case is one pass of a user's program through the public entry points, on
lattices that the program owns as torch tensors and hands over by address (the
C ABI takes plain device pointers).  Kinds of pass:

  sweep       one UpdateLattice (Metropolis and overrelaxation passes) with no
              measurement, with the plaquette summed inside the sweep, or
              followed by the separate plaquette and Polyakov-loop passes of
              the classic run loop; the chain moves on from pass to pass
  ensemble    measured sweeps of a batch of independent replicas
  correlator  Polyakov-loop volume (analytic or stochastic multihit) and its
              correlator C(R)
  multilevel  the two-level multilevel correlator with its per-site field
  fields      lexicographic copy of the lattice and its six plaquette fields

The input links are a random pure gauge plus Gaussian fluctuations, whose mean
plaquette is that of a thermalised lattice at beta = 1 (about 0.58).
`exact` restates the same computations in binary64 on plain torch tensors.
"""
import ctypes
import math

import torch

import latticeu1_amd as u1

PI = math.pi
SIGMA = 0.52  # width of the link fluctuations: <cos P> = exp(-2 SIGMA^2) = 0.58
BENCH = {"proposal": 1, "nhit": 4, "step": 0.5}  # theta + U[-0.5, 0.5), four hits
REFERENCE = {"proposal": 0, "nhit": 1, "step": 0.0}  # an independent angle, one hit
HIT100 = {"proposal": 1, "nhit": 100, "step": 0.5}  # stochastic multihit


def listed():
    return [
        # the smallest lattice anyone runs: a few thousand sites, one sweep and
        # its plaquette per call, all latency and launches
        dict(name="sweep 8^4 f64", **sweep((8, 8, 8, 8), 64, plaq="fused")),
        # the default program: 24^3 x 12, plain Metropolis, then plaquette and
        # Polyakov loop after every sweep
        dict(name="runloop 24^3x12 f64", **sweep((24, 24, 24, 12), 64, plaq="separate", metro=REFERENCE)),
        # decorrelation sweeps of an anisotropic finite-temperature lattice
        dict(name="sweep 24^3x48 xi f32", **sweep((24, 24, 24, 48), 32, beta=2**0.5, xi=2**0.5)),
        # uneven extents: planes and time slices that divide nothing evenly
        dict(name="sweep 28x20x36x22 f32", **sweep((28, 20, 36, 22), 32, plaq="fused")),
        # the headline lattice in both precisions, plaquette after every sweep
        dict(name="sweep 48^4 f32", **sweep((48, 48, 48, 48), 32, plaq="fused")),
        dict(name="sweep 48^4 f64", **sweep((48, 48, 48, 48), 64, plaq="fused")),
        # the largest lattice: 1.4 GB of links, beyond every cache
        dict(name="sweep 96^4 f32", **sweep((96, 96, 96, 96), 32)),
        # a beta scan: 64 replicas of 8^4 ... 24^3 x 32 in one batch
        dict(name="ensemble 64 f32", kind="ensemble", prec=32, nrep=64, sweeps=8, mix=2024),
        # static potential, stochastic multihit with 100 hits per temporal link
        dict(name="corr stoch 24^3x48 f32", **correlator((24, 24, 24, 48), 32, "stochastic", 2**0.5, 2**0.5)),
        # static potential, analytic multihit
        dict(name="corr analytic 32^3x16 f64", **correlator((32, 32, 32, 16), 64, "analytic")),
        # multilevel at 24^4: slabs of four and two slices
        dict(name="multilevel 24^4 f32", **multilevel((24, 24, 24, 24), 32, n4=2, n2=10)),
        # flux-tube analysis: plaquette components per site, lexicographic output
        dict(name="fields 24^4 f64", kind="fields", prec=64, beta=1.0, xi=1.0, spacetime=True, **extents((24,) * 4)),
    ]


def extents(dims):
    return {"nx": dims[0], "ny": dims[1], "nz": dims[2], "nt": dims[3]}


def sweep(dims, prec, plaq="none", metro=BENCH, beta=1.0, xi=1.0, metrop=1, ovrn=3):
    return dict(kind="sweep", prec=prec, plaq=plaq, beta=beta, xi=xi, metrop=metrop, ovrn=ovrn, **metro,
                **extents(dims))


def correlator(dims, prec, mode, beta=1.0, xi=1.0):
    return dict(kind="correlator", prec=prec, mode=mode, beta=beta, xi=xi, **HIT100, **extents(dims))


def multilevel(dims, prec, n4, n2):
    return dict(kind="multilevel", prec=prec, beta=1.0, xi=1.0, n4=n4, n2=n2, metrop=1, ovrn=3, **BENCH,
                **extents(dims))


def draw(rng):
    """One more case: volumes over their logarithm, extents uneven."""

    def dims(vlo, vhi, tmul=2, most=128):
        side = math.exp(rng.uniform(math.log(vlo), math.log(vhi))) ** 0.25
        n = [max(4, min(most, 2 * round(side * math.exp(rng.uniform(-0.35, 0.35)) / 2))) for _ in range(3)]
        return (*n, max(4, tmul * round(side * math.exp(rng.uniform(-0.35, 0.35)) / tmul)))

    beta, xi = round(rng.uniform(0.9, 1.1), 4), rng.choice([1.0, 1.0, round(rng.uniform(0.8, 2.0), 3)])
    prec = rng.choice([32, 64])
    kind = rng.choice(["sweep"] * 6 + ["ensemble", "correlator", "correlator", "multilevel", "fields"])
    if kind == "sweep":
        return sweep(dims(4e3, 3e7 if prec == 32 else 8e6), prec, rng.choice(["none", "fused", "separate"]),
                     rng.choice([BENCH, BENCH, REFERENCE, {"proposal": 1, "nhit": 3, "step": 0.7}]), beta, xi,
                     rng.choice([1, 1, 2]), rng.choice([0, 1, 3, 3, 4]))
    if kind == "ensemble":
        return dict(kind="ensemble", prec=prec, nrep=rng.randint(4, 80), sweeps=rng.randint(1, 8),
                    mix=rng.randint(1, 10**6))
    if kind == "correlator":
        return correlator(dims(4e3, 2e6, most=64), prec, rng.choice(["analytic", "stochastic", "plain"]), beta, xi)
    if kind == "multilevel":
        return multilevel(dims(4e3, 3e5, tmul=4, most=32), prec, rng.randint(1, 3), rng.randint(2, 16))
    return dict(kind="fields", prec=prec, beta=beta, xi=xi, spacetime=rng.choice([True, False]),
                **extents(dims(4e3, 2e6)))


def geometry(case):
    return case["nx"], case["ny"], case["nz"], case["nt"]


def volume(dims):
    return dims[0] * dims[1] * dims[2] * dims[3]


def replicas(case):
    """Extents, couplings, Philox seeds and hot/cold starts of an ensemble."""
    import random

    rng = random.Random(case["mix"])
    shapes = [(8, 8, 8, 8), (12, 12, 12, 16), (16, 16, 16, 16), (16, 16, 16, 32), (24, 24, 24, 32)]
    return [(rng.choice(shapes), rng.uniform(0.9, 1.1), rng.randrange(2)) for _ in range(case["nrep"])]


# ------------------------------------------------------------------ a program
def links(dims, seed, device="cuda"):
    """Input angles (binary64) as full arrays [mu][t, z, y, x]."""
    gen = torch.Generator(device=device).manual_seed(seed)
    shape = tuple(reversed(dims))
    gauge = (torch.rand(shape, generator=gen, device=device, dtype=torch.float64) * 2 - 1) * PI
    out = []
    for mu in range(4):
        noise = torch.randn(shape, generator=gen, device=device, dtype=torch.float64)
        out.append(wrap(gauge - torch.roll(gauge, -1, 3 - mu) + SIGMA * noise))
    return out


def wrap(x):
    return x - 2 * PI * torch.floor((x + PI) / (2 * PI))


def odd_rows(dims, device):
    """(y + z + t) & 1 as [t, z, y, 1]."""
    y, z, t = (torch.arange(n, device=device) for n in dims[1:])
    return ((t[:, None, None] + z[None, :, None] + y[None, None, :]) & 1).bool()[..., None]


def to_eo(full, dims):
    """[mu][t, z, y, x] -> flat even/odd storage lat[mu V + parity V/2 + lex / 2]."""
    odd = odd_rows(dims, full[0].device)
    out = []
    for f in full:
        s = f.reshape(*f.shape[:3], dims[0] // 2, 2)
        out += [torch.where(odd, s[..., 1], s[..., 0]).reshape(-1), torch.where(odd, s[..., 0], s[..., 1]).reshape(-1)]
    return torch.cat(out)


class Buffer:
    """Device memory of a torch tensor, for u1.Lattice."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())


def prec_of(case):
    return u1.F64 if case["prec"] == 64 else u1.F32


def prepare(case, seed):
    u1.init(0)
    if case["kind"] == "ensemble":
        reps = replicas(case)
        ens = u1.Ensemble([u1.geom(d, b) for d, b, _ in reps], [seed * 1000 + i for i in range(len(reps))],
                          [h for _, _, h in reps], prec_of(case), 1, 3, u1.metro(**BENCH))
        ens.sweep_plaquette(2)  # launch shapes and graph settled, as after the first sweeps of a run
        return {"case": case, "ens": ens}
    dims = geometry(case)
    v = volume(dims)
    theta = to_eo(links(dims, seed), dims).to(torch.float64 if case["prec"] == 64 else torch.float32)
    state = {"case": case, "seed": seed, "sweep": 0, "theta": theta,
             "lat": u1.Lattice(u1.geom(dims, case["beta"], case["xi"]), prec_of(case), Buffer(theta))}
    sv = v // dims[3]
    if case["kind"] == "correlator":
        state["P"] = torch.empty(2 * sv, dtype=torch.float64, device="cuda")
    elif case["kind"] == "multilevel":
        state["field"] = torch.empty(2 * sv * (dims[0] // 2) * 3, dtype=torch.float64, device="cuda")
    elif case["kind"] == "fields":
        state["lex"] = torch.empty_like(theta)
        state["field"] = torch.empty(12 * (v if case["spacetime"] else sv), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()  # the library works on a stream of its own
    return state


def metro_of(case):
    return u1.metro(case["proposal"], case["nhit"], case["step"])


def address(tensor):
    return ctypes.c_void_p(tensor.data_ptr())


def doubles(n):
    return (ctypes.c_double * n)()


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ensemble":
        return {"plaquette": state["ens"].sweep_plaquette(case["sweeps"])}
    lat, g = state["lat"], ctypes.byref(state["lat"].g)
    if kind == "sweep":
        args = (case["metrop"], case["ovrn"], metro_of(case), state["seed"], state["sweep"])
        state["sweep"] += 1
        if case["plaq"] == "fused":
            return {"lattice": state["theta"], "plaquette": lat.update_plaquette(*args)}
        lat.update(*args)
        if case["plaq"] == "separate":
            p, loop = lat.plaquette(), lat.polyakov()
            return {"lattice": state["theta"], "plaquette": p,
                    "polyakov": torch.tensor([loop.real, loop.imag], dtype=torch.float64)}
        return {"lattice": state["theta"]}
    if kind == "correlator":
        mode = {"plain": u1.POLY_PLAIN, "analytic": u1.POLY_MULTIHIT, "stochastic": u1.POLY_MULTIHIT_STOCHASTIC}
        rmax = case["nx"] // 2
        corr = doubles(2 * rmax)
        u1.call("u1_poly_volume", g, lat.prec, lat.buf.ptr, mode[case["mode"]], ctypes.byref(metro_of(case)),
                state["seed"], u1.STREAM_MULTIHIT, 0, 0, address(state["P"]))
        u1.call("u1_pp", g, address(state["P"]), rmax, corr)
        return {"P": state["P"], "C": torch.tensor(list(corr), dtype=torch.float64)}
    if kind == "multilevel":
        corr = doubles(2 * (case["nx"] // 2))
        u1.call("u1_multilevel", g, lat.prec, lat.buf.ptr, case["n4"], 1, case["n2"], 1, case["metrop"], case["ovrn"],
                ctypes.byref(metro_of(case)), u1.POLY_MULTIHIT, None, state["seed"], 0, corr,
                address(state["field"]))
        return {"field": state["field"], "C": torch.tensor(list(corr), dtype=torch.float64)}
    means = doubles(12)
    u1.call("u1_convert_layout", g, lat.prec, lat.buf.ptr, address(state["lex"]), 1)
    u1.call("u1_plaquette_fields", g, lat.prec, lat.buf.ptr, 1 if case["spacetime"] else 0, 1,
            address(state["field"]), means)
    return {"lex": state["lex"], "field": state["field"], "means": torch.tensor(list(means), dtype=torch.float64)}


# ---------------------------------------------------------------- bytes, flops
STAPLE = 6 * (4 + 2 + 4)  # six staples: angle sums, sine and cosine, complex sum
HIT = 10  # proposal, sine and cosine, Re(S e^{i theta}), exp, two comparisons


def link_flops(metrop, ovrn, nhit):
    return metrop * (STAPLE + 6 + nhit * HIT) + ovrn * (STAPLE + 6)


def work(case):
    size = case["prec"] // 8
    if case["kind"] == "ensemble":
        v = sum(volume(d) for d, _, _ in replicas(case))
        return {"bytes": case["sweeps"] * 8 * v * size,
                "flops": case["sweeps"] * 4 * v * link_flops(1, 3, BENCH["nhit"])}
    dims = geometry(case)
    v, sv, lat = volume(dims), volume(dims) // dims[3], 4 * volume(dims) * size
    if case["kind"] == "sweep":
        return {"bytes": 2 * lat, "flops": 4 * v * link_flops(case["metrop"], case["ovrn"], case["nhit"])}
    rmax = dims[0] // 2
    if case["kind"] == "correlator":
        link = {"plain": 2, "analytic": STAPLE + 40, "stochastic": STAPLE + case["nhit"] * (HIT + 2)}[case["mode"]]
        read = lat // 4 if case["mode"] == "plain" else lat
        return {"bytes": read + 16 * sv, "flops": v * (link + 6) + sv * 3 * rmax * 8}
    if case["kind"] == "multilevel":
        steps = case["n4"] * case["n2"]
        links_moved = steps * 2.5 * v  # half the slices of spatial links stay frozen
        return {"bytes": lat + 16 * sv * rmax * 3,
                "flops": links_moved * link_flops(case["metrop"], case["ovrn"], case["nhit"])
                + steps * (v * (STAPLE + 40) + sv * rmax * 3 * dims[3] / 2 * 8)}
    return {"bytes": 2 * lat + 96 * (v if case["spacetime"] else sv), "flops": 6 * v * 6}


# ------------------------------------------------------------ binary64 restated
def ahead(f, mu, n=1):
    """f(x + n e_mu)."""
    return torch.roll(f, -n, 3 - mu)


def staple(th, mu, xi):
    """Sum of the six staples of every mu link: real and imaginary part."""
    re = im = 0.0
    for nu in range(4):
        if nu == mu:
            continue
        w = xi if mu == 3 or nu == 3 else 1 / xi
        up = ahead(th[nu], mu) - ahead(th[mu], nu) - th[nu]
        lo = ahead(th[nu] - th[mu] - ahead(th[nu], mu), nu, -1)
        re = re + w * (torch.cos(up) + torch.cos(lo))
        im = im + w * (torch.sin(up) + torch.sin(lo))
    return re, im


def philox(seed, c0, c1, c2, c3):
    """Philox4x32-10 (Salmon et al., SC'11): four words for every link index in c0."""
    mask = 0xFFFFFFFF
    c = [c0] + [torch.full_like(c0, w) for w in (c1, c2, c3)]
    k0, k1 = seed & mask, (seed >> 32) & mask
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57  # low 64 bits of the products
        c = [((p1 >> 32) & mask) ^ c[1] ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ c[3] ^ k1, p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c


def hits(th, sre, sim, index, beta, m, seed, c1, stream, pass_, after=None):
    """nhit Metropolis hits of every link with its staple fixed; after(theta) after each."""
    re = sre * torch.cos(th) - sim * torch.sin(th)
    for h in range(m["nhit"]):
        if h % 2 == 0:
            w = philox(seed, index, c1, stream << 24 | pass_ << 12 | h // 2, 0)
        u, b = (x.to(torch.float64) * 2.0**-32 for x in w[2 * (h % 2):2 * (h % 2) + 2])
        new = PI * (2 * u - 1) if m["proposal"] == 0 else wrap(th + m["step"] * (2 * u - 1))
        re_new = sre * torch.cos(new) - sim * torch.sin(new)
        ok = torch.exp(beta * (re_new - re)) > b
        th, re = torch.where(ok, new, th), torch.where(ok, re_new, re)
        if after:
            after(th)
    return th


def link_index(dims, mu, device):
    """eo + parity V/2 + mu V of every site, and the odd sites, as [t, z, y, x]."""
    v = volume(dims)
    shape = tuple(reversed(dims))
    odd = odd_rows(dims, device) ^ (torch.arange(dims[0], device=device) & 1).bool()
    return (torch.arange(v, device=device).reshape(shape) >> 1) + odd * (v // 2) + mu * v, odd


def sweep_exact(th, case, seed, c1):
    dims = geometry(case)
    passes = [(True, p) for p in range(case["metrop"])] + [(False, p) for p in range(case["ovrn"])]
    for metropolis, p in passes:
        for parity in range(2):
            for mu in range(4):
                sre, sim = staple(th, mu, case["xi"])
                index, odd = link_index(dims, mu, th[0].device)
                if metropolis:
                    new = hits(th[mu], sre, sim, index, case["beta"], case, seed, c1, u1.STREAM_UPDATE, p)
                else:
                    new = wrap(-th[mu] - 2 * torch.atan2(sim, sre))
                th[mu] = torch.where(odd == bool(parity), new, th[mu])


def plaq_angle(th, mu, nu):
    return th[mu] + ahead(th[nu], mu) - ahead(th[mu], nu) - th[nu]


def plaquette_exact(th):
    out = torch.zeros(4, dtype=torch.float64)
    for nu in range(4):
        for mu in range(nu):
            p = plaq_angle(th, mu, nu)
            k = 2 if nu == 3 else 0
            out[k] += (1 - torch.cos(p)).sum().item()
            out[k + 1] -= torch.sin(p).sum().item()
    return (out / (3 * th[0].numel())).numpy()


def multihit_exact(th, case, seed):
    """Temporal links [t, z, y, x]: plain, or their mean with the staple fixed."""
    if case["mode"] == "plain":
        return torch.polar(torch.ones_like(th[3]), th[3])
    sre, sim = staple(th, 3, case["xi"])
    if case["mode"] == "analytic":
        s = torch.sqrt(sre * sre + sim * sim)
        x = case["beta"] * s
        ratio = torch.special.i1e(x) / torch.special.i0e(x) / s
        return torch.complex(ratio * sre, -ratio * sim)
    total = [torch.zeros_like(sre), torch.zeros_like(sre)]

    def add(t):
        total[0] += torch.cos(t)
        total[1] += torch.sin(t)

    index, _ = link_index(geometry(case), 3, sre.device)
    hits(th[3], sre, sim, index, case["beta"], case, seed, 0, u1.STREAM_MULTIHIT, 0, add)
    return torch.complex(total[0] / case["nhit"], total[1] / case["nhit"])


def exact(case, seed):
    """What run returns on a new state, in binary64.  None for an ensemble and
    the multilevel correlator: both are long chaotic chains of updates."""
    if case["kind"] in ("ensemble", "multilevel"):
        return None
    dims = geometry(case)
    device = "cuda" if torch.cuda.is_available() else "cpu"
    th = links(dims, seed, device)
    if case["prec"] == 32:
        th = [t.to(torch.float32).to(torch.float64) for t in th]
    if case["kind"] == "sweep":
        sweep_exact(th, case, seed, 0)
        out = {"lattice": to_eo(th, dims)}
        if case["plaq"] != "none":
            out["plaquette"] = plaquette_exact(th)
        if case["plaq"] == "separate":
            loop = th[3].sum(0)
            out["polyakov"] = torch.stack([torch.cos(loop).mean(), torch.sin(loop).mean()])
        return out
    if case["kind"] == "correlator":
        P = torch.prod(multihit_exact(th, case, seed), 0)
        corr = []
        for r in range(1, dims[0] // 2 + 1):
            c = sum((P * torch.roll(P, -r, d).conj()).sum() for d in range(3)) / (3 * P.numel())
            corr += [c.real.item(), c.imag.item()]
        return {"P": torch.view_as_real(P).reshape(-1), "C": torch.tensor(corr, dtype=torch.float64)}
    pairs = [(0, 3), (1, 3), (2, 3), (1, 2), (2, 0), (0, 1)]
    comps = []
    for mu, nu in pairs:
        p = plaq_angle(th, mu, nu)
        f = torch.complex(1 - torch.cos(p), -torch.sin(p))
        comps.append(f if case["spacetime"] else f.mean(0))
    field = torch.view_as_real(torch.stack(comps)).reshape(-1)
    means = torch.stack([torch.view_as_real(c.mean()) for c in comps]).reshape(-1)
    return {"lex": torch.cat([t.reshape(-1) for t in th]), "field": field, "means": means.cpu()}
