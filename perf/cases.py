"""The work that users of this framework run, as measurable cases.

A case is a plain dict; ``prepare`` builds what a program holds before the call
(links uploaded into a field, an HMC handle, a batch), ``run`` makes one pass
through the public entry points of ``klft_amd``, and ``exact`` computes the same
outputs in 64 bits with plain torch.  Kinds of work:

* ``chain``    n Metropolis sweeps of one lattice, then the observables that the
               run loop measures between sweeps (the per-site plaquette and,
               with ``loops``, temporal and planar Wilson loops);
* ``batch``    n sweeps of many independent chains at once, then every chain's
               plaquette;
* ``ptbc``     n replica steps (a sweep of every replica and the swaps);
* ``traj``     one HMC trajectory with its accept step;
* ``md``       one molecular-dynamics integration without the accept step;
* ``measure``  the plaquette and a block of temporal Wilson loops.

The fields live on the device and a program sees them through measurements, so
a pass returns acceptance rates and the plaquette of every site: each link of
the updated field enters six of those values.  Values that the framework
computes from FP32 links are returned as FP32.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import klft_amd as ka

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
_DIMS = ("L0", "L1", "L2", "L3")


def _chain(name, nc, dims, storage, beta, delta, nhits, n, loops=False):
    c = {"name": name, "kind": "chain", "nd": len(dims), "nc": nc, "storage": storage, "beta": beta,
         "delta": delta, "nhits": nhits, "n": n, "loops": loops}
    c.update(zip(_DIMS, dims))
    return c


def _hmc(name, kind, nc, dims, storage, beta, tau, nsteps):
    c = {"name": name, "kind": kind, "nd": len(dims), "nc": nc, "storage": storage, "beta": beta, "tau": tau,
         "nsteps": nsteps}
    c.update(zip(_DIMS, dims))
    return c


def _measure(name, nc, dims, storage, beta, lmax, tmax):
    c = {"name": name, "kind": "measure", "nd": len(dims), "nc": nc, "storage": storage, "beta": beta,
         "lmax": lmax, "tmax": tmax}
    c.update(zip(_DIMS, dims))
    return c


def listed():
    return [
        # the README's input: U(1) on 8^4, ten sweeps between measurements of
        # the plaquette, four temporal and nine planar loops; latency counts
        _chain("u1_8_f64", 1, (8, 8, 8, 8), "f64", 2.0, 0.1, 10, 10, True),
        # an ordinary lattice of uneven extents, whose sublattices fill no
        # whole number of blocks
        _chain("su2_18x10x14x12_f64", 2, (18, 10, 14, 12), "f64", 2.3, 0.1, 10, 5),
        # the usual SU(3) production lattice of one chain
        _chain("su3_16_f64", 3, (16, 16, 16, 16), "f64", 6.0, 0.1, 10, 5),
        # the headline lattice, plain FP64 method
        _chain("su3_32_f64", 3, (32, 32, 32, 32), "f64", 6.0, 0.1, 10, 4),
        # the headline lattice, compressed FP32 links
        _chain("su3_32_f32rows", 3, (32, 32, 32, 32), "f32_rows", 6.0, 0.1, 10, 6),
        # 64 independent U(1) and SU(2) chains of uneven extents in one batch
        {"name": "batch64_mixed_f32", "kind": "batch", "chains": 64, "group": "u1su2", "storage": "f32", "lo": 8,
         "hi": 20, "pick": 4, "beta0": 1.5, "beta1": 2.5, "delta": 0.1, "nhits": 10, "n": 4},
        # sixteen tempered SU(3) replicas with a 2^3 defect
        {"name": "ptbc16_su3_16_f32", "kind": "ptbc", "chains": 16, "nc": 3, "storage": "f32", "L0": 16, "L1": 16,
         "L2": 16, "L3": 16, "beta": 6.0, "defect": 2, "delta": 0.2, "nhits": 8, "n": 4},
        # HMC of an SU(2) lattice, twenty leapfrog steps
        _hmc("hmc_su2_16_f64", "traj", 2, (16, 16, 16, 16), "f64", 2.3, 1.0, 20),
        # HMC of the headline lattice with a step size that is accepted
        _hmc("hmc_su3_32_f64", "traj", 3, (32, 32, 32, 32), "f64", 6.0, 0.25, 20),
        # the molecular dynamics alone on FP32 links, uneven extents
        _hmc("md_su3_28x24x20x32_f32", "md", 3, (28, 24, 20, 32), "f32", 6.0, 0.25, 20),
        # the measurement of a stored configuration: 64 temporal loops
        _measure("measure_su3_32_f64", 3, (32, 32, 32, 32), "f64", 6.0, 8, 8),
        # the same on FP32 links of a long lattice
        _measure("measure_su3_16x16x24x48_f32", 3, (16, 16, 24, 48), "f32", 6.0, 6, 10),
    ]


_BETA = {1: (1.0, 2.5), 2: (1.8, 2.8), 3: (5.0, 6.5)}
_MAXV = {3: 1 << 19, 2: 1 << 19, 1: 1 << 19}


def _draw_dims(rng, nd, vmin, vmax):
    """nd even extents whose volume is spread over the logarithm of [vmin, vmax]."""
    v = math.exp(rng.uniform(math.log(vmin), math.log(vmax)))
    for _ in range(200):
        side = v ** (1.0 / nd)
        dims = [max(4, 2 * round(0.5 * side * math.exp(rng.uniform(-0.35, 0.35)))) for _ in range(nd)]
        if vmin <= math.prod(dims) <= vmax:
            return dims
    return [2 * max(2, round(0.5 * vmin ** (1.0 / nd)) + 1)] * nd


def draw(rng: random.Random):
    kind = rng.choice(["chain", "chain", "chain", "batch", "ptbc", "traj", "md", "measure"])
    storage = rng.choice(["f64", "f64", "f32", "f32_rows"])
    nc = rng.choice([1, 2, 3, 3])
    nd = rng.choice([2, 3, 4, 4, 4, 4])
    beta = round(rng.uniform(*_BETA[nc]), 2)
    if kind == "chain":
        dims = _draw_dims(rng, nd, 1024, _MAXV[nc])
        c = _chain("", nc, dims, storage, beta, rng.choice([0.05, 0.1, 0.2]), rng.choice([1, 4, 5, 8, 10, 16]),
                   rng.randint(1, 5), nd == 4 and max(dims) <= 24 and rng.random() < 0.3)
    elif kind == "batch":
        c = {"kind": "batch", "chains": rng.randint(2, 48), "group": rng.choice(["u1su2", "su3"]),
             "storage": storage, "lo": 4, "hi": 16, "pick": rng.randrange(1, 1 << 20), "beta0": 1.5, "beta1": 2.5,
             "delta": 0.1, "nhits": rng.choice([4, 8, 10]), "n": rng.randint(1, 5)}
    elif kind == "ptbc":
        dims = [2 * rng.randint(2, 7) for _ in range(4)]
        c = {"kind": "ptbc", "chains": rng.randint(3, 16), "nc": nc, "storage": storage, "beta": beta,
             "defect": rng.choice([1, 2, 3]), "delta": 0.2, "nhits": rng.choice([4, 8, 10]), "n": rng.randint(1, 4)}
        c.update(zip(_DIMS, dims))
    elif kind in ("traj", "md"):
        dims = _draw_dims(rng, 4 if nd == 2 else nd, 2048, _MAXV[nc])
        # the accept step of FP32 links hangs on the last digits of dH
        storage = "f64" if kind == "traj" else rng.choice(["f32", "f32_rows", "f64"])
        c = _hmc("", kind, nc, dims, storage, beta, rng.choice([0.25, 0.5]), rng.randint(10, 24))
    else:
        dims = _draw_dims(rng, max(3, nd), 2048, _MAXV[nc])
        c = _measure("", nc, dims, storage, beta, rng.randint(1, 8), rng.randint(1, 8))
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
# how far the links of a start scatter around the identity: plaquettes near
# those of the ensembles at the betas above
_SPREAD = {1: 0.25, 2: 0.29, 3: 0.22}


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _gen(seed, stream):
    g = torch.Generator(device=_device())
    g.manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _links(nd, nc, dims, gen):
    """SU(N) links scattered around the identity: complex128, (nd, nc, nc, *dims)."""
    dev, s = _device(), _SPREAD[nc]
    U = torch.empty((nd, nc, nc, *dims), dtype=torch.complex128, device=dev)
    for mu in range(nd):
        z = s * torch.randn((max(1, nc - 1), nc, 2, *dims), generator=gen, dtype=torch.float64, device=dev)
        r = [[torch.complex(z[i, j, 0] + (1.0 if i == j else 0.0), z[i, j, 1]) for j in range(nc)]
             for i in range(max(1, nc - 1))]
        _unit(r[0])
        if nc == 2:
            r.append([-r[0][1].conj(), r[0][0].conj()])
        if nc == 3:
            p = sum(r[0][j].conj() * r[1][j] for j in range(3))
            r[1] = [r[1][j] - p * r[0][j] for j in range(3)]
            _unit(r[1])
            r.append(_cross(r[0], r[1]))
        for i in range(nc):
            for j in range(nc):
                U[mu, i, j] = r[i][j]
    return U


def _unit(row):
    n = torch.sqrt(sum(v.real ** 2 + v.imag ** 2 for v in row))
    for j in range(len(row)):
        row[j] = row[j] / n


def _cross(a, b):
    return [(a[(k + 1) % 3] * b[(k + 2) % 3] - a[(k + 2) % 3] * b[(k + 1) % 3]).conj() for k in range(3)]


def _image(U):
    """The host image of a field: complex128, (*dims, nd, nc, nc)."""
    nd = U.dim() - 3
    return U.permute(*range(3, 3 + nd), 0, 1, 2).contiguous().cpu().numpy()


def _dims(case):
    return tuple(case[k] for k in _DIMS[: case.get("nd", 4)])


def _chains(case):
    """(nc, dims, beta) of every chain of a batch."""
    r = random.Random(case["pick"])
    sides = list(range(case["lo"], case["hi"] + 1, 4)) if case["hi"] > 16 else list(range(case["lo"], case["hi"] + 1, 2))
    n, out = case["chains"], []
    for i in range(n):
        nc = 3 if case["group"] == "su3" else 1 + i % 2
        b = case["beta0"] + (case["beta1"] - case["beta0"]) * i / max(1, n - 1)
        out.append((nc, tuple(r.choice(sides) for _ in range(4)), b * 2.6 if nc == 3 else b))
    return out


def _run_seed(seed):
    return (int(seed) * 2654435761 + 32091) & 0x7FFFFFFF


def _momenta(case, dims, seed):
    ng = ka.ngen(case["nc"])
    return torch.randn((case["nd"], ng, *dims), generator=_gen(seed, 2), dtype=torch.float64, device=_device())


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": dict(case), "seed": _run_seed(seed), "at": 0}
    if kind == "batch":
        chains = _chains(case)
        st["batch"] = b = ka.Batch(chains, case["storage"])
        for i, (nc, dims, _) in enumerate(chains):
            b.upload(i, _image(_links(4, nc, dims, _gen(seed, 100 + i))))
        return st
    if kind == "ptbc":
        n, dims = case["chains"], _dims(case)
        c = [1.0 - i / max(1, n - 1) for i in range(n)]
        st["batch"] = b = ka.PTBC(n, case["nc"], dims, case["beta"], case["defect"], (0, 0, 0), c, case["storage"])
        for i in range(n):
            b.upload(i, _image(_links(4, case["nc"], dims, _gen(seed, 100 + i))))
        return st
    dims = _dims(case)
    st["field"] = g = ka.GaugeField(case["nd"], case["nc"], dims, case["storage"])
    g.upload(_image(_links(case["nd"], case["nc"], dims, _gen(seed, 1))))
    if kind == "chain":
        p = ka.MetropolisParams(Ndims=case["nd"], Nd=case["nd"], Nc=case["nc"], nHits=case["nhits"], seed=st["seed"],
                                beta=case["beta"], delta=case["delta"])
        for k, v in zip(_DIMS, dims):
            setattr(p, k, v)
        st["params"] = p
    elif kind in ("traj", "md"):
        st["hmc"] = h = ka.HMC(g, case["beta"], case["tau"], case["nsteps"], st["seed"])
        if kind == "md":
            P = _momenta(case, dims, seed)
            h.set_momenta(P.permute(*range(2, P.dim()), 0, 1).contiguous().cpu().numpy())
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
_TEMPORAL = ((2, 2), (3, 4), (4, 3), (4, 4))
_PLANES = ((0, 1), (1, 2), (3, 2))
_PLANAR = ((2, 2), (3, 3), (4, 3))


def _pairs(case):
    return [(l, t) for l in range(1, case["lmax"] + 1) for t in range(1, case["tmax"] + 1)]


def _site_values(case, v):
    """Per-site values in the precision of the links they come from."""
    return v if case["storage"] == "f64" else v.astype(np.float32)


def _values(case, w):
    return np.array([x[-1] for x in w], dtype=np.float64 if case["storage"] == "f64" else np.float32)


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "chain":
        g, n = st["field"], case["n"]
        rates = ka.metropolis_run(g, st["params"], st["at"], n)
        st["at"] += n
        plaq, site = ka.GaugePlaquette(g, per_site=True)
        out = {"rates": rates, "plaquette": plaq, "site": _site_values(case, site)}
        if case["loops"]:
            out["temporal"] = _values(case, ka.WilsonLoop_temporal(g, _TEMPORAL))
            for mu, nu in _PLANES:
                out["planar%d%d" % (mu, nu)] = _values(case, ka.WilsonLoop_mu_nu(g, mu, nu, _PLANAR))
        return out
    if kind == "batch":
        b, n = st["batch"], case["n"]
        if n > 1:
            b.run(case["nhits"], case["delta"], st["seed"], st["at"], n - 1)
        rates = b.sweep(case["nhits"], case["delta"], st["seed"], st["at"] + n - 1)
        st["at"] += n
        return {"rates": rates, "plaquette": b.plaquette()}
    if kind == "ptbc":
        b, swaps = st["batch"], []
        for _ in range(case["n"]):
            swaps.append(b.step(case["nhits"], case["delta"], st["seed"], st["at"]))
            st["at"] += 1
        return {"swaps": np.stack(swaps), "labels": b.labels(), "plaquette": b.plaquette()}
    g = st["field"]
    if kind == "traj":
        dH, acc = st["hmc"].trajectory(st["at"])
        st["at"] += 1
        plaq, site = ka.GaugePlaquette(g, per_site=True)
        return {"dH": dH, "accepted": int(acc), "plaquette": plaq, "site": site}
    if kind == "md":
        h = st["hmc"]
        h.integrate()
        plaq, site = ka.GaugePlaquette(g, per_site=True)
        return {"kinetic": h.kinetic(), "plaquette": plaq, "site": _site_values(case, site)}
    plaq, site = ka.GaugePlaquette(g, per_site=True)
    return {"plaquette": plaq, "site": _site_values(case, site),
            "temporal": _values(case, ka.WilsonLoop_temporal(g, _pairs(case)))}


# ---------------------------------------------------------------------------
# bytes and operations of one pass
# ---------------------------------------------------------------------------
def _link_bytes(storage, nc):
    comps = nc * nc if storage != "f32_rows" or nc == 1 else (nc - 1) * nc
    return comps * (16 if storage == "f64" else 8)


def _mm(nc):
    """Operations of one complex matrix product."""
    return 8 * nc ** 3


# real operations of one hit: the proposal, Re Tr(r M) and the accept test
_HIT = {1: 30, 2: 90, 3: 300}


def _sweep_work(V, nd, nc, storage, nhits):
    """One sweep: every link read once and written once; per link the staple
    (each of its 2 (nd - 1) terms two products, the first product of an upper
    term shared between two directions), M = S U and the hits."""
    links = V * nd
    terms = 2 * (nd - 1)
    return 2 * links * _link_bytes(storage, nc), links * ((2 * terms - (nd - 1) / 2 + 1) * _mm(nc) + nhits * _HIT[nc])


def _plaq_work(V, nd, nc, storage):
    return V * nd * _link_bytes(storage, nc) + 8 * V, V * nd * (nd - 1) / 2 * (2 * _mm(nc) + 4 * nc * nc)


def _loop_work(V, nc, storage, nplanes, pairs):
    """Lines of every extent, then two products and a trace per loop."""
    ls = len({l for l, _ in pairs})
    return nplanes * 2 * V * _link_bytes(storage, nc), nplanes * V * (ls * _mm(nc) + len(pairs) * (2 * _mm(nc) + 4 * nc * nc))


def work(case):
    kind = case["kind"]
    if kind == "batch":
        parts = [_sweep_work(math.prod(d), 4, nc, case["storage"], case["nhits"]) for nc, d, _ in _chains(case)]
        plaq = [_plaq_work(math.prod(d), 4, nc, case["storage"]) for nc, d, _ in _chains(case)]
        return {"bytes": sum(case["n"] * p[0] + q[0] for p, q in zip(parts, plaq)),
                "flops": sum(case["n"] * p[1] + q[1] for p, q in zip(parts, plaq))}
    V, nd, nc, storage = math.prod(_dims(case)), case.get("nd", 4), case["nc"], case["storage"]
    pb, pf = _plaq_work(V, nd, nc, storage)
    if kind == "ptbc":
        b, f = _sweep_work(V, 4, nc, storage, case["nhits"])
        return {"bytes": case["chains"] * (case["n"] * b + pb), "flops": case["chains"] * (case["n"] * f + pf)}
    if kind == "chain":
        b, f = _sweep_work(V, nd, nc, storage, case["nhits"])
        b, f = case["n"] * b + pb, case["n"] * f + pf
        if case["loops"]:
            for planes, pairs in [(nd - 1, _TEMPORAL)] + [(1, _PLANAR)] * len(_PLANES):
                lb, lf = _loop_work(V, nc, storage, planes, pairs)
                b, f = b + lb, f + lf
        return {"bytes": b, "flops": f}
    if kind == "measure":
        lb, lf = _loop_work(V, nc, storage, nd - 1, _pairs(case))
        return {"bytes": pb + lb, "flops": pf + lf}
    # one MD step: links and momenta read and written, the staples, U S, the
    # exponential (two products) and its product with the link
    mom = ka.ngen(nc) * (8 if storage == "f64" else 4)
    terms = 2 * (nd - 1)
    steps = case["nsteps"] + 1
    b = steps * V * nd * 2 * (_link_bytes(storage, nc) + mom)
    f = steps * V * nd * (2 * terms - (nd - 1) / 2 + 4) * _mm(nc)
    extra = 3 if kind == "traj" else 1
    return {"bytes": b + extra * pb, "flops": f + extra * pf}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits, in plain torch
# ---------------------------------------------------------------------------
# matrices are lists of rows of complex128 tensors over the lattice
def _mul(a, b):
    n = len(a)
    return [[sum(a[i][k] * b[k][j] for k in range(n)) for j in range(n)] for i in range(n)]


def _dag(a):
    n = len(a)
    return [[a[j][i].conj() for j in range(n)] for i in range(n)]


def _add(a, b):
    return [[x + y for x, y in zip(p, q)] for p, q in zip(a, b)]


def _retr(a, b):
    """Re Tr(a b^dagger)."""
    return sum(x.real * y.real + x.imag * y.imag for p, q in zip(a, b) for x, y in zip(p, q))


def _shift(a, mu, k):
    """a(x + k mu)."""
    return [[torch.roll(x, -k, dims=mu) for x in row] for row in a]


def _rows(U, mu):
    return [list(U[mu, i]) for i in range(U.shape[1])]


def _planes(U):
    nd = U.shape[0]
    for mu in range(nd):
        for nu in range(mu + 1, nd):
            a, b = _rows(U, mu), _rows(U, nu)
            yield _retr(_mul(a, _shift(b, mu, 1)), _mul(b, _shift(a, nu, 1)))


def _site_plaquette(U):
    return sum(_planes(U))


def _plaq_out(case, U):
    site = _site_plaquette(U)
    nd, nc = U.shape[0], U.shape[1]
    plaq = float(site.sum()) / (site.numel() * (nd * (nd - 1) // 2) * nc)
    return plaq, _site_values(case, site.reshape(-1).cpu().numpy())


def _loops(U, mu, nu, pairs):
    """Mean Re Tr of the planar loops, per pair, divided by Nc."""
    a, b = _rows(U, mu), _rows(U, nu)
    lines = {}
    for d, links, top in ((0, a, max(l for l, _ in pairs)), (1, b, max(t for _, t in pairs))):
        cur = links
        lines[d, 1] = cur
        for k in range(1, top):
            cur = _mul(cur, _shift(links, (mu, nu)[d], k))
            lines[d, k + 1] = cur
    out = []
    for l, t in pairs:
        f, g = lines[0, l], lines[1, t]
        w = _retr(_mul(f, _shift(g, mu, l)), _mul(g, _shift(f, nu, t)))
        out.append(float(w.mean()) / U.shape[1])
    return out


def _loops_out(case, v):
    return np.array(v, dtype=np.float64 if case["storage"] == "f64" else np.float32)


def _temporal(U, pairs):
    nd = U.shape[0]
    per = [_loops(U, mu, nd - 1, pairs) for mu in range(nd - 1)]
    return [sum(p[i] for p in per) / (nd - 1) for i in range(len(pairs))]


def _staple(U, mu):
    nd, t = U.shape[0], None
    m = _rows(U, mu)
    for nu in range(nd):
        if nu == mu:
            continue
        v = _rows(U, nu)
        up = _mul(_mul(_shift(v, mu, 1), _dag(_shift(m, nu, 1))), _dag(v))
        dn = _shift(_mul(_mul(_dag(_shift(v, mu, 1)), _dag(m)), v), nu, -1)
        t = _add(up, dn) if t is None else _add(t, _add(up, dn))
    return t


# counter-based random words, Philox4x32-10 (Salmon et al., SC'11), the keyed
# streams of the library: counter {c0, c1, c2, tag << 28 | mu << 16 | block}
_M32 = 0xFFFFFFFF


def _mulhilo(m, c):
    lo, hi = c & 0xFFFF, c >> 16
    p0, p1 = m * lo, m * hi  # both below 2^48
    s = p0 + ((p1 & 0xFFFF) << 16)
    return (p1 >> 16) + (s >> 32), s & _M32


def _philox(seed, tag, c0, c1, c2, mu, block):
    c0 = c0.to(torch.int64)
    c1, c2 = torch.full_like(c0, c1), torch.full_like(c0, c2)
    c3 = torch.full_like(c0, (tag << 28) | (mu << 16) | block)
    k0, k1 = seed & _M32, (seed >> 32) & _M32
    for _ in range(10):
        h0, l0 = _mulhilo(0xD2511F53, c0)
        h1, l1 = _mulhilo(0xCD9E8D57, c2)
        c0, c1, c2, c3 = (h1 ^ c1 ^ k0) & _M32, l1, (h0 ^ c3 ^ k1) & _M32, l0
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return [c0, c1, c2, c3]


def _uniforms(seed, tag, site, c1, c2, mu, n):
    """n uniforms of 53 bits from each site's stream."""
    w = []
    for j in range((2 * n + 3) // 4):
        w += _philox(seed, tag, site, c1, c2, mu, j)
    return [((w[2 * i] >> 5).double() * 67108864.0 + (w[2 * i + 1] >> 6).double()) / 9007199254740992.0 for i in range(n)]


def _proposal(nc, u, delta):
    """The proposal matrix of one hit and its accept uniform."""
    if nc == 1:
        th = -delta * math.pi + 2 * delta * math.pi * u[0]
        return [[torch.polar(torch.ones_like(th), th)]], u[1]
    if nc == 2:
        al, z, th = 2 * math.pi * delta * u[0], -1 + 2 * u[1], 2 * math.pi * u[2]
        sa, s = torch.sin(al), torch.sqrt(1 - z * z)
        a = torch.complex(torch.cos(al), z * sa)
        b = torch.complex(s * torch.sin(th) * sa, s * torch.cos(th) * sa)
        return [[a, b], [-b.conj(), a.conj()]], u[3]
    v = [delta * x for x in u]
    r0 = [torch.complex(v[2 * j], v[2 * j + 1]) for j in range(3)]
    _unit(r0)
    r1 = [torch.complex(v[6 + 2 * j], v[7 + 2 * j]) for j in range(3)]
    _unit(r1)
    z = sum(r0[j].conj() * r1[j] for j in range(3))
    r1 = [r1[j] - z * r0[j] for j in range(3)]
    _unit(r1)
    return [r0, r1, _cross(r0, r1)], u[12]


def _restore(a):
    n = len(a)
    if n == 2:
        s = torch.sqrt(sum(v.real ** 2 + v.imag ** 2 for v in a[0]))
        return [[x / s for x in row] for row in a]
    a = [list(r) for r in a]
    _unit(a[0])
    if n == 3:
        _unit(a[1])
        a[2] = _cross(a[0], a[1])
        a[1] = _cross(a[2], a[0])
    return a


def _sweep(U, case, seed, sweep):
    """One checkerboarded Metropolis sweep, in place; the acceptance rate."""
    nd, nc = U.shape[0], U.shape[1]
    dims = U.shape[3:]
    V, acc = math.prod(dims), 0
    index = torch.arange(V, device=U.device).reshape(dims)
    draws = {1: 2, 2: 4, 3: 13}[nc]
    for p in range(1 << nd):
        cut = tuple(slice((p >> (nd - 1 - d)) & 1, None, 2) for d in range(nd))
        site = index[cut].reshape(-1)
        for mu in range(nd):
            S = [[x[cut].reshape(-1) for x in row] for row in _staple(U, mu)]
            u0 = [[U[mu, i, j][cut].reshape(-1) for j in range(nc)] for i in range(nc)]
            for hit in range(case["nhits"]):
                r, a = _proposal(nc, _uniforms(seed, 1, site, sweep, hit, mu, draws), case["delta"])
                new = _mul(u0, r)
                Sd = _dag(S)
                dS = -(case["beta"] / nc) * (_retr(new, Sd) - _retr(u0, Sd))
                ok = (dS < 0) | (a < torch.exp(-dS))
                acc += int(ok.sum())
                new = _restore(new)
                u0 = [[torch.where(ok, x, y) for x, y in zip(q, w)] for q, w in zip(new, u0)]
            for i in range(nc):
                for j in range(nc):
                    U[mu, i, j][cut] = u0[i][j].reshape(U[mu, i, j][cut].shape)
    return acc / (V * nd * case["nhits"])


def _generators(nc, dev):
    if nc == 1:
        t = [[[1]]]
    elif nc == 2:
        t = [[[0, 1], [1, 0]], [[0, -1j], [1j, 0]], [[1, 0], [0, -1]]]
    else:
        s = 1 / math.sqrt(3)
        t = [[[0, 1, 0], [1, 0, 0], [0, 0, 0]], [[0, -1j, 0], [1j, 0, 0], [0, 0, 0]],
             [[1, 0, 0], [0, -1, 0], [0, 0, 0]], [[0, 0, 1], [0, 0, 0], [1, 0, 0]],
             [[0, 0, -1j], [0, 0, 0], [1j, 0, 0]], [[0, 0, 0], [0, 0, 1], [0, 1, 0]],
             [[0, 0, 0], [0, 0, -1j], [0, 1j, 0]], [[s, 0, 0], [0, s, 0], [0, 0, -2 * s]]]
    return [[[complex(v) for v in row] for row in m] for m in t]


def _kick(U, P, beta, dt):
    nd, nc = U.shape[0], U.shape[1]
    T = _generators(nc, U.device)
    for mu in range(nd):
        M = _mul(_rows(U, mu), _staple(U, mu))
        for a, t in enumerate(T):
            tr = sum(t[i][j] * M[j][i] for i in range(nc) for j in range(nc) if t[i][j] != 0)
            P[mu, a] -= dt * (beta / nc) * tr.imag


def _drift(U, P, dt):
    nd, nc = U.shape[0], U.shape[1]
    T = _generators(nc, U.device)
    new = torch.empty_like(U)
    for mu in range(nd):
        zero = torch.zeros_like(U[mu, 0, 0])
        Q = [[1j * dt * (zero + sum(t[i][j] * P[mu, a] for a, t in enumerate(T) if t[i][j] != 0)) for j in range(nc)]
             for i in range(nc)]
        one = [[torch.ones_like(zero) if i == j else zero for j in range(nc)] for i in range(nc)]
        big = max(float(sum(x.abs() for x in row).max()) for row in Q)
        half = max(0, math.ceil(math.log2(max(big, 1e-9) / 0.25)))
        Q = [[x / 2 ** half for x in row] for row in Q]
        e, term, k = _add(one, Q), Q, 1
        while 0.25 ** k / math.factorial(k) > 1e-18:
            k += 1
            term = [[x / k for x in row] for row in _mul(term, Q)]
            e = _add(e, term)
        for _ in range(half):
            e = _mul(e, e)
        w = _mul(e, _rows(U, mu))
        for i in range(nc):
            for j in range(nc):
                new[mu, i, j] = w[i][j]
    return new


def _leapfrog(U, P, case):
    dt = case["tau"] / case["nsteps"]
    for i in range(case["nsteps"] + 1):
        _kick(U, P, case["beta"], dt / 2 if i == 0 else dt)
        U = _drift(U, P, dt)
    _kick(U, P, case["beta"], dt / 2)
    out = torch.empty_like(U)
    for mu in range(U.shape[0]):
        for i, row in enumerate(_restore(_rows(U, mu))):
            for j, x in enumerate(row):
                out[mu, i, j] = x
    return out


def _gauss(case, dims, seed, traj):
    nd, ng = case["nd"], ka.ngen(case["nc"])
    site = torch.arange(math.prod(dims), device=_device())
    P = torch.empty((nd, ng, *dims), dtype=torch.float64, device=_device())
    for mu in range(nd):
        u = _uniforms(seed, 2, site, traj, 0, mu, ng + ng % 2)
        for a in range(0, ng, 2):
            r, t = torch.sqrt(-2 * torch.log(1 - u[a])), 2 * math.pi * u[a + 1]
            P[mu, a] = (r * torch.cos(t)).reshape(dims)
            if a + 1 < ng:
                P[mu, a + 1] = (r * torch.sin(t)).reshape(dims)
    return P


def exact(case, seed):
    kind = case["kind"]
    # the decisions of a chain of FP32 links depend on their rounding
    if kind in ("batch", "ptbc") or (kind == "chain" and case["storage"] != "f64"):
        return None
    dims = _dims(case)
    V, nd, nc = math.prod(dims), case["nd"], case["nc"]
    if kind == "chain" and V * nd * nc ** 2 * case["n"] > 2_500_000 * 5:
        return None
    if kind in ("traj", "md") and V * nd * nc ** 2 * case["nsteps"] > 400_000_000:
        return None
    U = _links(nd, nc, dims, _gen(seed, 1))
    if kind == "chain":
        rates = np.array([_sweep(U, case, _run_seed(seed), s) for s in range(case["n"])])
        plaq, site = _plaq_out(case, U)
        out = {"rates": rates, "plaquette": plaq, "site": site}
        if case["loops"]:
            out["temporal"] = _loops_out(case, _temporal(U, _TEMPORAL))
            for mu, nu in _PLANES:
                out["planar%d%d" % (mu, nu)] = _loops_out(case, _loops(U, mu, nu, _PLANAR))
        return out
    if kind == "measure":
        plaq, site = _plaq_out(case, U)
        return {"plaquette": plaq, "site": site, "temporal": _loops_out(case, _temporal(U, _pairs(case)))}
    if kind == "md":
        P = _momenta(case, dims, seed)
        U = _leapfrog(U, P, case)
        plaq, site = _plaq_out(case, U)
        return {"kinetic": 0.5 * float((P * P).sum()), "plaquette": plaq, "site": site}
    P = _gauss(case, dims, _run_seed(seed), 0)
    c = -case["beta"] / nc
    k0, g0 = 0.5 * float((P * P).sum()), c * float(_site_plaquette(U).sum())
    new = _leapfrog(U, P, case)
    k1, g1 = 0.5 * float((P * P).sum()), c * float(_site_plaquette(new).sum())
    dH, ok = (k1 - k0) + (g1 - g0), True
    if dH > 0:
        one = torch.zeros(1, dtype=torch.int64, device=_device())
        ok = float(_uniforms(_run_seed(seed), 7, one, 0, 0, 0, 1)[0]) <= math.exp(-dH)
    plaq, site = _plaq_out(case, new if ok else U)
    return {"dH": dH, "accepted": int(ok), "plaquette": plaq, "site": site}
