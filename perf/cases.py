"""Timed workloads of the elemental-generation framework.

Each case is one thing that a user's program does over and over: a pass over
the timeslices of one configuration through ``ElementalGenerator`` (FP64 or
mixed form, single lattices or a batch), the reference-style ``calc(t)`` loop,
a whole configuration (load, link smearing, elementals), displacement
elementals, a forward + backward step, and the Laplacian block application of
the eigenvector feed.  The sizes are those of the benchmark's workloads (A to
E) with fewer timeslices, and of the tests' uneven shapes; ``draw`` spreads
over the ranges between them.

``exact`` restates the same maps in complex128 torch operations only.
"""

import itertools
import math

import numpy as np
import torch

from easydistillation_amd import (
    DisplacementElementalGenerator,
    ElementalGenerator,
    set_backend,
)
from easydistillation_amd._native import ED_BOPT_H16, ED_BOPT_ORDER, ED_OPT_MIXED_WS
from easydistillation_amd.autograd import ElementalEngine, profiled_loss
from easydistillation_amd.batch import ElementalBatch
from easydistillation_amd.eigen import EigenvectorGenerator
from easydistillation_amd.tune import autotune

DEV = "cuda:0"


def _case(name, kind, L, Lt, Ne, **more):
    c = {"name": name, "kind": kind, "Lx": L[0], "Ly": L[1], "Lz": L[2], "Lt": Lt, "Ne": Ne,
         "moms": "n2<=4", "nabla": 2, "mode": "fp64"}
    c.update(more)
    return c


def listed():
    return [
        # the reference test's driver, for t: data[t] = calc(t), on its own 4^3 x 8, Ne 20 configuration:
        # host arrays, launch and copy latency
        _case("loop_4c8_ne20", "loop", (4, 4, 4), 8, 20, nabla=1, moms="n2<=1"),
        # a small uneven lattice with blended (stochastic) weights, as in the parity tests
        _case("fp64_odd_ne37_blended", "calc", (10, 14, 9), 6, 37, blended=True),
        # the 16^3, Nev 100, 33 momenta, 13 derivatives workload in FP64
        _case("fp64_16c_ne100", "calc", (16, 16, 16), 8, 100),
        # downstream readers' largest momentum table (|n|^2 <= 9) on a mid-size lattice
        _case("fp64_20c_mom9", "calc", (20, 20, 20), 4, 70, nabla=1, moms="n2<=9"),
        # the headline shape, 32^3, Nev 200, 33 momenta, 13 derivatives: one 8-timeslice launch, FP64
        _case("fp64_32c_ne200", "calc", (32, 32, 32), 8, 200),
        # the same in the mixed form, with the tuned contraction a production run uses
        _case("mixed_32c_ne200", "calc", (32, 32, 32), 8, 200, mode="mixed", tuned=True),
        # the mixed form of the 16^3, Nev 100 workload
        _case("mixed_16c_ne100", "calc", (16, 16, 16), 32, 100, mode="mixed", tuned=True),
        # three lattices of different size in one graph launch (workload D with an eighth of the timeslices)
        _case("batch_mixed", "batch", (32, 32, 32), 8, 256, mode="mixed", nabla=1, moms="n2<=2"),
        # a training step on links, eigenvectors and profile weights (workload E with an eighth of the timeslices)
        _case("gradient_24c_ne128", "grad", (24, 24, 24), 8, 128, nabla=1, moms="n2<=1"),
        # displacement elementals (straight paths up to 6 links)
        _case("displacement_16c_ne64", "disp", (16, 16, 16), 8, 64, distance=6, moms="n2<=2"),
        # a production configuration from its links and eigenvectors: load, project, stout-smear, all elementals
        _case("configuration_24c_ne70", "config", (24, 24, 24), 8, 70, nabla=1, moms="n2<=2", nstep=10),
        # the eigensolver's inner operation: the Laplacian on a block of Nev + guard vectors
        _case("laplacian_24c_160", "lap", (24, 24, 24), 1, 160),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["calc", "calc", "calc", "calc", "mixed", "mixed", "loop", "disp", "grad", "config", "lap"])
        L = tuple(_log(rng, 4, 32) for _ in range(3))
        Lt, Ne = _log(rng, 1, 16), _log(rng, 1, 200)
        moms = rng.choice(["n2<=0", "n2<=1", "n2<=2", "n2<=3", "n2<=4", "n2<=9", "reftest"])
        more = {"moms": moms, "nabla": rng.choice([0, 1, 1, 2, 2, 2])}
        if kind == "mixed":
            L = tuple(_log(rng, 16, 32) for _ in range(3))
            more.update(mode="mixed", split16=rng.random() < 0.7)
        elif kind == "calc":
            more.update(blended=rng.random() < 0.2)
        elif kind == "loop":
            L, Lt, Ne = tuple(_log(rng, 4, 12) for _ in range(3)), _log(rng, 2, 16), _log(rng, 8, 64)
        elif kind == "disp":
            more.update(distance=rng.randint(1, 8), nabla=0)
        elif kind == "grad":
            more.update(nabla=rng.choice([0, 1, 1]), moms=rng.choice(["n2<=1", "n2<=2", "reftest"]))
        elif kind == "config":
            more.update(nabla=rng.choice([0, 1, 2]), nstep=rng.randint(1, 20))
        elif kind == "lap":
            Ne = _log(rng, 16, 256)
        c = _case("", {"mixed": "calc"}.get(kind, kind), L, Lt, Ne, **more)
        del c["name"]
        v3 = L[0] * L[1] * L[2]
        if 3 * v3 >= Ne and _cost(c) <= most and work(c)["bytes"] < 4e9:
            return c


def _cost(c):
    w = work(c)
    return w["bytes"] / 4e12 + w["flops"] / (5e13 if c["mode"] == "fp64" else 1.5e14)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _momenta(spec):
    if spec == "reftest":  # the list of the reference's elemental test
        return [(0, 0, 0), (0, 0, 1), (0, 1, 1), (1, 1, 1), (0, 0, 2), (0, 1, 2), (1, 1, 2)]
    n2 = int(spec.split("<=")[1])
    r = math.isqrt(n2)
    all_n = [n for n in itertools.product(range(-r, r + 1), repeat=3) if sum(v * v for v in n) <= n2]
    return sorted(all_n, key=lambda n: (sum(v * v for v in n), n))


def _links(c, seed, spread=0.4):
    """SU(3) links [3, Lt, Lz, Ly, Lx, 3, 3] near the identity (Gram-Schmidt of 1 + spread x Gaussian)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n = 3 * c["Lt"] * c["Lz"] * c["Ly"] * c["Lx"]
    Z = torch.view_as_complex(torch.randn((n, 3, 3, 2), generator=g, dtype=torch.float64, device=DEV)) * spread
    Z = Z + torch.eye(3, dtype=torch.complex128, device=DEV)
    a, b = Z[:, :, 0], Z[:, :, 1]
    a = a / torch.linalg.vector_norm(a, dim=1, keepdim=True)
    b = b - (a.conj() * b).sum(1, keepdim=True) * a
    b = b / torch.linalg.vector_norm(b, dim=1, keepdim=True)
    d = torch.linalg.cross(a, b, dim=1).conj()
    return torch.stack([a, b, d], 2).reshape(3, c["Lt"], c["Lz"], c["Ly"], c["Lx"], 3, 3).contiguous()


def _vectors(c, seed):
    """Orthonormal eigenvector stand-ins [Lt, Ne, Lz, Ly, Lx, 3], complex64 as the reference stages them."""
    g = torch.Generator(device=DEV).manual_seed(seed + 1000003)
    K = 3 * c["Lx"] * c["Ly"] * c["Lz"]
    V = torch.empty((c["Lt"], c["Ne"], K), dtype=torch.complex64, device=DEV)
    for t in range(c["Lt"]):
        A = torch.view_as_complex(torch.randn((c["Ne"], K, 2), generator=g, dtype=torch.float64, device=DEV))
        for _ in range(2):
            G = (A @ A.conj().transpose(0, 1).contiguous()).cpu()
            A = torch.linalg.inv(torch.linalg.cholesky(G)).to(DEV) @ A
        V[t] = A.to(torch.complex64)
    return V.reshape(c["Lt"], c["Ne"], c["Lz"], c["Ly"], c["Lx"], 3)


def _dilution(Ne):
    """Two dilution blocks: half of the eigenvectors exact, the rest sampled 1 in 2."""
    a = Ne // 2
    return ([a, 2 * (Ne - a)], [a, Ne - a]) if min(a, Ne - a) > 1 else ([Ne + 1], [Ne])


def _blended(c):
    return bool(c.get("blended")) and c["Ne"] > 1


def _members(c):
    """The lattices of a batch: (latt, Ne), the largest as in the case."""
    L, Lt, Ne = (c["Lx"], c["Ly"], c["Lz"]), c["Lt"], c["Ne"]
    half = tuple(l // 2 for l in L)
    mid = tuple(3 * l // 4 for l in L)
    return [dict(c, Lx=a[0], Ly=a[1], Lz=a[2], Lt=t, Ne=n)
            for a, t, n in ((half, Lt // 2, Ne // 4), (mid, 3 * Lt // 4, Ne // 2), (L, Lt, Ne))]


def _generator(c):
    latt = [c["Lx"], c["Ly"], c["Lz"], c["Lt"]]
    moms = _momenta(c["moms"])
    if c["kind"] == "disp":
        return DisplacementElementalGenerator(latt, None, None, c["distance"], moms, Ne=c["Ne"], mode=c["mode"])
    blend = _blended(c)
    g = ElementalGenerator(latt, None, None, c["nabla"], moms, dilution=_dilution(c["Ne"]) if blend else None,
                           is_blending=blend, Ne=c["Ne"], mode=c["mode"])
    if c.get("split16"):
        g.set_option(ED_OPT_MIXED_WS, 2)
    return g


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c}
    if kind == "batch":
        gens = []
        for k, m in enumerate(_members(c)):
            g = _generator(m)
            g.load_arrays(_links(m, 16 * seed + k), _vectors(m, 16 * seed + k))
            gens.append(g)
        b = ElementalBatch(gens)
        b.set_option(ED_BOPT_H16, 1)  # the choices the batch tuner makes for these lattices
        b.set_option(ED_BOPT_ORDER, 1)
        return dict(s, batch=b)
    U = _links(c, seed)
    if kind == "lap":
        e = EigenvectorGenerator([c["Lx"], c["Ly"], c["Lz"], c["Lt"]], None, c["Ne"])
        e.load_links(U)
        g = torch.Generator(device=DEV).manual_seed(seed + 7)
        F = torch.randn((c["Ne"], c["Lz"], c["Ly"], c["Lx"], 3, 2), generator=g, dtype=torch.float64, device=DEV)
        return dict(s, eig=e, F=torch.view_as_complex(F))
    V = _vectors(c, seed)
    if kind == "grad":
        w = torch.rand(c["Ne"], dtype=torch.float64, device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed + 9))
        eng = ElementalEngine([c["Lx"], c["Ly"], c["Lz"], c["Lt"]], c["Ne"], c["nabla"], _momenta(c["moms"]))
        return dict(s, eng=eng, U=U, V=V.to(torch.complex128), w=w + 0.5)
    gen = _generator(c)
    if kind == "config":
        # links off the group, as smeared or read in single precision
        U = U * (1 + 1e-3 * torch.cos(U.real * 50))
        return dict(s, gen=gen, U=U, V=V)
    gen.load_arrays(U, V)
    if c.get("tuned"):
        autotune(gen)
    if kind == "loop":
        shape = (c["Lt"], gen.num_derivative, gen.num_momentum, c["Ne"], c["Ne"])
        return dict(s, gen=gen, data=np.zeros(shape, dtype=np.complex128))
    out = torch.empty((c["Lt"], gen.num_derivative, gen.num_momentum, c["Ne"], c["Ne"]), dtype=torch.complex128, device=DEV)
    return dict(s, gen=gen, out=out)


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "loop":
        set_backend("hip")
        gen, data = state["gen"], state["data"]
        for t in range(c["Lt"]):
            data[t] = gen.calc(t)
        return data
    set_backend("torch")
    if kind == "batch":
        return state["batch"].run()
    if kind == "lap":
        return state["eig"].laplacian(0, state["F"])
    if kind == "grad":
        # new leaves each pass: a step of an optimiser has new inputs
        U, V, w = (state[k].detach().requires_grad_() for k in ("U", "V", "w"))
        loss = profiled_loss(U, V, w, state["eng"])
        gU, gV, gw = torch.autograd.grad(loss, [U, V, w])
        return {"loss": loss.detach(), "gU": gU, "gV": gV, "gw": gw}
    gen = state["gen"]
    if kind == "config":
        gen.load_arrays(state["U"], state["V"])
        gen.project_SU3()
        gen.stout_smear(c["nstep"], 0.1)
        return {"E": gen.calc_all(), "U": gen.gauge()}
    return gen.calc_range(0, c["Lt"], out=state["out"])


# ---------------------------------------------------------------------------
# work of one pass
# ---------------------------------------------------------------------------
def _tuples(nabla):
    return [t for k in range(nabla + 1) for t in itertools.product(range(3), repeat=k)]


def _splits(t):
    """Merged (left, right) -> coefficient of the two-sided derivative t."""
    acc = {}
    for pick in range(1 << len(t)):
        right = tuple(t[j] for j in range(len(t)) if pick >> j & 1)
        left = tuple(t[j] for j in range(len(t)) if not pick >> j & 1)[::-1]
        acc[left, right] = acc.get((left, right), 0) + (-1) ** len(right)
    return {k: v for k, v in acc.items() if v}


def work(case):
    c = case
    if c["kind"] == "batch":
        ws = [work(dict(m, kind="calc")) for m in _members(c)]
        return {k: sum(w[k] for w in ws) for k in ws[0]}
    V3, Lt, Ne = c["Lx"] * c["Ly"] * c["Lz"], c["Lt"], c["Ne"]
    links, vec = 3 * 9 * 16 * V3, 3 * V3 * Ne
    if c["kind"] == "lap":
        return {"bytes": 2 * 16 * vec + links, "flops": 6 * 72.0 * V3 * Ne}
    moms = _momenta(c["moms"])
    nx = {abs(n[0]) for n in moms}
    fx = sum(2 if n else 1 for n in nx)  # real functions of x the momenta need
    pair = 0.0  # flops per site: split sum per pair, then the sum over one lattice axis against fx functions
    if c["kind"] == "disp":
        D, hops = c["distance"] + 1, 6 * c["distance"]
        pair = D * Ne * Ne * (24.0 + 4 * fx)
    else:
        ts = _tuples(c["nabla"])
        D, hops = len(ts), len(ts) - 1
        for t in ts:
            if t <= t[::-1]:  # E of the reversed tuple is the Hermitian conjugate
                pairs = Ne * (Ne + 1) / 2 if t == t[::-1] else Ne * Ne
                pair += pairs * (24.0 * len(_splits(t)) + 4 * fx)
    flops = Lt * (V3 * pair + hops * 144.0 * V3 * Ne)
    out = 16.0 * D * len(moms) * Ne * Ne * Lt
    b = Lt * (links + 8 * vec) + out
    if c["kind"] == "grad":
        # cotangent in, both gradients out; the split sums of the reverse pass go to both operands
        flops += Lt * V3 * Ne * Ne * sum(4.0 * fx + 48 * len(_splits(t)) for t in _tuples(c["nabla"]))
        b += out + Lt * (links + 16 * vec) + Lt * 8 * vec
    if c["kind"] == "config":
        b += Lt * links * (1 + 2 * c["nstep"])
        flops += Lt * 3 * V3 * c["nstep"] * 2500.0
    return {"bytes": float(b), "flops": float(flops)}


# ---------------------------------------------------------------------------
# the same maps in complex128 torch operations
# ---------------------------------------------------------------------------
def _apply(U, F):
    """U [Z, Y, X, 3, 3] on F [n, Z, Y, X, 3]."""
    return (U.unsqueeze(0) * F.unsqueeze(-2)).sum(-1)


def _forward(U, mu, F):
    """U_mu(x) F(x + mu)."""
    return _apply(U[mu], torch.roll(F, -1, 3 - mu))


def _backward(U, mu, F):
    """U_mu(x - mu)^dagger F(x - mu)."""
    return torch.roll(_apply(U[mu].conj().transpose(-1, -2), F), 1, 3 - mu)


def _phases(c, moms):
    ax = [torch.arange(c[k], dtype=torch.float64, device=DEV) / c[k] for k in ("Lx", "Ly", "Lz")]
    ph = []
    for n in moms:
        a = 2 * math.pi * (n[2] * ax[2][:, None, None] + n[1] * ax[1][None, :, None] + n[0] * ax[0][None, None, :])
        ph.append(torch.polar(torch.ones_like(a), a).reshape(-1).repeat_interleave(3))
    return ph


def _weights(c):
    tot, used = _dilution(c["Ne"])
    W, edge = torch.empty((c["Ne"], c["Ne"]), dtype=torch.float64), np.cumsum([0] + used)
    for i, (ti, ui) in enumerate(zip(tot, used)):
        for j, (tj, uj) in enumerate(zip(tot, used)):
            b = W[edge[i]:edge[i + 1], edge[j]:edge[j + 1]]
            b[:] = ti * tj / (ui * uj) if i != j else ti * (ti - 1) / (ui * (ui - 1))
            if i == j:
                b.fill_diagonal_(ti / ui)
    return W.to(DEV)


def _terms(c, U, V):
    """Per output d the list of (coefficient, left [Ne, K], right [Ne, K]) of one timeslice."""
    Ne = c["Ne"]
    if c["kind"] == "disp":
        out = [[(1.0, V.reshape(Ne, -1), V.reshape(Ne, -1))]]
        P = [V] * 6
        for _ in range(c["distance"]):
            P = [_forward(U, mu, P[mu]) for mu in range(3)] + [_backward(U, mu, P[3 + mu]) for mu in range(3)]
            out.append([(1.0, V.reshape(Ne, -1), (sum(P) / 6).reshape(Ne, -1))])
        return out
    W = {(): V}
    for t in _tuples(c["nabla"])[1:]:
        p = W[t[:-1]]
        W[t] = _forward(U, t[-1], p) - _backward(U, t[-1], p)
    flat = {k: v.reshape(Ne, -1) for k, v in W.items()}
    return [[(float(cf), flat[l], flat[r]) for (l, r), cf in _splits(t).items()] for t in _tuples(c["nabla"])]


def _elementals(c, U, V, ph):
    E = []
    for terms in _terms(c, U, V):
        R = torch.cat([r for _, _, r in terms], 1).transpose(0, 1).contiguous()
        row = []
        for p in ph:
            row.append(torch.cat([cf * l.conj() * p for cf, l, _ in terms], 1) @ R)
        E.append(torch.stack(row))
    E = torch.stack(E)
    return E * _weights(c) if _blended(c) else E


def _polar(U):
    for _ in range(12):
        U = 0.5 * (U + torch.linalg.inv(U).conj().transpose(-1, -2))
    return U


def _stout(U, rho):
    """One 3-D stout step on U [3, Z, Y, X, 3, 3]."""
    def dag(m):
        return m.conj().transpose(-1, -2)

    new = []
    for mu in range(3):
        C = 0
        for nu in range(3):
            if nu == mu:
                continue
            up, sm = torch.roll(U[mu], -1, 2 - nu), torch.roll(U[nu], -1, 2 - mu)
            C = C + U[nu] @ up @ dag(sm)
            C = C + torch.roll(dag(U[nu]) @ U[mu] @ sm, 1, 2 - nu)
        Om = rho * C @ dag(U[mu])
        Q = 0.5j * (dag(Om) - Om)
        Q = Q - torch.diagonal(Q, dim1=-2, dim2=-1).sum(-1)[..., None, None] / 3 * torch.eye(3, dtype=Q.dtype, device=DEV)
        new.append(torch.linalg.matrix_exp(1j * Q) @ U[mu])
    return torch.stack(new)


def _exact_all(c, U, V):
    ph = _phases(c, _momenta(c["moms"]))
    return torch.stack([_elementals(c, U[:, t], V[t].to(torch.complex128), ph) for t in range(c["Lt"])])


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "batch":
        return [_exact_all(dict(m, kind="calc"), _links(m, 16 * seed + k), _vectors(m, 16 * seed + k))
                for k, m in enumerate(_members(c))]
    U = _links(c, seed)
    if kind == "lap":
        g = torch.Generator(device=DEV).manual_seed(seed + 7)
        F = torch.randn((c["Ne"], c["Lz"], c["Ly"], c["Lx"], 3, 2), generator=g, dtype=torch.float64, device=DEV)
        F = torch.view_as_complex(F)
        return 6 * F - sum(_forward(U[:, 0], mu, F) + _backward(U[:, 0], mu, F) for mu in range(3))
    V = _vectors(c, seed)
    if kind == "grad":
        g = torch.Generator(device=DEV).manual_seed(seed + 9)
        w = torch.rand(c["Ne"], dtype=torch.float64, device=DEV, generator=g) + 0.5
        ph, loss, gU, gV, gw = _phases(c, _momenta(c["moms"])), 0.0, [], [], 0.0
        for t in range(c["Lt"]):
            u, v, x = (a.detach().requires_grad_() for a in (U[:, t], V[t].to(torch.complex128), w))
            E = _elementals(c, u, v, ph)
            part = ((torch.diagonal(E, dim1=-2, dim2=-1) * x).sum(-1).abs() ** 2).sum()
            a, b, d = torch.autograd.grad(part, [u, v, x], allow_unused=True)
            loss, gw = loss + part.detach(), gw + d
            gU.append(a if a is not None else torch.zeros_like(u))
            gV.append(b)
        return {"loss": loss, "gU": torch.stack(gU, 1), "gV": torch.stack(gV), "gw": gw}
    if kind == "config":
        U = _polar(U * (1 + 1e-3 * torch.cos(U.real * 50)))
        for _ in range(c["nstep"]):
            U = torch.stack([_stout(U[:, t], 0.1) for t in range(c["Lt"])], 1)
        return {"E": _exact_all(c, U, V), "U": U}
    return _exact_all(c, U, V)
