"""Performance cases: what a lattice-gauge program has the engine do, through the
public Python entry points.

A case is one pass of one kind of work:

  step        one Markov step call by call (heatbath, overrelaxation sweeps,
              reunitarisation, plaquette, Polyakov loop) and the configuration handed
              to the host
  generate    a stretch of the generation driver on one lattice
  batch       the same for many small lattices at once
  loops       the Wilson loops W(r, T) of a configuration
  potential   the static-potential measurement: a copy of the configuration is APE
              smeared, its temporal links multihit averaged, W(r, T) measured
  smear       one smearing (or link averaging) of a copy of the configuration, looked at
              through its small Wilson loops or, for small lattices, as links
  operators   operator-basis Wilson loops (the A0 or the 33 family)

Start fields are made from the seed with torch: a random gauge transform of links
scattered about the identity, so wide that the plaquette is about 0.6 as in a
thermalised field at the couplings used here.

An update's links stay on the device, and the one public way to look at them is a copy
of the whole field to the host, which takes many times longer than the update itself:
small cases return their links, the others the observables that the call gives back,
which every link enters.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import sun_amd

SPATIAL = ("x", "y", "z")
BETA = {2: 2.4, 3: 6.0, 4: 10.8}
# scatter of the links about the identity that gives a plaquette of about 0.6
SCATTER = {2: 0.30, 3: 0.24, 4: 0.21}
HYP_ALPHAS = (0.75, 0.6, 0.3)
NOPS = {0: 10, 1: 25}


# ---- cases ---------------------------------------------------------------------------
def _case(kind, dims, nc, storage, precision, **more):
    return {"kind": kind, "x": dims[0], "y": dims[1], "z": dims[2], "t": dims[3], "nc": nc, "storage": storage,
            "precision": precision, "beta": more.pop("beta", BETA[nc]), **more}


def listed():
    cases = {
        # the smallest lattice in common use, driven call by call in double precision by a
        # program that analyses every configuration on the host: launches and latency
        "step_8x4_su3_f64": _case("step", (8, 8, 8, 8), 3, 18, 8, n_or=4),
        # a small SU(2) ensemble, short graph-replayed stretches
        "generate_16x4_su2_f32": _case("generate", (16, 16, 16, 16), 2, 18, 4, n_iter=4, n_or=4, shape=""),
        # the benchmark's lattice with the benchmark's launch shapes
        "generate_32x4_su3_f32_12": _case("generate", (32, 32, 32, 32), 3, 12, 4, n_iter=8, n_or=4, shape="32"),
        # double precision throughout, rows of 12 sites
        "generate_24x3x48_su3_f64": _case("generate", (24, 24, 24, 48), 3, 18, 8, n_iter=2, n_or=4, shape=""),
        # large-N generation, the largest volume of the SU(4) jobs the benchmark serves
        "generate_32x4_su4_f32": _case("generate", (32, 32, 32, 32), 4, 18, 4, n_iter=2, n_or=4, shape=""),
        # the largest lattice, compressed links
        "generate_64x4_su3_f32_8": _case("generate", (64, 64, 64, 64), 3, 8, 4, n_iter=2, n_or=4, shape="64",
                                         beta=6.2),
        # an ensemble scan: lattices of several volumes and couplings updated together
        "batch_mixed_su3_f32_12": _case("batch", (0, 0, 0, 0), 3, 12, 4, n_iter=2, n_or=4, lattices=20,
                                        volumes="8x8x8x8 12x12x12x12 16x16x16x16 16x16x16x32 24x24x24x24"),
        # the measurements between updates
        "loops_32x4_su3_f32_12": _case("loops", (32, 32, 32, 32), 3, 12, 4, rmax=16, tmax=16),
        "potential_24x3x32_su3_f32_12": _case("potential", (24, 24, 24, 32), 3, 12, 4, steps=25, hits=100, rmax=12,
                                              tmax=16),
        "smear_hyp_16x3x32_su3_f64": _case("smear", (16, 16, 16, 32), 3, 18, 8, method="hyp", steps=2, links=False),
        "operators_a0_24x3x32_su3_f64": _case("operators", (24, 24, 24, 32), 3, 18, 8, family=0, rmax=4, tmax=12),
        "operators_33_16x3x32_su3_f32_12": _case("operators", (16, 16, 16, 32), 3, 12, 4, family=1, rmax=4, tmax=16),
    }
    return [{"name": name, **c} for name, c in cases.items()]


def _even(rng, lo, hi):
    """an even extent, spread over its logarithm"""
    return max(lo, min(hi, 2 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2)))


def _dims(rng, lo, hi, most):
    """a cubic spatial volume (one in three of them not cubic) and a time extent, of at most `most` sites"""
    while True:
        s = _even(rng, lo, hi)
        d = [s, s, s, _even(rng, max(lo, 4), 2 * hi)]
        if rng.random() < 1 / 3:
            d = [_even(rng, lo, hi) for _ in range(3)] + [d[3]]
        if math.prod(d) <= most:
            return d


def _group(rng):
    """N, storage, precision: mostly SU(3)"""
    nc = rng.choice((2, 3, 3, 3, 3, 4))
    precision = rng.choice((4, 4, 8))
    return nc, rng.choice((18, 12, 12, 8)) if nc == 3 else 18, precision


def draw(rng):
    kind = rng.choice(("step", "generate", "generate", "generate", "batch", "loops", "potential", "smear",
                       "operators", "operators"))
    nc, storage, precision = _group(rng)
    if kind == "step":
        return _case(kind, _dims(rng, 4, 12, 1 << 14), nc, storage, precision, n_or=rng.randint(1, 6))
    if kind == "generate":
        return _case(kind, _dims(rng, 6, 32, 1 << 19), nc, storage, precision, n_iter=rng.randint(1, 4),
                     n_or=rng.randint(1, 6), shape="")
    if kind == "batch":
        volumes = " ".join("x".join(map(str, _dims(rng, 6, 16, 1 << 16))) for _ in range(4))
        return _case(kind, (0, 0, 0, 0), nc, storage, precision, n_iter=rng.randint(1, 3), n_or=rng.randint(1, 6),
                     lattices=rng.randint(3, 24), volumes=volumes)
    if kind == "smear":
        method = rng.choice(("ape", "stout", "hyp", "multihit", "multihit_ext"))
        links = rng.random() < 1 / 3
        d = _dims(rng, 6, 12 if links else 24, 1 << (14 if links else 16 if method == "multihit_ext" else 18))
        steps = {"ape": (5, 30), "stout": (5, 30), "hyp": (1, 3), "multihit": (10, 100), "multihit_ext": (2, 8)}[method]
        return _case(kind, d, 3 if method == "stout" else nc, storage if nc == 3 else 18, precision, method=method,
                     steps=rng.randint(*steps), links=links)
    d = _dims(rng, 6, 28 if kind == "loops" else 20, 1 << {"operators": 16, "potential": 17, "loops": 19}[kind])
    least = min(d[:3])
    if kind == "operators":
        return _case(kind, d, nc, storage, precision, family=rng.randint(0, 1), rmax=rng.randint(2, min(4, least)),
                     tmax=rng.randint(2, min(16, d[3])))
    c = _case(kind, d, nc, storage, precision, rmax=rng.randint(2, least // 2 + 1), tmax=rng.randint(2, d[3] // 2))
    return {**c, "steps": rng.randint(5, 30), "hits": rng.choice((0, 20, 50, 100))} if kind == "potential" else c


# ---- fields --------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _mm(a, b):
    """product of N x N matrices over any leading dimensions"""
    return sum(a[..., :, k, None] * b[..., k, None, :] for k in range(a.shape[-1]))


def _dag(a):
    return a.conj().transpose(-1, -2)


def _det(m):
    n = m.shape[-1]
    if n == 1:
        return m[..., 0, 0]
    rest = m[..., 1:, :]
    keep = [[c for c in range(n) if c != j] for j in range(n)]
    return sum((-1) ** j * m[..., 0, j] * _det(rest[..., keep[j]]) for j in range(n))


def _special_unitary(a):
    """rows made orthonormal one after another, the determinant's phase taken out of the last"""
    rows = []
    for i in range(a.shape[-1]):
        r = a[..., i, :]
        for q in rows:
            r = r - (q.conj() * r).sum(-1, keepdim=True) * q
        rows.append(r / r.abs().square().sum(-1, keepdim=True).sqrt())
    m = torch.stack(rows, -2)
    m[..., -1, :] *= _det(m).conj()[..., None]
    return m


def _axis(mu):
    """the tensor dimension of direction mu in [t, z, y, x, ...]"""
    return 3 - mu


def _at(a, mu, n=1):
    """a(x + n e_mu)"""
    return torch.roll(a, -n, _axis(mu)) if n else a


def _field(dims, nc, storage, precision, seed):
    """links[mu][t, z, y, x] in 64 bits, as the lattice's storage and precision hold them"""
    dev = _device()
    gen = torch.Generator(dev).manual_seed(seed)
    shape = (dims[3], dims[2], dims[1], dims[0], nc, nc)

    def gauss():
        return torch.view_as_complex(torch.randn(*shape, 2, generator=gen, device=dev, dtype=torch.float64))

    one = torch.eye(nc, device=dev, dtype=torch.complex128)
    g = _special_unitary(gauss())
    out = []
    for mu in range(4):
        u = _special_unitary(one + SCATTER[nc] * gauss())
        u = _mm(_mm(g, u), _dag(_at(g, mu)))
        if precision == 4:
            u = u.to(torch.complex64).to(torch.complex128)
        if storage == 12:
            u[..., 2, :] = torch.linalg.cross(u[..., 0, :], u[..., 1, :]).conj()
        out.append(u)
    return out


def _site_order(dims):
    """lexicographic index (x fastest) of the sites in even/odd order"""
    x, y, z, t = dims
    lex = np.arange(x * y * z * t)
    odd = (lex % x + lex // x % y + lex // (x * y) % z + lex // (x * y * z)) & 1
    return np.argsort(odd, kind="stable")


def _to_host_order(links, dims):
    order = torch.from_numpy(_site_order(dims)).to(links[0].device)
    n = links[0].shape[-1]
    return torch.stack([u.reshape(-1, n, n)[order] for u in links]).cpu().numpy()


_context = None


def _ctx():
    """one context for the program, as a program keeps it"""
    global _context
    if _context is None:
        _context = sun_amd.Context(0)
    return _context


class _Held(dict):
    """a state whose handles are given back with it"""

    def __del__(self):
        for h in self.get("handles", ()):
            h.close()


# launch shapes (kernel 0 heatbath, 1 overrelaxation) that the benchmark pins
SHAPES = {
    "32": {0: dict(block=256, brick=(2, 0, 2), lds=40960, piped=2), 1: dict(block=256, brick=(2, 0, 2), lds=54272, piped=2)},
    "64": {0: dict(block=256, brick=(0, 1, 2), lds=0, piped=0), 1: dict(block=256, brick=(0, 1, 2), lds=32768, piped=1)},
}


def _lattice(case, dims, seed, storage=None, beta=None):
    lat = sun_amd.Lattice(_ctx(), case["nc"], dims, case["beta"] if beta is None else beta,
                          storage or case["storage"], case["precision"])
    for kernel, shape in SHAPES.get(case.get("shape"), {}).items():
        lat.set_launch(kernel, **shape)
    if seed is None:
        return lat
    if math.prod(dims) > 1 << 21:
        # a host field of this volume would be 10 GB: start from a Haar field as a production run does
        lat.hot_start(seed)
        lat.generate(seed=seed, n_iter=1, measure=False)
    else:
        lat.from_host(_to_host_order(_field(dims, case["nc"], case["storage"], case["precision"], seed), dims))
    return lat


def _case_dims(case):
    return case["x"], case["y"], case["z"], case["t"]


def _volumes(case):
    names = case["volumes"].split()
    return [tuple(map(int, names[i % len(names)].split("x"))) for i in range(case["lattices"])]


def prepare(case, seed):
    kind, dims = case["kind"], _case_dims(case)
    if kind == "batch":
        rng = np.random.default_rng(seed)
        lats = [_lattice(case, d, seed + 7919 * i, beta=case["beta"] * rng.uniform(0.95, 1.05))
                for i, d in enumerate(_volumes(case))]
        batch = sun_amd.Batch(_ctx(), lats, [seed + i for i in range(len(lats))])
        return _Held(case=case, seed=seed, sweep=0, batch=batch, handles=[batch, *lats])
    lat = _lattice(case, dims, seed)
    state = _Held(case=case, seed=seed, sweep=1, lat=lat, handles=[lat])
    if kind == "potential" or (kind == "smear" and not case["method"].startswith("multihit")):
        state["work"] = _lattice(case, dims, None)
        state["handles"].append(state["work"])
    if case.get("hits") or case.get("method", "").startswith("multihit"):
        state["mean"] = _lattice(case, dims, None, storage=18)  # the averaged links are not in SU(N)
        state["handles"].append(state["mean"])
    return state


# ---- one pass ------------------------------------------------------------------------
def _out(case, a):
    """an FP32 lattice's results as the single-precision numbers they are"""
    a = np.asarray(a)
    if case["precision"] == 8:
        return a
    return a.astype(np.complex64 if a.dtype.kind == "c" else np.float32)


def _next_sweep(state, n):
    first = state["sweep"]
    state["sweep"] = first + n
    return first


def _run_step(state, case):
    lat, sweep = state["lat"], _next_sweep(state, 1)
    lat.heatbath(state["seed"], sweep)
    for _ in range(case["n_or"]):
        lat.overrelax()
    lat.reunitarize()
    plaq, poly = lat.plaquette(), lat.polyakov()
    return {"observables": _out(case, [plaq[0], plaq[1], poly.real, poly.imag]), "links": _out(case, lat.to_host())}


def _run_generate(state, case):
    n = case["n_iter"]
    return _out(case, state["lat"].generate(seed=state["seed"], n_iter=n, n_or=case["n_or"],
                                            first_sweep=_next_sweep(state, n)))


def _run_batch(state, case):
    n = case["n_iter"]
    return _out(case, state["batch"].generate(_next_sweep(state, n), n, n_or=case["n_or"]))


def _run_loops(state, case):
    return _out(case, state["lat"].wilson_loops(case["rmax"], case["tmax"]))


def _run_potential(state, case):
    work = state["work"]
    work.copy_from(state["lat"])
    work.ape_smear(0.2, case["steps"], 10)
    if case["hits"]:
        work.multihit(state["mean"], state["seed"], case["hits"])
        work = state["mean"]
    return _out(case, work.wilson_loops(case["rmax"], case["tmax"]))


def _run_smear(state, case):
    lat, method, steps = state["lat"], case["method"], case["steps"]
    if method == "multihit":
        lat.multihit(state["mean"], state["seed"], steps)
        work = state["mean"]
    elif method == "multihit_ext":
        lat.multihit_ext(state["mean"], state["seed"], steps)
        work = state["mean"]
    else:
        work = state["work"]
        work.copy_from(lat)
        if method == "ape":
            work.ape_smear(0.2, steps, 10)
        elif method == "stout":
            work.stout_smear(0.1, steps)
        else:
            work.hyp_smear(HYP_ALPHAS, steps, 10)
    return _out(case, work.to_host() if case["links"] else work.wilson_loops(4, 4))


def _run_operators(state, case):
    return _out(case, state["lat"].wilson_loops_ops(case["rmax"], case["tmax"], case["family"]))


_RUN = {"step": _run_step, "generate": _run_generate, "batch": _run_batch, "loops": _run_loops,
        "potential": _run_potential, "smear": _run_smear, "operators": _run_operators}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


# ---- the work of a pass --------------------------------------------------------------
def work(case):
    """Bytes: the links of every (parity, mu) launch of an update (all 4V read, V/2
    written: the next launch depends on it, and a field is larger than the on-chip
    memories), one read and one write of the smeared directions per smearing step, one
    read of the field per measurement, what goes to the host.  Operations: the matrix
    products, 8 N^3 each, and traces, 8 N^2, of the shortest form of each path."""
    nc, kind = case["nc"], case["kind"]
    mm, tr = 8 * nc ** 3, 8 * nc ** 2
    blocks = nc * (nc - 1) // 2
    rotate = blocks * (2 * mm // nc + 40)  # one SU(2) block after another: projection and rotation of two rows
    real = 2 * nc * nc if case["storage"] == 18 else case["storage"]
    link = real * case["precision"]
    full = 2 * nc * nc * case["precision"]
    if kind in ("step", "generate", "batch"):
        volume = sum(map(math.prod, _volumes(case))) if kind == "batch" else math.prod(_case_dims(case))
        sweeps = case["n_or"] + 1
        n = case.get("n_iter", 1)
        host = 2 * 4 * volume * 16 * nc * nc if kind == "step" else 0
        return {"bytes": n * 4 * volume * link * (9 * sweeps + 3) + host,
                "flops": n * 4 * volume * (sweeps * (12 * mm + rotate) + 3 * mm)}
    volume = math.prod(_case_dims(case))
    links = 4 * volume

    def loops(rmax, tmax):
        return 3 * volume * (rmax * mm + (rmax + 1) * (2 * mm + (tmax + 1) * tr))

    if kind == "loops":
        return {"bytes": links * link, "flops": loops(case["rmax"], case["tmax"])}
    if kind == "operators":
        nop = NOPS[case["family"]]
        paths, pairs = (36, nop * nop) if case["family"] == 0 else (32, nop * nop)
        each = volume * (paths * 2 * mm + nop * 2 * mm + (case["tmax"] + 1) * pairs * tr // 2)
        rs = case["rmax"] - 1
        return {"bytes": links * link + rs * 3 * nop * volume * full * 2, "flops": rs * 3 * each}
    if kind == "potential":
        ape = case["steps"] * 3 * volume * (8 * mm + 10 * rotate)
        hits = volume * (12 * mm + case["hits"] * rotate)
        return {"bytes": case["steps"] * 6 * volume * link + 2 * links * link,
                "flops": ape + (hits if case["hits"] else 0) + loops(case["rmax"], case["tmax"])}
    method, steps = case["method"], case["steps"]
    flops = {"ape": steps * 3 * volume * (8 * mm + 10 * rotate), "stout": steps * 3 * volume * 12 * mm,
             "hyp": steps * volume * (12 * (4 * mm + 10 * rotate) + 12 * (8 * mm + 10 * rotate) + 3 * (12 * mm + 10 * rotate)),
             "multihit": volume * (12 * mm + steps * rotate),
             "multihit_ext": volume * 27 * steps * (12 * mm + rotate)}[method]
    moved = volume * link * 6 * steps if not method.startswith("multihit") else links * (link + full)
    host = 2 * links * 16 * nc * nc if case["links"] else links * full
    return {"bytes": moved + host, "flops": flops + (0 if case["links"] else loops(4, 4))}


# ---- the same in 64 bits -------------------------------------------------------------
def _block_pairs(n):
    return [(i, i + d) for d in range(1, n) for i in range(n - d)]


def _project(w, q, hits):
    """SU(2)-subgroup maximisation of Re Tr(w q^+), `hits` rounds"""
    w, q = w.clone(), _dag(q)
    for _ in range(hits):
        for x, y in _block_pairs(w.shape[-1]):
            rows = w[..., [x, y], :]
            m = sum(rows[..., :, k, None] * q[..., k, None, [x, y]] for k in range(w.shape[-1]))
            r = torch.stack([m[..., 0, 0].real + m[..., 1, 1].real, m[..., 0, 1].imag + m[..., 1, 0].imag,
                             m[..., 0, 1].real - m[..., 1, 0].real, m[..., 0, 0].imag - m[..., 1, 1].imag])
            r = r / r.square().sum(0).sqrt()
            a, b = torch.complex(r[0], -r[3])[..., None], torch.complex(-r[2], -r[1])[..., None]
            w[..., x, :] = a * rows[..., 0, :] + b * rows[..., 1, :]
            w[..., y, :] = -b.conj() * rows[..., 0, :] + a.conj() * rows[..., 1, :]
    return w


def _staple(a, b, mu, nu):
    """up and down staple of direction mu in the plane (mu, nu): sides a, the opposite link b"""
    up = _mm(_mm(a, _at(b, nu)), _dag(_at(a, mu)))
    down = _mm(_mm(_dag(a), b), _at(a, mu))
    return up + _at(down, nu, -1)


def _exact_ape(u, steps):
    n = u[0].shape[-1]
    one = torch.eye(n, device=u[0].device, dtype=torch.complex128)
    for _ in range(steps):
        new = []
        for mu in range(3):
            s = sum(_staple(u[nu], u[mu], mu, nu) for nu in range(3) if nu != mu)
            v = (u[mu] + 0.2 * s) / 2.2
            new.append(_project(one.expand_as(v) if n == 3 else u[mu], v, 10))
        u = new + [u[3]]
    return u


def _exact_stout(u, steps):
    one = torch.eye(3, device=u[0].device, dtype=torch.complex128)
    for _ in range(steps):
        new = []
        for mu in range(3):
            om = 0.1 * _mm(sum(_staple(u[nu], u[mu], mu, nu) for nu in range(3) if nu != mu), _dag(u[mu]))
            q = 0.5 * (_dag(om) - om)  # Q = i q
            q = q - q.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None] / 3 * one
            e = one + torch.zeros_like(q)
            for k in range(24, 0, -1):  # exp(i Q) = exp(-q)
                e = one - _mm(q, e) / k
            new.append(_mm(e, u[mu]))
        u = new + [u[3]]
    return u


def _exact_hyp(u, steps):
    a1, a2, a3 = HYP_ALPHAS
    for _ in range(steps):
        bar = {(m, e): _project(u[m], 0.5 * a3 * _staple(u[e], u[m], m, e) + (1 - a3) * u[m], 10)
               for m in range(4) for e in range(4) if m != e}
        til = {}
        for m in range(4):
            for n in range(4):
                if m != n:
                    s = sum(_staple(bar[r, 6 - m - n - r], bar[m, 6 - m - n - r], m, r) for r in range(4) if r not in (m, n))
                    til[m, n] = _project(u[m], 0.25 * a2 * s + (1 - a2) * u[m], 10)
        u = [_project(u[m], a1 / 6 * sum(_staple(til[n, m], til[m, n], m, n) for n in range(4) if n != m)
                      + (1 - a1) * u[m], 10) for m in range(3)] + [u[3]]
    return u


def _exact_loops(u, rmax, tmax):
    """W(r, T): the time lines first, then every spatial line moved along them"""
    n, volume = u[0].shape[-1], u[0][..., 0, 0].numel()
    one = torch.eye(n, device=u[0].device, dtype=torch.complex128).expand_as(u[0])
    w = torch.zeros(rmax + 1, tmax + 1, dtype=torch.complex128, device=u[0].device)
    time = [one]
    for t in range(tmax):
        time.append(_mm(time[-1], _at(u[3], 3, t)))
    for mu in range(3):
        line = one
        for r in range(rmax + 1):
            for t in range(tmax + 1):
                # Tr(L t1 (t0 L(x + T))^+)
                w[r, t] += (_mm(line, _at(time[t], mu, r)) * _mm(time[t], _at(line, 3, t)).conj()).sum()
            if r < rmax:
                line = _mm(line, _at(u[mu], mu, r))
    return (w / (3 * n * volume)).cpu().numpy()


def _exact_a0(u, rmax, tmax):
    """the A0 family: the line, its four staples of heights 1..8, a zero slot"""
    n, volume = u[0].shape[-1], u[0][..., 0, 0].numel()
    out = np.zeros((rmax - 1, 100, tmax + 1))
    one = torch.eye(n, device=u[0].device, dtype=torch.complex128).expand_as(u[0])

    def lines(mu, most):
        got = [one]
        for k in range(most):
            got.append(_mm(got[-1], _at(u[mu], mu, k)))
        return got

    time = lines(3, tmax)
    for mu in range(3):
        sides = {d: lines(d, 8) for d in range(3) if d != mu}
        base = lines(mu, rmax)
        for r in range(2, rmax + 1):
            ops = [base[r]]
            for h in range(1, 9):
                acc = 0
                for d in sides:
                    s = sides[d][h]
                    acc = acc + _mm(_mm(s, _at(base[r], d, h)), _dag(_at(s, mu, r)))
                    acc = acc + _at(_mm(_mm(_dag(s), base[r]), _at(s, mu, r)), d, -h)
                ops.append(acc / 2)
            ops.append(torch.zeros_like(one))
            for t in range(tmax + 1):
                left = torch.stack([_mm(o, _at(time[t], mu, r)).reshape(-1) for o in ops])
                right = torch.stack([_mm(time[t], _at(o, 3, t)).reshape(-1) for o in ops])
                c = torch.view_as_real(left).reshape(10, -1) @ torch.view_as_real(right).reshape(10, -1).T
                out[r - 2, :, t] += c.reshape(100).cpu().numpy()
    return out / (3 * n * volume)


def exact(case, seed):
    """None where a heatbath comes in (its accept/reject decisions belong to the
    lattice's precision: in 64 bits some fall the other way and their links differ
    altogether) and for the 33 family, whose path tables are the engine's own."""
    kind, nc = case["kind"], case["nc"]
    if kind not in ("loops", "potential", "smear", "operators") or case.get("family") == 1 or case.get("hits"):
        return None
    if kind == "smear" and case["method"].startswith("multihit"):
        return None
    dims = _case_dims(case)
    u = _field(dims, nc, case["storage"], case["precision"], seed)
    if kind == "operators":
        return _exact_a0(u, case["rmax"], case["tmax"])
    if kind == "potential":
        u = _exact_ape(u, case["steps"])
    elif kind == "smear":
        u = {"ape": _exact_ape, "stout": _exact_stout, "hyp": _exact_hyp}[case["method"]](u, case["steps"])
    if kind == "smear" and case["links"]:
        return _to_host_order(u, dims)
    return _exact_loops(u, case["rmax"] if kind != "smear" else 4, case["tmax"] if kind != "smear" else 4)
