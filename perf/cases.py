"""The work that a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values.  ``prepare`` makes the system (coordinates,
charges, tables) from a seed and what a program keeps between calls: the
library context, the neighbour list, the captured graph of a period.  ``run``
is one pass through the public entry points of sponge_amd.

Kinds:
  md       one neighbour-list period of whole MD steps (forces, middle
           Langevin, SETTLE): what a trajectory spends its time on
  force    one neighbour-list period of force evaluations at fixed
           coordinates (the benchmark's own step), list rebuild included
  energy   one force step with energies and virials (printing and pressure)
  pair     the LJ + direct-space Coulomb module alone
  pme      the reciprocal module alone
  rebuild  a forced list rebuild with the reference-layout list written, and
           the pair forces from it (a refresh step of a drop-in host)
  batch    one period of a step batch over several water boxes (serving)
  f64      one all-FP64 force evaluation (precision studies)
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "sponge2.0_amd", "python"))

from sponge_amd.lib import Nonbonded, StepBatch  # noqa: E402
from sponge_amd.native_io import CHARGE_SCALE, box_to_cell  # noqa: E402

WATER_VOLUME = 29.915  # A^3 per TIP3P water at 1.0 g/cm^3
SKIN = 2.0
EWALD_TOLERANCE = 1e-5


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest serving segment: a period is bound by launches and latency
        _case("md", 500, 0, cutoff=9.0, graph=True, name="md_1500"),
        # 3,000 waters, the 9,000-atom NVT configuration, launched eagerly
        _case("md", 3000, 0, cutoff=10.0, graph=False, name="md_9000"),
        # the headline workload: 30,000 waters and 3,000 chain beads, PME 96^3
        _case("md", 30000, 3000, cutoff=10.0, graph=True, name="md_93000_mixed"),
        # a mid-size box that is not a cube, at the serving cutoff
        _case("force", 8333, 0, cutoff=9.0, graph=False, stretch=1.3, name="force_24999"),
        # 333,334 waters, list rebuilt every 20 steps, PME 216^3
        _case("force", 333334, 0, cutoff=10.0, graph=True, interval=20, name="force_1000002"),
        # the headline workload on a step that prints energies and pressure
        _case("energy", 30000, 3000, cutoff=10.0, name="energy_93000_mixed"),
        # single modules, as a host program calls them one by one
        _case("pair", 10000, 1003, cutoff=10.0, name="pair_31003"),
        _case("pme", 17501, 0, cutoff=9.0, energy=False, name="pme_52503"),
        _case("rebuild", 15000, 0, cutoff=10.0, name="rebuild_45000"),
        # eight segments of the serving stream in lockstep
        {"kind": "batch", "members": 8, "smallest": 1500, "largest": 40000, "cutoff": 9.0,
         "interval": 10, "name": "batch_8"},
        # one force evaluation of the FP64 trajectory of a precision study
        _case("f64", 3000, 0, cutoff=10.0, name="f64_9000"),
    ]


def _case(kind, waters, beads, cutoff, graph=False, interval=10, stretch=1.0, **more):
    """A case on one box of `waters` TIP3P waters and `beads` chain beads; the box is `stretch`
    times longer along z than along x."""
    return dict(kind=kind, waters=int(waters), beads=int(beads), cutoff=float(cutoff),
                graph=bool(graph), interval=int(interval), stretch=float(stretch), **more)


def draw(rng):
    kind = rng.choice(["md", "md", "force", "force", "energy", "pair", "pme", "rebuild", "batch",
                       "f64"])
    log = lambda a, b: math.exp(rng.uniform(math.log(a), math.log(b)))  # noqa: E731
    if kind == "batch":
        largest = int(log(6000, 50000))
        return {"kind": "batch", "members": rng.randint(2, 10), "smallest": rng.randint(1500, 3000),
                "largest": largest, "cutoff": 9.0, "interval": 10}
    top = {"md": 60000, "force": 200000, "energy": 60000, "pair": 100000, "pme": 200000,
           "rebuild": 60000, "f64": 8000}[kind]
    waters = int(log(500, top))
    beads = rng.choice([0, 0, rng.randint(20, 1 + waters // 10)])
    # a small box stays a cube: its edges are to hold twice the list radius
    stretch = rng.choice([1.0, 1.0, round(rng.uniform(1.0, 1.6), 2)]) if waters >= 1500 else 1.0
    more = {"energy": rng.random() < 0.5} if kind == "pme" else {}
    return _case(kind, waters, min(beads, 3000), cutoff=rng.choice([8.0, 9.0, 10.0]),
                 graph=rng.random() < 0.5, interval=rng.choice([10, 10, 20]), stretch=stretch,
                 **more)


# ---------------------------------------------------------------------------
# systems
# ---------------------------------------------------------------------------
def _smooth(n):
    """The smallest even 2-3-5-7-smooth number >= n."""
    n = int(math.ceil(n))
    while True:
        m = n
        for p in (2, 3, 5, 7):
            while m % p == 0:
                m //= p
        if m == 1 and n % 2 == 0:
            return n
        n += 1


def _box(case):
    """Box edges of a case: 1.0 g/cm^3 of water, the beads at the same volume per atom."""
    v = WATER_VOLUME * (case["waters"] + case["beads"] / 3.0)
    if case["waters"] == 30000 and case["beads"] == 3000:
        v = 96.5 ** 3  # the headline workload's box
    a = (v / case["stretch"]) ** (1.0 / 3.0)
    return np.array([a, a, a * case["stretch"]], np.float32)


def _grid(box):
    return tuple(_smooth(float(b) * 0.99) for b in box)


def _system(case, seed):
    """A TIP3P box with bead chains in the native conventions (charges x18.2223,
    LJ tables x12 / x6).  Waters sit on a jittered lattice in random
    orientations.  A chain is a zigzag (bond 1.53 A, angle 111 deg) along x
    that drifts in y so that its turns through the periodic box lie apart;
    every bead has an LJ type of its own, exclusions reach the third neighbour."""
    rng = np.random.default_rng(seed)
    nw, nb = case["waters"], case["beads"]
    box = _box(case)
    L = box.astype(np.float64)
    beads = np.zeros((0, 3))
    chain, index = np.zeros(0, int), np.zeros(0, int)
    if nb:
        step = 1.53 * math.sin(math.radians(55.5))
        # a chain's turns are at least 6 A apart in y
        most = max(20, min(1000, int(L[0] / step * (L[1] / 6.0 - 1.0))))
        nchain = -(-nb // most)
        per = -(-nb // nchain)
        chain, index = np.arange(nb) // per, np.arange(nb) % per
        turns = per * step / L[0]
        beads = np.stack([index * step, index * step / L[0] * (L[1] / (turns + 1.0)),
                          (chain + 0.5) / nchain * L[2]
                          + 0.5 * 1.53 * math.cos(math.radians(55.5)) * (2 * (index % 2) - 1)], 1)
        beads += rng.uniform(0, 1, 3) * L + rng.normal(0.0, 0.01, beads.shape)
        beads %= L
    # water sites: a lattice with enough of them clear of the beads
    per_axis = np.maximum(1, np.round(L / WATER_VOLUME ** (1 / 3.0)).astype(int))
    while True:
        if per_axis.prod() >= nw:
            g = [(np.arange(p) + 0.5) * (l / p) for p, l in zip(per_axis, L)]
            sites = np.stack(np.meshgrid(*g, indexing="ij"), -1).reshape(-1, 3)
            sites = (sites + rng.uniform(-0.15, 0.15, sites.shape)) % L
            if nb:
                sites = sites[_clear(sites, beads, L, 2.6)]
            if len(sites) >= nw:
                break
        per_axis[np.argmin(per_axis / L)] += 1
    sites = sites[np.sort(rng.permutation(len(sites))[:nw])]
    q = rng.normal(size=(nw, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    h = math.radians(104.52 / 2)
    crd = np.repeat(sites[:, None, :], 3, axis=1)
    for k, sgn in ((1, 1.0), (2, -1.0)):
        a, b = sgn * 0.9572 * math.sin(h), 0.9572 * math.cos(h)
        crd[:, k, 0] += a * (1 - 2 * (y * y + z * z)) + b * 2 * (x * y - z * w)
        crd[:, k, 1] += a * 2 * (x * y + z * w) + b * (1 - 2 * (x * x + z * z))
        crd[:, k, 2] += a * 2 * (x * z - y * w) + b * 2 * (y * z + x * w)
    crd = np.concatenate([crd.reshape(-1, 3), beads]) % L
    n = 3 * nw + nb
    qb = rng.normal(0.0, 0.3, nb)
    qb -= qb.mean() if nb else 0.0
    charge = np.concatenate([np.tile([-0.834, 0.417, 0.417], nw), qb]) * CHARGE_SCALE
    sig = np.concatenate([[3.15061, 0.0], rng.uniform(3.0, 4.0, nb)])
    eps = np.concatenate([[0.1521, 0.0], rng.uniform(0.02, 0.25, nb)])
    hi, lo = np.tril_indices(len(sig))
    s6 = (0.5 * (sig[hi] + sig[lo])) ** 6
    e4 = 4.0 * np.sqrt(eps[hi] * eps[lo])
    lj_a = (e4 * s6 * s6).astype(np.float32) * np.float32(12.0)
    lj_b = (e4 * s6).astype(np.float32) * np.float32(6.0)
    ltype = np.concatenate([np.tile([0, 1, 1], nw), 2 + np.arange(nb)]).astype(np.int32)
    mass = np.concatenate([np.tile([15.999, 1.008, 1.008], nw), np.full(nb, 14.027)])
    # exclusions: each list holds the higher ids, ascending
    length = np.bincount(chain) if nb else np.zeros(0, int)
    left = length[chain] - 1 - index if nb else np.zeros(0, int)
    num = np.concatenate([np.tile([2, 1, 0], nw), np.minimum(3, left)]).astype(np.int32)
    start = np.zeros(n, np.int32)
    start[1:] = np.cumsum(num)[:-1]
    at = np.repeat(np.arange(n), num)
    lst = (at + 1 + np.arange(len(at)) - start[at]).astype(np.int32)
    cell, rcell = box_to_cell(box)
    d = dict(n=n, crd=crd.astype(np.float32), charge=charge.astype(np.float32),
             lj_ntypes=len(sig), lj_a=lj_a, lj_b=lj_b, lj_type=ltype,
             mass=mass.astype(np.float32), box=box,
             angle=np.array([90.0, 90.0, 90.0], np.float32), cell=cell, rcell=rcell,
             excl_start=start, excl_numbers=num, excl_list=lst, cutoff=case["cutoff"],
             pme_grid=_grid(box), n_waters=nw)
    if nb:
        first = 3 * nw + np.arange(nb, dtype=np.int32)
        a14 = first[left >= 3]
        t1, t2 = ltype[a14], ltype[a14 + 3]
        p = np.maximum(t1, t2) * (np.maximum(t1, t2) + 1) // 2 + np.minimum(t1, t2)
        d["nb14"] = (a14, a14 + np.int32(3), np.float32(0.5) * lj_a[p], np.float32(0.5) * lj_b[p],
                     np.full(len(a14), 0.833, np.float32))
        ba = first[left >= 1]
        d["bonds"] = (ba, ba + np.int32(1), np.full(len(ba), 310.0, np.float32),
                      np.full(len(ba), 1.53, np.float32))
    return d


def _clear(sites, points, L, reach):
    """Which sites are at least `reach` from every point (minimum image)."""
    dev = torch.device("cuda")
    s = torch.as_tensor(sites, dtype=torch.float32, device=dev)
    p = torch.as_tensor(points, dtype=torch.float32, device=dev)
    box = torch.as_tensor(L, dtype=torch.float32, device=dev)
    ok = torch.empty(len(s), dtype=torch.bool, device=dev)
    for k in range(0, len(s), 16384):
        d = s[k:k + 16384, None, :] - p[None, :, :]
        d -= box * torch.round(d / box)
        ok[k:k + 16384] = d.square().sum(-1).amin(1) >= reach * reach
    return ok.cpu().numpy()


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
class _Groups:
    """The library's ATOM_GROUP array as int32[n][4] (numbers, ghosts, row pointer)."""

    def __init__(self, nb):
        self.__cuda_array_interface__ = {"shape": (nb.n, 4), "typestr": "<i4", "version": 3,
                                         "data": (nb.d_nl.value, False)}
        self.owner = nb


def _context(sysd, case, stream=None):
    # a corner cell takes the remainder of both the box edges: 256 atoms per cell
    return Nonbonded(sysd, cutoff=case["cutoff"], skin=SKIN, tolerance=EWALD_TOLERANCE,
                     refresh_interval=case["interval"], max_atom_in_grid_numbers=256,
                     stream=stream)


def _capture(nb, steps):
    """A HIP graph of the calls that steps() makes, recorded on a side stream."""
    graph, side, home = torch.cuda.CUDAGraph(), torch.cuda.Stream(), nb.stream
    nb.sync()
    torch.cuda.synchronize()
    nb.set_stream(side)
    try:
        with torch.cuda.graph(graph, stream=side):
            steps()
    finally:
        nb.set_stream(home)
    torch.cuda.synchronize()
    return graph


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed)
    sysd = _system(case, seed)
    nb = _context(sysd, case)
    st = {"case": case, "nb": nb, "k": case["interval"], "graph": None}
    if kind != "rebuild":
        nb.set_export(False)  # no other module reads the reference-layout list
    if kind == "md":
        nb.md_initial(sysd, temperature=300.0, tau=0.1, seed=seed % 100003, dt=0.002)
        for k in range(case["interval"]):
            nb.md_step(step=k, forced_nl=(k == 0))
    elif kind == "f64":
        st["crd64"] = nb.crd.double()
        st["frc64"] = torch.zeros_like(st["crd64"])
        nb.nl_update(forced=True)
    elif kind != "pme":
        nb.nl_update(forced=True)
        if kind == "rebuild":
            st["groups"] = torch.as_tensor(_Groups(nb), device="cuda")
        if kind in ("force", "energy"):
            nb.step(step=0)
    if case["graph"] and kind in ("md", "force"):
        st["graph"] = _capture(nb, lambda: _period(st))
    torch.cuda.synchronize()
    return st


def _period(st):
    nb, P = st["nb"], st["case"]["interval"]
    for k in range(st["k"], st["k"] + P):
        if st["case"]["kind"] == "md":
            nb.md_step(step=k)
        else:
            nb.frc.zero_()
            nb.step(step=k)
    st["k"] += P


def _sizes(case):
    m, a, b = case["members"], case["smallest"], case["largest"]
    return [max(2, int(round(a * (b / a) ** (k / max(1, m - 1)) / 3.0))) for k in range(m)]


def _member(case, waters):
    return _case("md", waters, 0, case["cutoff"], interval=case["interval"])


def _prepare_batch(case, seed):
    stream, nbs = torch.cuda.Stream(), []
    P = case["interval"]
    with torch.cuda.stream(stream):
        for k, w in enumerate(_sizes(case)):
            c = _member(case, w)
            s = _system(c, seed * 64 + k)
            nb = _context(s, c, stream=stream)
            nb.set_pme_overlap(False)
            nb.set_export(False)
            if nb.window_info()["windowed"]:
                nb.set_window_shape(2, 2, 2)
            nb.md_initial(s, temperature=300.0, tau=0.1, seed=(seed * 64 + k) % 100003, dt=0.002)
            for i in range(P):
                nb.md_step(step=i, forced_nl=(i == 0))
            nbs.append(nb)
        stream.synchronize()
        batch = StepBatch()
        for nb in nbs:
            batch.record(nb, P, P)
        batch.plan()
        batch.launch(stream)  # the plan's first period runs eagerly
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            batch.launch(stream)
    torch.cuda.synchronize()
    return {"case": case, "nbs": nbs, "batch": batch, "graph": graph}


def run(state):
    kind = state["case"]["kind"]
    if kind == "batch":
        state["graph"].replay()
        return {"crd": [nb.crd for nb in state["nbs"]], "vel": [nb.vel for nb in state["nbs"]]}
    nb = state["nb"]
    if kind in ("md", "force"):
        if state["graph"] is not None:
            state["graph"].replay()
        else:
            _period(state)
        return {"crd": nb.crd, "vel": nb.vel} if kind == "md" else {"frc": nb.frc}
    if kind == "f64":
        state["frc64"].zero_()
        nb.f64_force(state["crd64"], state["frc64"], step=0)
        return {"frc": state["frc64"]}
    if kind == "energy":
        nb.zero_outputs()
        nb.step(step=0, need_energy=True, need_virial=True)
        return {"frc": nb.frc, "atom_energy": nb.atom_energy, "direct": nb.direct_energy,
                "atom_virial": nb.atom_virial, "virial": nb.virial, "potential": nb.potential}
    nb.frc.zero_()
    if kind == "pme":
        ev = state["case"]["energy"]
        nb.virial.zero_()
        nb.potential.zero_()
        nb.reciprocal(step=0, need_energy=ev, need_virial=ev)
        return {"frc": nb.frc, "virial": nb.virial, "potential": nb.potential}
    if kind == "rebuild":
        nb.nl_update(forced=True)
    nb.lj_direct()
    return {"frc": nb.frc, "counts": state["groups"][:, 0]} if kind == "rebuild" else {
        "frc": nb.frc}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _step_work(case, kind):
    """Bytes and operations of one step: list entries (4 B each) and atom
    records read and forces written for the pair part, grids read and written
    once per pass of the reciprocal part, about 60 operations per pair within
    the cutoff, 5 N log2 N per transform."""
    box = _box(case).astype(np.float64)
    n = 3 * case["waters"] + case["beads"]
    rho = n / box.prod()
    ball = 2.0 / 3.0 * math.pi * rho * n
    entries, pairs = ball * (case["cutoff"] + SKIN) ** 3, ball * case["cutoff"] ** 3
    g = _grid(box)
    points = float(g[0] * g[1] * g[2])
    pair = (4.0 * entries + 44.0 * n, 60.0 * pairs)
    pme = (12.0 * points + 18.0 * points + 56.0 * n, 10.0 * points * math.log2(points) + 900.0 * n)
    build = (4.0 * entries + 32.0 * n, 12.0 * entries)
    if kind == "pair":
        return pair
    if kind == "pme":
        return pme
    if kind == "rebuild":
        return pair[0] + build[0], pair[1] + build[1]
    out = {"energy": 44.0 * n, "md": 52.0 * n, "f64": 48.0 * n}.get(kind, 24.0 * n)
    period = 1.0 / case["interval"] if kind in ("md", "force") else 0.0
    return (pair[0] + pme[0] + out + build[0] * period, pair[1] + pme[1] + build[1] * period)


def work(case):
    if case["kind"] == "batch":
        each = [_step_work(_member(case, w), "md") for w in _sizes(case)]
        return {"bytes": case["interval"] * sum(b for b, _ in each),
                "flops": case["interval"] * sum(f for _, f in each)}
    b, f = _step_work(case, case["kind"])
    steps = case["interval"] if case["kind"] in ("md", "force") else 1
    return {"bytes": b * steps, "flops": f * steps}


def tolerance(case):
    """Forces are sums of float terms in integers.  Against 64 bits the pair forces show 2e-6, and
    6e-6 where the transforms (or, with chains, the stretch of a bond) stand alone: about four
    times that.  The FP64 evaluation leaves the rounding of its sums at 2^-40."""
    if case["kind"] == "f64":
        return {"rel": 1e-9, "max": 1e-7}
    rel = 2.5e-5 if case["kind"] in ("pme", "energy") else 1e-5
    return {"rel": rel, "max": 40 * rel}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _beta(cutoff):
    """Ewald splitting with erfc(beta rc) / rc = tolerance, as a float."""
    lo, hi = 0.0, 5.0
    for _ in range(200):
        mid = 0.5 * (lo + hi)
        if math.erfc(mid * cutoff) / cutoff > EWALD_TOLERANCE:
            lo = mid
        else:
            hi = mid
    return float(np.float32(0.5 * (lo + hi)))


class _Exact:
    def __init__(self, case, seed):
        self.s = s = _system(case, seed)
        dev, f64 = torch.device("cuda"), torch.float64
        self.n, self.rc, self.beta = s["n"], case["cutoff"], _beta(case["cutoff"])
        self.x = torch.as_tensor(s["crd"], device=dev).to(f64)
        self.q = torch.as_tensor(s["charge"], device=dev).to(f64)
        self.L = torch.as_tensor(s["box"], device=dev).to(f64)
        self.t = torch.as_tensor(s["lj_type"], device=dev).long()
        self.A = torch.as_tensor(s["lj_a"], device=dev).to(f64)
        self.B = torch.as_tensor(s["lj_b"], device=dev).to(f64)
        num = torch.as_tensor(s["excl_numbers"], device=dev).long()
        self.ei = torch.repeat_interleave(torch.arange(self.n, device=dev), num)
        self.ej = torch.as_tensor(s["excl_list"], device=dev).long()
        z = lambda *k: torch.zeros(*k, dtype=f64, device=dev)  # noqa: E731
        self.frc, self.e, self.direct, self.vir = z(self.n, 3), z(self.n), z(self.n), z(self.n, 6)
        self.virial, self.potential = z(6), z(1)

    def disp(self, i, j):
        d = self.x[j] - self.x[i]
        return d - self.L * torch.round(d / self.L)

    def add(self, i, j, d, fa, e=None):
        """fa * d on i and its opposite on j; energy and virial of the pair on i."""
        f = fa[:, None] * d
        self.frc.index_add_(0, i, f)
        self.frc.index_add_(0, j, -f)
        if e is not None:
            self.e.index_add_(0, i, e)
        x, y, z = d.T
        u, v, w = f.T
        self.vir.index_add_(0, i, -torch.stack(
            [u * x, u * y + v * x, v * y, u * z + w * x, v * z + w * y, w * z], 1))

    def pair(self):
        n, dev = self.n, self.x.device
        rows = max(1, 24_000_000 // n)
        skip = self.ei * n + self.ej  # sorted
        idx = torch.arange(n, device=dev)
        for i0 in range(0, n, rows):
            i1 = min(n, i0 + rows)
            r2 = 0.0
            for c in range(3):
                d = self.x[None, i0:, c] - self.x[i0:i1, None, c]
                d -= self.L[c] * torch.round(d / self.L[c])
                r2 = r2 + d * d
            a, b = torch.nonzero((r2 < self.rc ** 2) & (idx[None, i0:] > idx[i0:i1, None]),
                                 as_tuple=True)
            i, j = a + i0, b + i0
            if len(skip):
                key = i * n + j
                at = torch.searchsorted(skip, key).clamp(max=len(skip) - 1)
                keep = skip[at] != key
                i, j = i[keep], j[keep]
            d = self.disp(i, j)
            r2 = d.square().sum(1)
            r = r2.sqrt()
            hi, lo = torch.maximum(self.t[i], self.t[j]), torch.minimum(self.t[i], self.t[j])
            p = hi * (hi + 1) // 2 + lo
            A, B, qq = self.A[p], self.B[p], self.q[i] * self.q[j]
            r6 = 1.0 / (r2 * r2 * r2)
            xb = self.beta * r
            ec = torch.special.erfc(xb)
            h = ec + 2.0 / math.sqrt(math.pi) * xb * torch.exp(-xb * xb)
            dir_e = qq * ec / r
            self.direct.index_add_(0, i, dir_e)
            self.add(i, j, d, (B - A * r6) * r6 / r2 - qq * h / (r2 * r),
                     (A / 12.0 * r6 - B / 6.0) * r6 + dir_e)

    def excluded(self):
        d = self.disp(self.ei, self.ej)
        r = d.square().sum(1).sqrt()
        xb, qq = self.beta * r, self.q[self.ei] * self.q[self.ej]
        erf = torch.special.erf(xb)
        g = 2.0 / math.sqrt(math.pi) * xb * torch.exp(-xb * xb)
        self.add(self.ei, self.ej, d, qq * (erf - g) / r ** 3, -qq * erf / r)

    def bonded(self):
        if "nb14" in self.s:
            a, b, A, B, cf = (torch.as_tensor(v, device=self.x.device) for v in self.s["nb14"])
            a, b, A, B, cf = a.long(), b.long(), A.double(), B.double(), cf.double()
            d = self.disp(a, b)
            r2 = d.square().sum(1)
            qq = cf * self.q[a] * self.q[b]
            self.add(a, b, d, -A / r2 ** 7 + B / r2 ** 4 - qq / r2 ** 1.5,
                     qq / r2.sqrt() + 0.08333333 * A / r2 ** 6 - 0.1666666 * B / r2 ** 3)
        if "bonds" in self.s:
            a, b, k, r0 = (torch.as_tensor(v, device=self.x.device) for v in self.s["bonds"])
            a, b, k, r0 = a.long(), b.long(), k.double(), r0.double()
            d = self.disp(a, b)
            r = d.square().sum(1).sqrt()
            self.add(a, b, d, 2.0 * k * (r - r0) / r, k * (r - r0) ** 2)

    def reciprocal(self):
        dev, f64 = self.x.device, torch.float64
        fx, fy, fz = g = self.s["pme_grid"]
        L, V = self.L, float(self.L.prod())
        F = torch.tensor(g, dtype=f64, device=dev)
        u = self.x / L
        u = (u - torch.floor(u)) * F
        base = torch.minimum(torch.floor(u), F - 1)
        t = (u - base)
        w = [t ** 3 / 6, -t ** 3 / 2 + t ** 2 / 2 + t / 2 + 1 / 6.0, t ** 3 / 2 - t ** 2 + 4 / 6.0,
             -t ** 3 / 6 + t ** 2 / 2 - t / 2 + 1 / 6.0]
        dw = [t ** 2 / 2, -1.5 * t ** 2 + t + 0.5, 1.5 * t ** 2 - 2 * t, -0.5 * t ** 2 + t - 0.5]
        base = base.long()

        def points():
            for kx in range(4):
                for ky in range(4):
                    for kz in range(4):
                        k = (kx, ky, kz)
                        p = [torch.remainder(base[:, c] - k[c], g[c]) for c in range(3)]
                        yield k, (p[0] * fy + p[1]) * fz + p[2]
        Q = torch.zeros(fx * fy * fz, dtype=f64, device=dev)
        for k, at in points():
            Q.index_add_(0, at, self.q * w[k[0]][:, 0] * w[k[1]][:, 1] * w[k[2]][:, 2])
        S = torch.fft.rfftn(Q.view(fx, fy, fz))
        fc = fz // 2 + 1
        m, b = [], []
        for c, num in enumerate(g):
            k = torch.arange(num, dtype=f64, device=dev)
            ang = 2.0 * math.pi * k / num
            re = 1 / 6.0 + 2 / 3.0 * torch.cos(ang) + 1 / 6.0 * torch.cos(2 * ang)
            im = 2 / 3.0 * torch.sin(ang) + 1 / 6.0 * torch.sin(2 * ang)
            b.append(1.0 / (re * re + im * im))
            m.append(torch.where(k > num // 2, k - num, k) / L[c])
        mx, my, mz = m[0][:, None, None], m[1][None, :, None], m[2][None, None, :fc]
        msq = mx * mx + my * my + mz * mz
        msq[0, 0, 0] = 1.0
        mpre = math.pi ** 2 / self.beta ** 2
        bc = torch.exp(-mpre * msq) / (math.pi * msq * V) * \
            b[0][:, None, None] * b[1][None, :, None] * b[2][None, None, :fc]
        bc[0, 0, 0] = 0.0
        a2 = (S.real ** 2 + S.imag ** 2) * bc
        full = torch.full((fc,), 2.0, dtype=f64, device=dev)
        full[0] = 1.0
        if fz % 2 == 0:
            full[-1] = 1.0
        half = torch.ones(fc, dtype=f64, device=dev)
        half[0] = half[-1] = 0.5
        hb, cf = half * 0.5 * a2, 2.0 / msq * (1.0 + mpre * msq)
        self.virial += -torch.stack([
            (hb * (one - cf * p * r)).sum() for one, p, r in (
                (1.0, mx, mx), (0.0, my, mx), (1.0, my, my), (0.0, mz, mx), (0.0, mz, my),
                (1.0, mz, mz))])
        self.potential += 0.5 * (full * a2).sum() - self.beta / math.sqrt(math.pi) * \
            self.q.square().sum() - 0.5 * math.pi / (self.beta ** 2 * V) * self.q.sum() ** 2
        phi = torch.fft.irfftn(S * bc, s=g, norm="forward").reshape(-1)
        for k, at in points():
            p = phi[at]
            for c in range(3):
                v = [dw[k[a]][:, a] if a == c else w[k[a]][:, a] for a in range(3)]
                self.frc[:, c] -= self.q * p * v[0] * v[1] * v[2] * F[c] / L[c]

    def long_range(self):
        hist = torch.bincount(self.t, minlength=self.s["lj_ntypes"]).double()
        hi, lo = np.tril_indices(self.s["lj_ntypes"])
        hi, lo = torch.as_tensor(hi, device=self.x.device), torch.as_tensor(lo, device=self.x.device)
        c6 = (hist[hi] * hist[lo] * self.B * torch.where(hi == lo, 1.0, 2.0)).sum()
        f = c6 * (-2.0 / 3.0 * math.pi / self.rc ** 3 / 6.0) / self.L.prod()
        self.potential += f
        self.virial += 2.0 * f * torch.tensor([1.0, 0, 1.0, 0, 0, 1.0], device=self.x.device)


def exact(case, seed):
    # a thermostatted period has noise of the library's own; a million atoms take too long
    if case["kind"] in ("md", "batch") or case["waters"] > 60000:
        return None
    E, kind = _Exact(case, seed), case["kind"]
    if kind != "pme":
        E.pair()
    if kind in ("force", "energy", "f64"):
        E.excluded()
        E.bonded()
    if kind in ("force", "energy", "f64", "pme"):
        E.reciprocal()
    if kind == "pme" and not case["energy"]:
        E.virial.zero_()
        E.potential.zero_()
    if kind == "energy":
        E.long_range()
        return {"frc": E.frc, "atom_energy": E.e, "direct": E.direct, "atom_virial": E.vir,
                "virial": E.virial, "potential": E.potential}
    if kind == "pme":
        return {"frc": E.frc, "virial": E.virial, "potential": E.potential}
    return {"frc": E.frc, "counts": None} if kind == "rebuild" else {"frc": E.frc}
