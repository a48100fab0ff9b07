"""The calls whose speed this library is judged by, with inputs made from a seed.

A case is one call of the public interface on one system: an (T) energy of an
uploaded job, a job taken from host blocks to its energies, the Lambda- and
CR-CCSD(T) energies, the t3 tiles of one task, one task through the
reference's per-call surface, a batch of small jobs.  `prepare` makes what a
program holds before the call (TCE blocks on the host, uploaded jobs, a
planned batch), `run` makes the call, `work` counts what it cannot do
without, `exact` gives the same outputs from plain FP64 matrix products.

The block files are random numbers in the layout of tce_t1_offset.F,
tce_t2_offset.F and tce_mo2e_offset.F: one canonical block per allowed tile
tuple in loop order, antisymmetric inside a pair of equal tiles, with the
amplitude and integral scales of the library's synthetic generator.
"""
from __future__ import annotations

import ctypes as C
import itertools
import math

import numpy as np
import torch

import nwchem_amd
from nwchem_amd.job import TILING_ORBITAL, TriplesBatch, TriplesJob, cr_ccsd_t, lambda_ccsd_t
from nwchem_amd.tiles import Blocks, TileModel

DEV = "cuda" if torch.cuda.is_available() else "cpu"
PRECISION = {"fp64": 0, "fp32": 1, "bf16x3": 2, "bf16x6": 3}


def _system(kind, name, no, nv, to, tv, precision="fp64", spins=1, irreps=1, restricted=False,
            tiling="default"):
    c = {"kind": kind, "no": no, "nv": nv, "to": to, "tv": tv, "spins": spins, "irreps": irreps,
         "restricted": restricted, "tiling": tiling, "precision": precision}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest job of the tests and the smoke run: 4 tasks, launch and latency bound
        _system("energy", "energy_no8_nv32", 8, 32, 8, 16),
        # a ragged job of the batch workload's sizes on its own
        _system("energy", "energy_ragged_no21_nv160", 21, 160, 16, 37),
        # the benchmark's tiling (occupied tiles of 20, virtual tiles of 40) at half its virtuals
        _system("energy", "energy_no40_nv160", 40, 160, 20, 40),
        # a closed-shell molecule as NWChem tiles it: alpha and beta tiles, restricted blocks
        _system("energy", "energy_restricted_no26_nv114", 26, 114, 13, 19, spins=2,
                restricted=True),
        # the benchmark's orbitals with spin and irrep labels (2 spins x 4 irreps)
        _system("energy", "energy_irreps_no40_nv320", 40, 320, 5, 40, spins=2, irreps=4),
        # split-BF16 with FP64-like energies, what large jobs are run in
        _system("energy", "energy_bf16x6_no40_nv200", 40, 200, 20, 40, "bf16x6"),
        # one (T) as a CCSD program calls it: blocks on the host, plan, upload, energies
        _system("cold", "cold_no20_nv80", 20, 80, 10, 20),
        # Lambda-CCSD(T): two jobs, Fock term
        _system("lambda", "lambda_no20_nv80", 20, 80, 10, 20),
        # CR-CCSD(T) after its intermediates
        _system("cr", "cr_no16_nv72", 16, 72, 8, 24),
        # t3 tiles of one task left in HBM for a consumer on the GPU
        _system("tiles", "tiles_no24_nv96", 24, 96, 12, 24),
        # one task of ccsd_t_gpu.F's loop through the reference-named entry points
        {"kind": "percall", "name": "percall_h12_p24", "h1": 12, "h2": 12, "h3": 12, "p4": 24,
         "p5": 24, "p6": 24},
        # small jobs together: each underfills the GPU alone
        {"kind": "batch", "name": "batch_24_small_jobs", "jobs": 24, "mix": 1, "no_lo": 6,
         "no_hi": 10, "nv_lo": 48, "nv_hi": 64, "precision": "fp64"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any size between the smallest and the largest listed
    ones, every label and precision a job can have, at most the work of the
    largest listed case of its kind."""
    kind = rng.choice(["energy"] * 6 + ["cold", "lambda", "cr", "tiles", "percall", "batch"])
    if kind == "percall":
        c = {"kind": kind}
        for k in ("h1", "h2", "h3"):
            c[k] = rng.randint(3, 13)
        for k in ("p4", "p5", "p6"):
            c[k] = rng.randint(5, 24)
        return c
    if kind == "batch":
        lo = rng.randint(6, 8)
        return {"kind": kind, "jobs": _log_uniform(rng, 4, 24), "mix": rng.randint(2, 10 ** 6),
                "no_lo": lo, "no_hi": rng.randint(lo, 10), "nv_lo": 48,
                "nv_hi": rng.randint(50, 64), "precision": "fp64"}
    top = {"energy": 160, "cold": 100, "lambda": 80, "cr": 80, "tiles": 96}[kind]
    while True:
        spins = rng.choice([1, 2])
        irreps = rng.choice([1, 1, 2, 4]) if spins == 2 else 1
        precision = "fp64"
        if kind == "energy":
            precision = rng.choice(["fp64", "fp64", "fp64", "fp32", "bf16x3", "bf16x6"])
        # reduced precision is for the jobs that take long in FP64
        no = _log_uniform(rng, 6 if precision == "fp64" else 16, 40 if kind == "energy" else 24)
        nv = _log_uniform(rng, 24 if precision == "fp64" else 96, 2 * top if irreps > 1 else top)
        no, nv = no + no % spins, nv + nv % spins
        if no < 2 * spins * irreps or nv < 4 * spins * irreps:
            continue
        restricted = spins == 2 and rng.random() < 0.5
        group = no // spins // irreps
        c = _system(kind, None, no, nv, rng.randint(max(2, group // 3), max(4, min(20, group))),
                    rng.randint(max(6, nv // spins // irreps // 5), 40), precision, spins, irreps,
                    restricted, rng.choice(["default", "default", "orbital"])
                    if kind in ("energy", "cold") else "default")
        if c["to"] * 8 < group or work(c)["flops"] > 1.7e13:
            continue
        if kind == "tiles":
            c["to"], c["tv"] = min(c["to"], 12), min(c["tv"], 24)
        return c


# ---------------------------------------------------------------- tiles and block tables


class _Tiling:
    """Tile lists of a system: alpha (and beta) holes, then particles, each
    spin cut by irrep and into tiles that differ by at most one orbital."""

    def __init__(self, c):
        self.no, self.nv, self.restricted = c["no"], c["nv"], bool(c["restricted"])
        spins, irreps = c["spins"], c["irreps"]
        rng, spin, sym, alpha = [], [], [], []
        for n, ts in ((self.no, c["to"]), (self.nv, c["tv"])):
            self.noab = first = len(rng)
            for s in range(1, spins + 1):
                at = 0
                for g in range(irreps):
                    k = n // spins // irreps + (1 if g < n // spins % irreps else 0)
                    if k == 0:
                        continue
                    nt = -(-k // ts)
                    for t in range(nt):
                        rng.append(k // nt + (1 if t < k % nt else 0))
                        spin.append(s)
                        sym.append(g)
                        alpha.append(first + at + 1)
                        at += 1
        self.rng, self.spin, self.sym, self.alpha = rng, spin, sym, alpha
        self.nvab = len(rng) - self.noab
        self.ofs = [0] + list(itertools.accumulate(rng))[:-1]
        self.O, self.V = range(1, self.noab + 1), range(self.noab + 1, len(rng) + 1)

    def r(self, *tiles):
        return [self.rng[b - 1] for b in tiles]

    def at(self, b):
        """Orbitals of tile b within its space."""
        o = self.ofs[b - 1] - (self.no if b > self.noab else 0)
        return slice(o, o + self.rng[b - 1])

    def conserved(self, left, right):
        y = 0
        for b in (*left, *right):
            y ^= self.sym[b - 1]
        return y == 0 and sum(self.spin[b - 1] for b in left) == sum(self.spin[b - 1] for b in right)

    def stored(self, left, right):
        s = sum(self.spin[b - 1] for b in (*left, *right))
        return self.conserved(left, right) and not (self.restricted and s == 2 * len(left + right))

    def image(self, *tiles):
        """All-beta blocks of a restricted run are read from their alpha images."""
        if self.restricted and all(self.spin[b - 1] == 2 for b in tiles):
            return tuple(self.alpha[b - 1] for b in tiles)
        return tiles

    def tasks(self):
        for p in itertools.combinations_with_replacement(self.V, 3):
            for h in itertools.combinations_with_replacement(self.O, 3):
                s = sum(self.spin[b - 1] for b in p + h)
                if self.conserved(p, h) and not (self.restricted and s > 8):
                    yield p + h

    def factor(self, t):
        f = 2.0 if self.restricted else 1.0
        for x in (t[:3], t[3:]):
            f /= {1: 6.0, 2: 2.0, 3: 1.0}[len(set(x))]
        return f

    def model(self, evl):
        return TileModel(range=np.array(self.rng), noab=self.noab, evl=evl,
                         spin=np.array(self.spin), sym=np.array(self.sym),
                         alpha=np.array(self.alpha), restricted=self.restricted)


def _pairs(tiles):
    return itertools.combinations_with_replacement(tiles, 2)


class _File:
    """A block file: the hash table [L, keys, offsets] and the blocks'
    random values, antisymmetric in equal tiles of a pair."""

    def __init__(self, T, blocks, sigma, gen):
        """blocks: (key, tiles, pairs of axes that are antisymmetric)"""
        self.at, off = {}, 0
        for key, tiles, _ in blocks:
            self.at[tiles] = off
            off += math.prod(T.r(*tiles))
        self.hash = np.array([len(blocks), *(b[0] for b in blocks), *self.at.values()], np.int64)
        x = torch.randn(max(off, 1), generator=gen, device=DEV, dtype=torch.float64).mul_(sigma)
        for _, tiles, anti in blocks:
            for i, j in anti:
                if tiles[i] == tiles[j]:
                    shape = T.r(*tiles)
                    v = x[self.at[tiles]:self.at[tiles] + math.prod(shape)].view(shape)
                    v.copy_((v - v.transpose(i, j)) * 0.5 ** 0.5)
        self.device, self.host = x, x.cpu().numpy()

    def block(self, T, tiles):
        shape, o = T.r(*tiles), self.at[tiles]
        return self.device[o:o + math.prod(shape)].view(shape)


class _Inputs:
    """Orbital energies and block files of a system, by the kind of call."""

    def __init__(self, c, seed):
        self.T = T = _Tiling(c)
        g = torch.Generator(device=DEV)
        g.manual_seed(int(seed))
        r = np.random.default_rng(int(seed))
        spins = c["spins"]
        eo = np.sort(r.uniform(-2.0, -0.3, T.no // spins))
        ev = np.sort(r.uniform(0.2, 4.0, T.nv // spins))
        self.evl = np.concatenate([eo] * spins + [ev] * spins)
        O, V, noab, nvab = T.O, T.V, T.noab, T.nvab
        N = noab + nvab

        def key(base, digits):
            k = 0
            for d, b in zip(digits, base):
                k = k * b + d
            return k

        p, h = lambda b: b - noab - 1, lambda b: b - 1  # noqa: E731
        t1 = [(p(a) * noab + h(i), (a, i), ()) for a in V for i in O if T.stored((a,), (i,))]
        t2 = [(key((nvab, nvab, noab, noab), (p(a), p(b), h(i), h(j))), (a, b, i, j),
               ((0, 1), (2, 3)))
              for a, b in _pairs(V) for i, j in _pairs(O) if T.stored((a, b), (i, j))]
        self.t1, self.t2 = _File(T, t1, 0.01, g), _File(T, t2, 0.02, g)
        v2 = []
        for g3, g4 in _pairs(range(1, N + 1)):
            if g4 <= noab:
                continue
            ket = _pairs(O) if g3 <= noab else itertools.chain.from_iterable(
                (((i, x) for x in range(i, N + 1)) for i in O))
            anti = ((2, 3),) if g3 <= noab else None
            for g1, g2 in ket:
                if T.stored((g3, g4), (g1, g2)):
                    v2.append((key((N,) * 4, (h(g3), h(g4), h(g1), h(g2))), (g3, g4, g1, g2),
                               anti or ((0, 1),) + (((2, 3),) if g2 <= noab else ())))
        self.v2 = _File(T, v2, 0.05, g)
        if c["kind"] == "lambda":
            y1 = [(h(i) * nvab + p(a), (i, a), ()) for i in O for a in V if T.stored((i,), (a,))]
            y2 = [(key((noab, noab, nvab, nvab), (h(i), h(j), p(a), p(b))), (i, j, a, b),
                   ((0, 1), (2, 3)))
                  for i, j in _pairs(O) for a, b in _pairs(V) if T.stored((i, j), (a, b))]
            f1 = [(h(x) * N + h(y), (x, y), ()) for x in range(1, N + 1) for y in range(1, N + 1)
                  if T.stored((x,), (y,))]
            self.y1, self.y2 = _File(T, y1, 0.01, g), _File(T, y2, 0.02, g)
            self.f1 = _File(T, f1, 0.1, g)
        if c["kind"] == "cr":
            a1 = [(key((nvab, noab, noab, noab), (p(a), h(m), h(i), h(j))), (a, m, i, j), ((2, 3),))
                  for a in V for m in O for i, j in _pairs(O) if T.stored((m, a), (i, j))]
            a2 = [(key((nvab, nvab, noab, nvab), (p(a), p(b), h(i), p(e))), (a, b, i, e), ((0, 1),))
                  for a, b in _pairs(V) for i in O for e in V if T.stored((a, b), (i, e))]
            self.i1, self.i2 = _File(T, a1, 0.05, g), _File(T, a2, 0.05, g)

    def host(self):
        """What a program keeps: the host copies only."""
        for f in vars(self).values():
            if isinstance(f, _File):
                f.device = None
        if torch.cuda.is_available():
            torch.cuda.empty_cache()
        self.blocks = Blocks(self.t1.host, self.t1.hash, self.t2.host, self.t2.hash, self.v2.host,
                             self.v2.hash)
        self.model = self.T.model(self.evl)
        return self


# ------------------------------------------------------------------------- the calls

_NAMES = ("h3", "h2", "h1", "p6", "p5", "p4")  # the t3 tile, fastest index first
# triplesx layouts (fastest first) and signs of the 27 contractions, ccsd_t_kernels_omp.F:5-1198
_HOLES = {"s1": ("h3 h2 h1", "h3 h1 h2", "h1 h3 h2"), "d1": ("h3 h2 h1", "h3 h1 h2", "h1 h3 h2"),
          "d2": ("h3 h2 h1", "h2 h1 h3", "h2 h3 h1")}
_PARTICLES = {"s1": ("p6 p5 p4", "p6 p4 p5", "p4 p6 p5"), "d1": ("p6 p5 p4", "p5 p4 p6", "p5 p6 p4"),
              "d2": ("p6 p5 p4", "p6 p4 p5", "p4 p6 p5")}
_SIGN = {"s1": (1, -1, 1, -1, 1, -1, 1, -1, 1), "d1": (-1, 1, -1, -1, 1, -1, 1, -1, 1),
         "d2": (-1, -1, 1, 1, 1, -1, -1, -1, 1)}
# operands, fastest index first (x: the contraction index)
_OPERANDS = {"s1": ("p4 h1", "h3 h2 p6 p5"), "d1": ("x p4 p5 h1", "h3 h2 p6 x"),
             "d2": ("x p4 h1 h2", "x h3 p6 p5")}


def _percall(c, seed):
    """(family, n, extents by name, t operand, v operand) of the 27 calls of
    one task, and its orbital energies."""
    r = np.random.default_rng(int(seed))
    tile = [c[k] for k in _NAMES]
    calls = []
    for fam in ("s1", "d1", "d2"):
        for n in range(9):
            layout = (_HOLES[fam][n % 3] + " " + _PARTICLES[fam][n // 3]).split()
            ext = dict(zip(layout, tile))
            ext["x"] = c["h1"] if fam == "d1" else c["p4"]
            a, b = ([ext[k] for k in op.split()] for op in _OPERANDS[fam])
            calls.append((fam, n, ext, r.standard_normal(a[::-1]) * 0.02,
                          r.standard_normal(b[::-1]) * 0.05))
    evl = [np.sort(r.uniform(-2.0, -0.3, c[k])) for k in ("h1", "h2", "h3")]
    evl += [np.sort(r.uniform(0.2, 4.0, c[k])) for k in ("p4", "p5", "p6")]
    return calls, evl


def _batch_systems(c):
    """Sizes and tiles of a batch's jobs (fixed by the case, not by the seed)."""
    r = np.random.default_rng(c["mix"])
    for _ in range(c["jobs"]):
        no = int(r.integers(c["no_lo"], c["no_hi"] + 1))
        nv = int(r.integers(c["nv_lo"], c["nv_hi"] + 1))
        yield _system("energy", None, no, nv, min(no, int(r.integers(6, 11))),
                      int(r.integers(16, 33)), c["precision"], tiling="orbital")


def _job(c, X):
    job = TriplesJob(X.model, tiling=TILING_ORBITAL if c["tiling"] == "orbital" else None)
    job.upload(X.blocks)
    return job


def _task(T):
    """The task the tile export runs on: distinct tiles where there are enough."""
    return max(T.tasks(), key=lambda t: (len(set(t)), t))


def prepare(case, seed):
    c = dict(case)
    nwchem_amd.init(0)
    if c["kind"] == "percall":
        calls, evl = _percall(c, seed)
        return {"c": c, "calls": calls, "evl": evl}
    if c["kind"] == "batch":
        jobs = []
        for k, s in enumerate(_batch_systems(c)):
            jobs.append(_job(s, _Inputs(s, seed * 1000 + k).host()))
        batch = TriplesBatch(jobs)
        batch.run(PRECISION[c["precision"]])  # plans and captures the launch
        return {"c": c, "batch": batch}
    X = _Inputs(c, seed).host()
    st = {"c": c, "prec": PRECISION[c["precision"]]}
    if c["kind"] == "cold":
        return dict(st, X=X)
    st["job"] = job = _job(c, X)
    if c["kind"] == "lambda":
        st["other"] = TriplesJob(X.model)
        st["other"].upload_lambda(X.y1.host, X.y1.hash, X.y2.host, X.y2.hash, X.v2.host, X.v2.hash)
        st["f1"], st["f1h"] = X.f1.host, X.f1.hash
    if c["kind"] == "cr":
        st["other"] = TriplesJob(X.model)
        st["other"].upload_cr(X.t1.host, X.t1.hash, X.t2.host, X.t2.hash, X.i1.host, X.i1.hash,
                              X.i2.host, X.i2.hash)
    if c["kind"] == "tiles":
        st["task"] = _task(X.T)
    if c["precision"] != "fp64":
        job.operands(st["prec"], 2)  # the reduced-precision copies a program keeps
    return st


class _DeviceArray:
    """An array in the job's tile buffer."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False),
                                         "version": 3}

    def tensor(self, job):
        x = torch.as_tensor(self, device="cuda")
        x.job = job  # the buffer lives as long as the job
        return x


def _energies(job, prec, tiling):
    e = job.run(prec)
    out = {"e_bt": e[0], "e_pt": e[1]}
    if tiling != "orbital":
        out["tasks"] = job.task_energies()
    return out


def run(state):
    c = state["c"]
    kind = c["kind"]
    if kind == "energy":
        return _energies(state["job"], state["prec"], c["tiling"])
    if kind == "cold":
        with _job(c, state["X"]) as job:
            return _energies(job, state["prec"], c["tiling"])
    if kind == "lambda":
        e1, e2, te = lambda_ccsd_t(state["job"], state["other"], state["f1"], state["f1h"],
                                   precision=state["prec"])
        return {"e1": e1, "e2": e2, "tasks": te}
    if kind == "cr":
        e1, e2, terms = cr_ccsd_t(state["job"], state["other"], state["prec"])
        return {"e1": e1, "e2": e2, "terms": terms}
    if kind == "tiles":
        p4, p5, p6, h1, h2, h3 = state["task"]
        s, d, n = state["job"].triples_tiles_device(h1, h2, h3, p4, p5, p6, state["prec"])
        return {"singles": _DeviceArray(s, n).tensor(state["job"]),
                "doubles": _DeviceArray(d, n).tensor(state["job"])}
    if kind == "batch":
        return {"energies": state["batch"].run(PRECISION[c["precision"]])}
    # percall: one pass of the task loop of ccsd_t_gpu.F with usedevice = 1
    L, dp = nwchem_amd.lib(), C.POINTER(C.c_double)
    dims = [C.byref(C.c_long(c[k])) for k in ("h1", "h2", "h3", "p4", "p5", "p6")]
    L.dev_mem_d_(*dims)
    L.dev_mem_s_(*dims)
    for fam, n, ext, a, b in state["calls"]:
        names = {"s1": "h1 h2 h3 p4 p5 p6", "d1": "h1 h2 h3 x p4 p5 p6",
                 "d2": "h1 h2 h3 p4 p5 p6 x"}[fam].split()
        args = [C.byref(C.c_long(ext[k])) for k in names]
        getattr(L, f"sd_t_{fam}_{n + 1}_cuda_")(*args, None, a.ctypes.data_as(dp),
                                                 b.ctypes.data_as(dp))
    energy = np.zeros(2)
    L.compute_en_(C.byref(C.c_double(1.0)), energy.ctypes.data_as(dp),
                  *[e.ctypes.data_as(dp) for e in state["evl"]], *dims, None, None)
    L.dev_release_()
    return {"energy": energy}


# ------------------------------------------------------------- what a pass cannot do without


def _unique(T, t):
    """t3 elements of task t that differ by more than a sign: a < b < c and
    i < j < k inside equal tiles."""
    n = 1
    for x in (t[:3], t[3:]):
        for b in set(x):
            n *= math.comb(T.rng[b - 1], x.count(b))
    return n


def _contracted(T, t):
    """Flops of one element's 18 d1/d2 and 9 s1 contractions, over the
    orbitals that spin and irrep allow."""
    classes = {}
    for b in range(1, T.noab + T.nvab + 1):
        k = (b > T.noab, T.spin[b - 1], T.sym[b - 1])
        classes[k] = classes.get(k, 0) + T.rng[b - 1]
    f = 18
    for L in t[:3]:
        for r, s in itertools.combinations(t[3:], 2):
            spin = T.spin[r - 1] + T.spin[s - 1] - T.spin[L - 1]
            sym = T.sym[r - 1] ^ T.sym[s - 1] ^ T.sym[L - 1]
            f += 2 * sum(classes.get((v, spin, sym), 0) for v in (False, True))
    return f


def work(case):
    c = dict(case)
    if c["kind"] == "percall":
        n = math.prod(c[k] for k in _NAMES)
        return {"flops": 18.0 * n * (1 + c["h1"] + c["p4"]) + 12.0 * n,
                "bytes": 8.0 * sum(a.size + b.size for _, _, _, a, b in _percall(c, 0)[0])}
    if c["kind"] == "batch":
        w = [work(s) for s in _batch_systems(c)]
        return {k: sum(x[k] for x in w) for k in ("flops", "bytes")}
    T = _Tiling(c)
    files = sum(math.prod(T.r(*b)) for b in itertools.product(T.V, T.O) if T.stored(b[:1], b[1:]))
    for left, right in ((_pairs(T.V), lambda: _pairs(T.O)), (_pairs(T.V), lambda: _pairs(T.O)),
                        (itertools.product(T.O, T.V), lambda: _pairs(T.O)),
                        (_pairs(T.V), lambda: itertools.product(T.O, T.V))):
        for l in left:
            files += sum(math.prod(T.r(*l, *r)) for r in right() if T.stored(l, r))
    sides = 2 if c["kind"] in ("lambda", "cr") else 1
    if c["kind"] == "tiles":
        t = _task(T)
        n = math.prod(T.r(*t))
        return {"flops": float(n * _contracted(T, t)), "bytes": 16.0 * n}
    return {"flops": float(sides * sum(_unique(T, t) * _contracted(T, t) for t in T.tasks())),
            "bytes": 8.0 * sides * files}


# ------------------------------------------------------------------ the same in plain FP64


def _dense(T, f, left, right, axes, anti_left, anti_right):
    """The dense tensor of a file over the spaces of `left` and `right` (lists
    of tiles): every tile tuple from its canonical block with the sign of the
    exchanges.  axes: the block's index order as positions of (left, right)."""
    space = {True: T.no, False: T.nv}
    x = torch.zeros([space[s[0] <= T.noab] for s in (*left, *right)], dtype=torch.float64,
                    device=DEV)
    for t in itertools.product(*left, *right):
        n = len(left)
        if not T.conserved(t[:n], t[n:]):
            continue
        u, sign, perm = list(t), 1.0, list(range(len(t)))
        for pair in ((0, 1),) * anti_left + ((2, 3),) * anti_right:
            if u[pair[0]] > u[pair[1]]:
                for v in (u, perm):
                    v[pair[0]], v[pair[1]] = v[pair[1]], v[pair[0]]
                sign = -sign
        u = T.image(*u)
        blk = f.block(T, tuple(u[k] for k in axes))
        blk = blk.permute([axes.index(k) for k in range(len(t))])  # in (left, right) order
        x[tuple(T.at(b) for b in t)] = sign * blk.permute(perm)
    return x


class _Exact:
    """t3 tiles (singles, doubles) of tasks from dense tensors."""

    def __init__(self, T, t1, t2, W, V, S):
        self.T, self.t1, self.S = T, t1, S
        # contraction index e then m, last: X[L][r][s], Y[p1][p2][h]
        self.X = torch.cat([t2.permute(0, 2, 3, 1), W.permute(1, 2, 3, 0)], 3)
        self.Y = torch.cat([V, t2], 3)

    def tile(self, task):
        T = self.T
        at = [T.at(b) for b in task]
        d = s = 0.0
        for L, sL in ((0, -1.0), (1, 1.0), (2, -1.0)):
            q = [x for x in (0, 1, 2) if x != L]
            for h, sh in ((5, 1.0), (4, -1.0), (3, 1.0)):
                r = [x for x in (3, 4, 5) if x != h]
                x = self.X[at[L], at[r[0]], at[r[1]]]
                y = self.Y[at[q[0]], at[q[1]], at[h]]
                w = x.reshape(-1, x.shape[3]) @ y.reshape(-1, y.shape[3]).T
                u = self.t1[at[L], at[h]]
                v = self.S[at[q[0]], at[q[1]], at[r[0]], at[r[1]]]
                w = w.view(*x.shape[:3], *y.shape[:3])
                order = (L, r[0], r[1], q[0], q[1], h)
                d = d + sL * sh * w.permute([order.index(k) for k in range(6)])
                order = (L, h, q[0], q[1], r[0], r[1])
                w = (u.reshape(-1, 1) * v.reshape(1, -1)).view(*u.shape, *v.shape)
                s = s - sL * sh * w.permute([order.index(k) for k in range(6)])
        return s, d

    def denominator(self, evl, task):
        T = self.T
        e = torch.tensor(evl, device=DEV)
        D = 0.0
        for k, b in enumerate(task):
            o = T.ofs[b - 1]
            x = e[o:o + T.rng[b - 1]] * (-1.0 if k < 3 else 1.0)
            D = D + x.view([-1 if q == k else 1 for q in range(6)])
        return D


def _exact_side(X, t1, t2):
    T = X.T
    O, V = list(T.O), list(T.V)
    return _Exact(T, t1, t2, _dense(T, X.v2, [O, V], [O, O], (0, 1, 2, 3), 0, 1),
                  _dense(T, X.v2, [V, V], [O, V], (0, 1, 2, 3), 1, 0),
                  _dense(T, X.v2, [V, V], [O, O], (0, 1, 2, 3), 1, 1))


def _too_long(c):
    """Whether the dense tensors or the tiles take more than a few seconds."""
    T = _Tiling(c)
    tuples = T.noab * T.nvab * (T.noab + T.nvab) ** 2
    tiles = sum(math.prod(T.r(*t)) for t in T.tasks())
    return tuples > 40000 or tiles * 36.0 * (T.no + T.nv) > 3e13 or c["nv"] ** 3 * c["no"] > 6e8


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "percall":
        calls, evl = _percall(c, seed)
        t3 = {"s": 0.0, "d": 0.0}
        letter = dict(zip(("h1", "h2", "h3", "p4", "p5", "p6", "x"), "ijkabcx"))
        for fam, n, _, a, b in calls:
            layout = (_HOLES[fam][n % 3] + " " + _PARTICLES[fam][n // 3]).split()
            sub = ["".join(letter[k] for k in reversed(q)) for q in
                   (*(op.split() for op in _OPERANDS[fam]), layout)]
            out = torch.einsum(f"{sub[0]},{sub[1]}->{sub[2]}", torch.tensor(a, device=DEV),
                               torch.tensor(b, device=DEV))
            t3[fam[0]] = t3[fam[0]] + _SIGN[fam][n] * out
        D = 0.0
        for k, e in zip((3, 4, 5, 0, 1, 2), evl):
            x = torch.tensor(e, device=DEV) * (1.0 if k > 2 else -1.0)
            D = D + x.view([-1 if q == k else 1 for q in range(6)])
        d = t3["d"]
        return {"energy": np.array([float((d * d / D).sum()),
                                    float((d * (d + t3["s"]) / D).sum())])}
    if c["kind"] == "batch":
        out = [exact(s, seed * 1000 + k) for k, s in enumerate(_batch_systems(c))]
        return {"energies": np.array([[e["e_bt"], e["e_pt"]] for e in out])}
    if _too_long(c):
        return None
    X = _Inputs(c, seed)
    T = X.T
    O, V = list(T.O), list(T.V)
    t1 = _dense(T, X.t1, [V], [O], (0, 1), 0, 0)
    t2 = _dense(T, X.t2, [V, V], [O, O], (0, 1, 2, 3), 1, 1)
    E = _exact_side(X, t1, t2)
    if c["kind"] == "tiles":
        s, d = E.tile(_task(T))
        return {"singles": s.reshape(-1).clone(), "doubles": d.reshape(-1).clone()}
    tasks = list(T.tasks())
    if c["kind"] in ("energy", "cold"):
        te = np.zeros((len(tasks), 2))
        for n, t in enumerate(tasks):
            s, d = E.tile(t)
            w = d * (T.factor(t) / E.denominator(X.evl, t))
            te[n] = float((w * d).sum()), float((w * (d + s)).sum())
        out = {"e_bt": float(te[:, 0].sum()), "e_pt": float(te[:, 1].sum())}
        return out if c["tiling"] == "orbital" else dict(out, tasks=te)
    if c["kind"] == "lambda":
        y1 = _dense(T, X.y1, [O], [V], (0, 1), 0, 0).T
        y2 = _dense(T, X.y2, [O, O], [V, V], (0, 1, 2, 3), 1, 1).permute(2, 3, 0, 1)
        F = _dense(T, X.f1, [O], [V], (0, 1), 0, 0)
        Y = _exact_side(X, y1, y2)
        te = np.zeros((len(tasks), 2))
        for n, t in enumerate(tasks):
            at = [T.at(b) for b in t]
            _, d = E.tile(t)
            ys, yd = Y.tile(t)
            for c_, sc in ((2, 1.0), (0, -1.0), (1, -1.0)):      # P(c/ab)
                for k, sk in ((5, 1.0), (3, -1.0), (4, -1.0)):   # P(k/ij)
                    q = [2 if x == c_ else x for x in (0, 1)]
                    r = [5 if x == k else x for x in (3, 4)]
                    w = torch.einsum("abij,kc->abcijk", y2[at[q[0]], at[q[1]], at[r[0]], at[r[1]]],
                                     F[at[k], at[c_]])
                    order = (*q, c_, *r, k)
                    yd = yd + sc * sk * w.permute([order.index(x) for x in range(6)])
            w = d * (T.factor(t) / E.denominator(X.evl, t))
            te[n] = float((w * yd).sum()), float((w * (yd + ys)).sum())
        return {"e1": float(te[:, 0].sum()), "e2": float(te[:, 1].sum()), "tasks": te}
    # CR-CCSD(T): the moment tile from the two intermediates, the denominator tile from t2 + t1 t1 / 3
    W = _dense(T, X.i1, [O, V], [O, O], (1, 0, 2, 3), 0, 1)
    I2 = _dense(T, X.i2, [V, V], [O, V], (0, 1, 2, 3), 1, 0)
    tt = torch.einsum("ai,bj->abij", t1, t1)
    M = _Exact(T, t1, t2, W, I2, t2 + (tt - tt.transpose(2, 3)) / 3.0)
    num1 = num2 = den1 = den2 = 0.0
    for t in tasks:
        ts, td = E.tile(t)
        q, m = M.tile(t)
        w = T.factor(t) / E.denominator(X.evl, t)
        num1 += float((w * m * td).sum())
        num2 += float((w * m * (td + ts)).sum())
        den1 += float((w * q * td).sum())
        den2 += float((w * q * (td + ts)).sum())
    den0 = float((t1 * t1).sum() + 0.25 * (t2 * t2).sum() + 0.5 * (tt * t2).sum())
    terms = {"num1": num1, "num2": num2, "den0": den0, "den1": den1, "den2": den2}
    return {"e1": num1 / (1.0 + den1 + den0), "e2": num2 / (1.0 + den2 + den0), "terms": terms}
