"""The per-call surface at the sizes where its kernels split the work another
way, against numpy.

Energy (compute_en_): hole blocks of 1 to 129 and of 2049 elements (as many
particle triples to a unit of work as 256 threads hold, two halves, one triple,
two LDS chunks), particle counts that fill no unit or leave a remainder.
Tolerance: max(1e-10, 1e-12 |E|), as for every FP64 energy.

Contractions (sd_t_*): each of the 27 calls at extents on both sides of the
rule that takes it to register tiles or to one element a thread: small, ragged
against the 4 x 4 tiles, a hole block of one element (not packed) and a particle
index longer than a grid's second dimension.
Tolerance: K products summed in any order, (K + 2) 2^-53 sum |a b| + 2^-52 |t3|
for every element.
"""
import ctypes as C

import numpy as np
import pytest

from nwchem_amd import _lib

pytestmark = pytest.mark.gpu

DP = C.POINTER(C.c_double)


def ptr(a):
    return a.ctypes.data_as(DP)


def refs(xs):
    return [C.byref(C.c_long(x)) for x in xs]


# h1 h2 h3 p4 p5 p6
ENERGY = [(1, 1, 1, 1, 1, 1), (1, 1, 1, 5, 7, 9), (1, 1, 1, 64, 17, 31), (1, 2, 1, 3, 3, 3),
          (3, 3, 3, 4, 5, 11), (4, 4, 8, 3, 5, 7), (3, 43, 1, 5, 2, 9), (5, 5, 5, 9, 8, 7),
          (3, 683, 1, 2, 3, 4)]


@pytest.mark.parametrize("dims", ENERGY, ids=["x".join(map(str, d)) for d in ENERGY])
def test_energy_of_small_hole_blocks(dims):
    L = _lib.lib()
    h1, h2, h3, p4, p5, p6 = dims
    r = np.random.default_rng(7)
    t1, vs = r.standard_normal((h1, p4)) * 0.1, r.standard_normal((p5, p6, h2, h3))
    t2, vd = r.standard_normal((h2, h1, p4, 3)) * 0.1, r.standard_normal((p5, p6, h3, 3))
    ev = [r.uniform(-2.0, -0.3, n) for n in dims[:3]] + [r.uniform(0.2, 4.0, n) for n in dims[3:]]
    print(f"percall energy {dims}", flush=True)
    d, dummy, e = refs(dims), np.zeros(1), np.zeros(2)
    L.dev_mem_d_(*d)
    L.dev_mem_s_(*d)
    L.sd_t_s1_1_cuda_(*d, ptr(dummy), ptr(t1), ptr(vs))
    L.sd_t_d2_1_cuda_(*d, C.byref(C.c_long(3)), ptr(dummy), ptr(t2), ptr(vd))
    L.compute_en_(C.byref(C.c_double(0.5)), ptr(e), *[ptr(x) for x in ev], *d, None, None)
    L.dev_release_()
    assert L.tce_t_legacy_status() == 0, L.tce_t_last_error()
    s = np.einsum("ia,bcjk->abcijk", t1, vs)
    t = -np.einsum("jiae,bcke->abcijk", t2, vd)
    D = 0.0
    for k, x in enumerate(ev):
        D = D + x.reshape([-1 if (k - 3) % 6 == n else 1 for n in range(6)]) * (1 if k < 3 else -1)
    w = 0.5 * t / D
    for got, want in zip(e, ((w * t).sum(), (w * (t + s)).sum())):
        assert abs(got - want) <= max(1e-10, 1e-12 * abs(want)), (got, want)


# layouts (fastest first) and signs of the 27 calls, ccsd_t_kernels_omp.F:5-1198; operands, fastest first
HOLES = {"s1": ("h3 h2 h1", "h3 h1 h2", "h1 h3 h2"), "d1": ("h3 h2 h1", "h3 h1 h2", "h1 h3 h2"),
         "d2": ("h3 h2 h1", "h2 h1 h3", "h2 h3 h1")}
PARTICLES = {"s1": ("p6 p5 p4", "p6 p4 p5", "p4 p6 p5"), "d1": ("p6 p5 p4", "p5 p4 p6", "p5 p6 p4"),
             "d2": ("p6 p5 p4", "p6 p4 p5", "p4 p6 p5")}
SIGN = {"s1": (1, -1, 1, -1, 1, -1, 1, -1, 1), "d1": (-1, 1, -1, -1, 1, -1, 1, -1, 1),
        "d2": (-1, -1, 1, 1, 1, -1, -1, -1, 1)}
OPERANDS = {"s1": ("p4 h1", "h3 h2 p6 p5"), "d1": ("x p4 p5 h1", "h3 h2 p6 x"),
            "d2": ("x p4 h1 h2", "x h3 p6 p5")}
LETTER = {"h1": "i", "h2": "j", "h3": "k", "p4": "a", "p5": "b", "p6": "c", "x": "x"}

# h1 h2 h3 p4 p5 p6, contraction
SIZES = [((3, 2, 4, 5, 3, 6), 3), ((5, 6, 7, 9, 10, 11), 4), ((5, 6, 7, 9, 10, 13), 24),
         ((7, 8, 9, 10, 13, 17), 4), ((1, 1, 1, 37, 41, 43), 70),
         ((1, 1, 1, 70000, 1, 1), 64), ((1, 1, 1, 1, 70000, 1), 64), ((1, 1, 1, 1, 1, 70000), 64)]


@pytest.mark.parametrize("fam", ["s1", "d1", "d2"])
@pytest.mark.parametrize("size", SIZES, ids=["x".join(map(str, d)) + f"_k{k}" for d, k in SIZES])
def test_contractions_at_the_rules_edges(size, fam):
    L = _lib.lib()
    dims, K = size
    ext = dict(zip(("h1", "h2", "h3", "p4", "p5", "p6"), dims), x=K)
    r = np.random.default_rng(11)
    names = "h3 h2 h1 p6 p5 p4" + ("" if fam == "s1" else " x")
    ops = [[k for k in op.split()] for op in OPERANDS[fam]]
    a, b = (r.standard_normal([ext[k] for k in reversed(op)]) for op in ops)
    sub = ["".join(LETTER[k] for k in reversed(op)) for op in ops]
    print(f"percall {fam} {dims} K={K}", flush=True)
    for n in range(9):
        layout = (HOLES[fam][n % 3] + " " + PARTICLES[fam][n // 3]).split()
        out = "".join(LETTER[k] for k in reversed(layout))
        t3 = r.standard_normal([ext[k] for k in reversed(layout)])
        eq = f"{sub[0]},{sub[1]}->{out}"
        want = t3 + SIGN[fam][n] * np.einsum(eq, a, b)
        bound = (max(K, 1) + 2) * 2.0 ** -53 * np.einsum(eq, np.abs(a), np.abs(b)) + 2.0 ** -52 * np.abs(t3)
        t3 = np.ascontiguousarray(t3)
        getattr(L, f"sd_t_{fam}_{n + 1}_")(*refs([ext[k] for k in names.split()]), ptr(t3), ptr(a), ptr(b))
        assert L.tce_t_legacy_status() == 0, L.tce_t_last_error()
        assert (np.abs(t3 - want) <= bound).all(), (n + 1, np.abs(t3 - want).max())
