"""The per-call surface at the sizes where its kernels split the work another
way, against numpy.

Energy (compute_en_): hole blocks of 1 to 129 and of 2049 elements (as many
particle triples to a unit of work as 256 threads hold, two halves, one triple,
two LDS chunks), particle counts that fill no unit or leave a remainder.
Tolerance: max(1e-10, 1e-12 |E|), as for every FP64 energy.
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
