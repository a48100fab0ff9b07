"""Launches of FP64 and FP32 jobs in which most half items are empty (particle
tiles of at most 4 orbitals: the second half of every particle box has no
element), many to a workgroup and in a row.

Tolerances: energies |dE| <= max(1e-10 Eh, 1e-12 |E|) against the oracle, for
the totals and every task's pair; FP32 1e-6 |E| against FP64 as in the Lambda
and CR tests; Lambda 1e-11 |E| + 1e-15 and CR 1e-10 |x| + 1e-15 against the
oracle; tiles 1e-12 of the largest element.
"""
import os
import sys

import numpy as np
import pytest

import oracle
from nwchem_amd import TriplesJob, tiles as tl
from nwchem_amd.job import FP32, cr_ccsd_t, lambda_ccsd_t

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import spin_systems  # noqa: E402

pytestmark = pytest.mark.gpu

# no, nv, occupied and virtual tile: 1 to 4 particles a tile; 40 to 7 half items a workgroup
TILINGS = [(9, 40, 4, 4), (6, 33, 3, 3), (10, 31, 5, 2), (4, 20, 4, 1)]


@pytest.mark.parametrize("size", TILINGS, ids=["no%d_nv%d_o%d_v%d" % s for s in TILINGS])
def test_energy_with_every_second_half_empty(size, monkeypatch):
    monkeypatch.setenv("TCE_T_KERNEL", "wg16")
    no, nv, to, tv = size
    tm = tl.TileModel.synthetic(no, nv, to, tv, 88)
    b = tl.synth_blocks(tm, 88)
    ref = oracle.ccsd_t(oracle.Tiles(tm.range, tm.noab, tm.evl), b.t1, b.t1h, b.t2, b.t2h, b.v2, b.v2h)
    print(f"empty halves no={no} nv={nv} tiles {to}/{tv}", flush=True)
    with TriplesJob(tm) as job:
        job.upload(b)
        got = job.run()
        te = job.task_energies()
        low = job.run(FP32)
        t = max(tm.tasks(), key=lambda t: (len(set(t)), t))  # distinct tiles: no element vanishes
        p4, p5, p6, h1, h2, h3 = (int(x) for x in t)
        gs, gd = job.triples_tiles(h1, h2, h3, p4, p5, p6)
    for x, y in zip(got, ref[:2]):
        assert abs(x - y) <= max(1e-10, 1e-12 * abs(y))
    assert (np.abs(te - ref[2]) <= np.maximum(1e-10, 1e-12 * np.abs(ref[2]))).all()
    for x, y in zip(low, ref[:2]):
        assert abs(x - y) <= 1e-6 * abs(y)
    rs, rd = oracle.task_tiles(oracle.Tiles(tm.range, tm.noab, tm.evl), b.t1, b.t1h, b.t2, b.t2h,
                               b.v2, b.v2h, t)
    for g, r in ((gs, rs), (gd, rd)):
        dev, size = np.abs(g - r).max(), np.abs(r).max()
        assert dev <= 1e-12 * size


def test_lambda_and_cr_with_every_second_half_empty():
    s = spin_systems.SpinSystem(sizes_o=[4, 2], sizes_v=[4, 3, 4], seed=31)
    L, I, b = s.lambda_inputs(), s.cr_inputs(), s.blocks
    print("pairs with empty halves", flush=True)
    with TriplesJob(s.tiles) as right, TriplesJob(s.tiles) as left, TriplesJob(s.tiles) as cj:
        right.upload(b)
        left.upload_lambda(L["y1"], L["y1h"], L["y2"], L["y2h"], b.v2, b.v2h)
        e1, e2, te = lambda_ccsd_t(right, left, L["f1"], L["f1h"])
        cj.upload_cr(b.t1, b.t1h, b.t2, b.t2h, I["i1_1"], I["i1_1h"], I["i1_2"], I["i1_2h"])
        c1, c2, terms = cr_ccsd_t(right, cj)
    want = oracle.lambda_ccsd_t(s.oracle_tiles(), b.t1, b.t1h, b.t2, b.t2h, L["y1"], L["y1h"],
                                L["y2"], L["y2h"], b.v2, b.v2h, L["f1"], L["f1h"], 0)
    np.testing.assert_allclose([e1, e2], want[:2], rtol=1e-11, atol=1e-15)
    np.testing.assert_allclose(te, want[2], rtol=1e-11, atol=1e-15)
    o1, o2, ot = oracle.cr_ccsd_t(s.oracle_tiles(), b.t1, b.t1h, b.t2, b.t2h, b.v2, b.v2h,
                                  I["i1_1"], I["i1_1h"], I["i1_2"], I["i1_2h"])
    for k in ("num1", "num2", "den0", "den1", "den2"):
        assert abs(terms[k] - ot[k]) <= 1e-10 * abs(ot[k]) + 1e-15, (k, terms[k], ot[k])
    for x, y in ((c1, o1), (c2, o2)):
        assert abs(x - y) <= 1e-10 * abs(y) + 1e-15
