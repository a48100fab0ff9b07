"""The fused kernel's boxes where its work split changes: equal hole or
particle boxes (distinct elements only), boxes past a ragged edge, a particle
half without any element, and launches with fewer items than workgroups,
against the oracle.

Tolerances as for the same sums elsewhere: (T) |dE| <= max(1e-10 Eh, 1e-12 |E|)
for the totals and every task's pair, Lambda 1e-11 |E| + 1e-15, CR 1e-10 |x| +
1e-15.
"""
import os
import sys

import numpy as np
import pytest

import oracle
from nwchem_amd import TriplesJob, tiles as tl
from nwchem_amd.job import cr_ccsd_t, lambda_ccsd_t

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import spin_systems  # noqa: E402

pytestmark = pytest.mark.gpu

BOXES = [
    (1, 5),    # a single hole: no triple, all energies 0
    (3, 3),    # one box of three holes, one of three particles
    (4, 8),    # I == J == K, a == b == c, all full
    (8, 4),    # equal and different hole boxes, half a particle box
    (5, 12),   # 4 + 1 holes, 8 + 4 particles
    (9, 20),   # 4 + 4 + 1 holes, 8 + 8 + 4 particles
    (12, 17),  # a particle box of one
]


@pytest.mark.parametrize("size", BOXES, ids=[f"no{o}_nv{v}" for o, v in BOXES])
def test_energy_of_equal_and_ragged_boxes(size, monkeypatch):
    monkeypatch.setenv("TCE_T_KERNEL", "wg16")
    no, nv = size
    tm = tl.TileModel.synthetic(no, nv, no, nv, 77)
    b = tl.synth_blocks(tm, 77)
    ref = oracle.ccsd_t(oracle.Tiles(tm.range, tm.noab, tm.evl), b.t1, b.t1h, b.t2, b.t2h, b.v2, b.v2h)
    print(f"boxes no={no} nv={nv} ranges={list(tm.range)}", flush=True)
    with TriplesJob(tm) as job:
        job.upload(b)
        got = job.run()
        te = job.task_energies()
    for x, y in zip(got, ref[:2]):
        assert abs(x - y) <= max(1e-10, 1e-12 * abs(y))
    assert te.shape == ref[2].shape
    assert (np.abs(te - ref[2]) <= np.maximum(1e-10, 1e-12 * np.abs(ref[2]))).all()


PAIRS = [dict(sizes_o=[4], sizes_v=[8], seed=21), dict(sizes_o=[5], sizes_v=[9], seed=22),
         dict(sizes_o=[5, 1], sizes_v=[4, 9], irreps_o=[0, 1], irreps_v=[0, 1], seed=23)]


@pytest.mark.parametrize("prm", PAIRS, ids=["full", "ragged", "ragged_irreps"])
def test_lambda_and_cr_of_equal_and_ragged_boxes(prm):
    s = spin_systems.SpinSystem(**prm)
    L, I, b = s.lambda_inputs(), s.cr_inputs(), s.blocks
    print(f"pair boxes {prm}", flush=True)
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
