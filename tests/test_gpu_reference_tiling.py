"""Jobs whose kernel tasks are the reference tiles: items whose boxes have the
same place in equal tiles are contracted once (as in one-box tasks), the others
in full; several boxes to a tile, ragged last boxes, spin and irrep labels.

Tolerances as for the same sums elsewhere: (T) |dE| <= max(1e-10 Eh, 1e-12 |E|)
for the totals and every task's pair, Lambda 1e-11 |E| + 1e-15, CR 1e-10 |x| +
1e-15 against the oracle; FP32 and BF16X6 1e-6 |E|, BF16X3 3e-5 |E| against FP64.
"""
import os
import sys

import numpy as np
import pytest

import oracle
from nwchem_amd import TriplesJob, tiles as tl
from nwchem_amd.job import BF16X3, BF16X6, FP32, TILING_REFERENCE, cr_ccsd_t, lambda_ccsd_t

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import spin_systems  # noqa: E402

pytestmark = pytest.mark.gpu

# no, nv, occupied and virtual tile
TILINGS = [(8, 16, 8, 16),    # 2 x 2 x 2 hole and particle boxes, all full
           (7, 19, 7, 19),    # 4 + 3 holes, 8 + 8 + 3 particles (empty halves)
           (14, 27, 9, 12),   # two tiles of each, 4 + 4 + 1 holes
           (12, 20, 4, 10)]   # one hole box to a tile


@pytest.mark.parametrize("size", TILINGS, ids=["no%d_nv%d_o%d_v%d" % s for s in TILINGS])
def test_energies_of_reference_tiles(size, monkeypatch):
    monkeypatch.setenv("TCE_T_KERNEL", "wg16")
    no, nv, to, tv = size
    tm = tl.TileModel.synthetic(no, nv, to, tv, 61)
    b = tl.synth_blocks(tm, 61)
    ref = oracle.ccsd_t(oracle.Tiles(tm.range, tm.noab, tm.evl), b.t1, b.t1h, b.t2, b.t2h, b.v2, b.v2h)
    print(f"reference tiles no={no} nv={nv} ranges={list(map(int, tm.range))}", flush=True)
    with TriplesJob(tm, tiling=TILING_REFERENCE) as job:
        job.upload(b)
        got = job.run()
        te = job.task_energies()
        low = {m: job.run(m) for m in (FP32, BF16X3, BF16X6)}
    for x, y in zip(got, ref[:2]):
        assert abs(x - y) <= max(1e-10, 1e-12 * abs(y))
    assert (np.abs(te - ref[2]) <= np.maximum(1e-10, 1e-12 * np.abs(ref[2]))).all()
    for m, e in low.items():
        for x, y in zip(e, got):
            assert abs(x - y) <= (3e-5 if m == BF16X3 else 1e-6) * abs(y), (m, x, y)


PAIRS = [dict(sizes_o=[6], sizes_v=[11], seed=62),
         dict(sizes_o=[5, 2], sizes_v=[9, 3], irreps_o=[0, 1], irreps_v=[1, 0], seed=63),
         dict(sizes_o=[5], sizes_v=[9], seed=64, flip_symmetric=True, restricted=True)]


@pytest.mark.parametrize("prm", PAIRS, ids=["spins", "irreps", "restricted"])
def test_lambda_and_cr_of_reference_tiles(prm):
    s = spin_systems.SpinSystem(**prm)
    L, I, b = s.lambda_inputs(), s.cr_inputs(), s.blocks
    print(f"reference-tiled pairs {prm}", flush=True)
    t = TILING_REFERENCE
    with TriplesJob(s.tiles, tiling=t) as right, TriplesJob(s.tiles, tiling=t) as left, \
            TriplesJob(s.tiles, tiling=t) as cj:
        right.upload(b)
        e = right.run()
        left.upload_lambda(L["y1"], L["y1h"], L["y2"], L["y2h"], b.v2, b.v2h)
        e1, e2, te = lambda_ccsd_t(right, left, L["f1"], L["f1h"])
        cj.upload_cr(b.t1, b.t1h, b.t2, b.t2h, I["i1_1"], I["i1_1h"], I["i1_2"], I["i1_2h"])
        c1, c2, terms = cr_ccsd_t(right, cj)
    ref = oracle.ccsd_t(s.oracle_tiles(), b.t1, b.t1h, b.t2, b.t2h, b.v2, b.v2h)
    for x, y in zip(e, ref[:2]):
        assert abs(x - y) <= max(1e-10, 1e-12 * abs(y))
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
