"""Pairs of jobs used again: the spill slots that the right-hand job keeps from
one Lambda- or CR-CCSD(T) call serve the next, of another mode (another slot
layout and size), another kind of call and other data.

Every call must give what the same call gives on jobs that made no other: the
sums are formed in a fixed order, so bit for bit.
"""
import os
import sys

import numpy as np
import pytest

from nwchem_amd import TriplesJob
from nwchem_amd.job import BF16X3, BF16X6, FP32, FP64, cr_ccsd_t, lambda_ccsd_t

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import spin_systems  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPE = dict(sizes_o=[5], sizes_v=[9, 3])


class Data:
    """Inputs of one seed for the tiles of another."""

    def __init__(self, seed):
        s = spin_systems.SpinSystem(seed=seed, **SHAPE)
        self.tiles, self.b, self.L, self.I = s.tiles, s.blocks, s.lambda_inputs(), s.cr_inputs()

    def triples(self, job):
        job.upload(self.b)

    def left(self, job):
        L, b = self.L, self.b
        job.upload_lambda(L["y1"], L["y1h"], L["y2"], L["y2h"], b.v2, b.v2h)

    def cr(self, job):
        b, I = self.b, self.I
        job.upload_cr(b.t1, b.t1h, b.t2, b.t2h, I["i1_1"], I["i1_1h"], I["i1_2"], I["i1_2h"])

    def run_lambda(self, right, left, mode):
        e1, e2, te = lambda_ccsd_t(right, left, self.L["f1"], self.L["f1h"], precision=mode)
        return np.concatenate([[e1, e2], np.ravel(te)])

    def run_cr(self, triples, cr, mode):
        e1, e2, t = cr_ccsd_t(triples, cr, mode)
        return np.array([e1, e2, t["num1"], t["num2"], t["den0"], t["den1"], t["den2"]])


def fresh(tiles, d, kind, mode):
    with TriplesJob(tiles) as a, TriplesJob(tiles) as b:
        d.triples(a)
        if kind == "lambda":
            d.left(b)
            return d.run_lambda(a, b, mode)
        d.cr(b)
        return d.run_cr(a, b, mode)


@pytest.mark.parametrize("modes", [(FP64, BF16X6, FP64), (BF16X3, FP64, FP32, BF16X6)],
                         ids=["fp64_first", "bf16_first"])
def test_cr_then_lambda_on_one_right_hand_job(modes):
    one, two = Data(51), Data(52)
    tiles = one.tiles
    print(f"reuse modes={modes}", flush=True)
    with TriplesJob(tiles) as other, TriplesJob(tiles) as right:
        for d in (one, two):
            d.triples(other)
            d.cr(right)
            for m in modes:
                assert np.array_equal(d.run_cr(other, right, m), fresh(tiles, d, "cr", m)), m
        for d in (one, two):  # the same job, as a Lambda call's right-hand one
            d.triples(right)
            d.left(other)
            for m in modes:
                assert np.array_equal(d.run_lambda(right, other, m), fresh(tiles, d, "lambda", m)), m
        two.triples(other)
        two.cr(right)
        assert np.array_equal(two.run_cr(other, right, FP64), fresh(tiles, two, "cr", FP64))
