"""The LW forward's kernels at the sizes between which the call chooses them:
every column's result is the same bits whichever kernel computes it, and
agrees with the oracle at the edges of units, tiles and of the choice."""
import numpy as np
import pytest

import pyoracle as po
from mima_amd.columns import make_columns, subset

pytestmark = pytest.mark.gpu

GASES = {"ch4vmr": 1.9e-6, "n2ovmr": 3.3e-7, "o2vmr": 0.209, "cfc11vmr": 2.2e-10, "cfc12vmr": 5e-10,
         "cfc22vmr": 2.5e-10, "ccl4vmr": 8e-11}
# FP64: the oracle's own sums in another order; mixed: the path's bound
ATOL = {"fp64": 1e-8, "mixed": 0.05}


@pytest.fixture(scope="module")
def rr():
    from mima_amd import rrtmg
    rrtmg.rrtmg_lw_ini()
    yield rrtmg
    rrtmg.set_precision("fp64")


@pytest.fixture(scope="module")
def cols():
    # 5041 columns: five tiles of 1008 and one column; moist to dry, so that
    # every branch of the species parameter occurs; a reflecting surface
    c = make_columns(71, 71, 23, seed=11, lapse_range=(4.0, 9.0), rh_range=(0.05, 1.0))
    for k, v in GASES.items():
        c[k][:] = v
    c["emis"][:] = np.random.default_rng(1).uniform(0.8, 1.0, c["emis"].shape)
    return c


def _lw(rr, c, prec):
    rr.set_precision(prec)
    return {k: v.cpu().numpy() for k, v in rr.lw_columns(rr.to_device(c)).items()}


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_every_kernel_gives_a_column_the_same_bits(rr, cols, prec):
    full = _lw(rr, cols, prec)          # the largest calls' kernel
    for lo, hi in ((0, 1), (1, 22), (22, 87), (87, 400), (400, 3000), (945, 5041)):
        part = _lw(rr, subset(cols, np.arange(lo, hi)), prec)
        for k in full:
            assert np.array_equal(part[k], full[k][:, lo:hi]), (prec, lo, hi, k)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_edges_against_oracle(rr, cols, prec):
    full = _lw(rr, cols, prec)
    pick = np.r_[0:70, 1000:1030, 2010:2020, 5030:5041]
    want = po.rrtmg_lw(subset(cols, pick))
    for k in ("uflx", "dflx", "hr"):
        assert np.max(np.abs(full[k][:, pick] - want[k])) < ATOL[prec], k


def test_not_a_number_stays_in_its_column(rr, cols):
    c = subset(cols, np.arange(0, 200))
    clean = _lw(rr, c, "mixed")
    c["h2ovmr"][5, 77] = np.nan
    got = _lw(rr, c, "mixed")
    keep = np.arange(200) != 77
    for k in got:
        assert np.array_equal(got[k][:, keep], clean[k][:, keep]), k
    assert np.isnan(got["uflx"][:, 77]).any()
