"""The forward kernels of both sides at the sizes between which the call chooses them:
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
    rrtmg.rrtmg_sw_ini()
    yield rrtmg
    rrtmg.set_precision("fp64")


@pytest.fixture(scope="module")
def cols():
    # 11449 columns: eleven tiles of 1008 and a rest; moist to dry, so that every
    # branch of the species parameter occurs; a reflecting surface; every sun
    # angle, half of the columns night
    c = make_columns(107, 107, 23, seed=11, lapse_range=(4.0, 9.0), rh_range=(0.05, 1.0))
    for k, v in GASES.items():
        c[k][:] = v
    c["emis"][:] = np.random.default_rng(1).uniform(0.8, 1.0, c["emis"].shape)
    return c


def _run(rr, c, prec):
    rr.set_precision(prec)
    d = rr.to_device(c)
    return {k: v.cpu().numpy() for k, v in dict(rr.lw_columns(d), **rr.sw_columns(d)).items()}


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_every_kernel_gives_a_column_the_same_bits(rr, cols, prec):
    full = _run(rr, cols, prec)          # the largest calls' kernel
    for lo, hi in ((40, 41), (1, 22), (22, 87), (87, 400), (400, 3000), (945, 7041), (1000, 10000)):
        part = _run(rr, subset(cols, np.arange(lo, hi)), prec)
        for k in full:
            assert np.array_equal(part[k], full[k][:, lo:hi]), (prec, lo, hi, k)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_edges_against_oracle(rr, cols, prec):
    full = _run(rr, cols, prec)
    pick = np.r_[0:70, 1000:1030, 2010:2020, 5660:5700, 11430:11449]
    c = subset(cols, pick)
    want = dict(po.rrtmg_lw(c), **po.rrtmg_sw(c))
    for k in ("uflx", "dflx", "hr", "swuflx", "swdflx", "swhr"):
        assert np.max(np.abs(full[k][:, pick] - want[k])) < ATOL[prec], k


def test_not_a_number_stays_in_its_column(rr, cols):
    c = subset(cols, np.arange(5600, 5800))
    c["coszen"][77] = 0.4
    clean = _run(rr, c, "mixed")
    c["h2ovmr"][5, 77] = np.nan
    got = _run(rr, c, "mixed")
    keep = np.arange(200) != 77
    for k in got:
        assert np.array_equal(got[k][:, keep], clean[k][:, keep]), k
    assert np.isnan(got["uflx"][:, 77]).any() and np.isnan(got["swuflx"][:, 77]).any()


def test_night_and_one_day_column(rr, cols):
    c = subset(cols, np.arange(0, 300))
    c["coszen"][:] = 0.0
    assert all(not np.any(v) for k, v in _run(rr, c, "mixed").items() if k.startswith("sw"))
    c["coszen"][[7, 299]] = (1e-9, 0.5)   # one g-point's beam all but horizontal
    got, want = _run(rr, c, "fp64"), po.rrtmg_sw(c)
    for k in ("swuflx", "swdflx", "swhr"):
        assert np.max(np.abs(got[k] - want[k])) < 1e-8, k
