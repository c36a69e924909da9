"""The LW backward kernels at the sizes between which the call chooses them:
every column's gradients, and the forward fluxes of a one-pass call, are the
same bits whichever kernel computes them (the finite-difference and adjoint
tests cover their values), and a NaN column stays alone."""
import numpy as np
import pytest

from mima_amd.columns import make_columns, subset

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rr():
    from mima_amd import rrtmg
    rrtmg.rrtmg_lw_ini()
    yield rrtmg
    rrtmg.set_precision("fp64")


@pytest.fixture(scope="module")
def cols():
    c = make_columns(67, 61, 19, seed=12, lapse_range=(4.0, 9.0), rh_range=(0.05, 1.0))  # 4087 columns
    c["emis"][:] = np.random.default_rng(1).uniform(0.8, 1.0, c["emis"].shape)
    g = np.random.default_rng(2)
    n, L = c["ncol"], c["nlay"]
    return c, dict(uflx_bar=g.normal(size=(L + 1, n)), dflx_bar=g.normal(size=(L + 1, n)), hr_bar=g.normal(size=(L, n)))


def _run(rr, c, cot, pick, prec):
    import torch
    rr.set_precision(prec)
    d = rr.to_device(subset(c, pick))
    bar = {k: torch.from_numpy(np.ascontiguousarray(v[:, pick])).cuda() for k, v in cot.items()}
    return {k: v.cpu().numpy() for k, v in rr.lw_vjp_columns(d, forward=True, **bar).items()}


# largest call: FP32 with its tables in LDS, FP64 a wave per unit; below 2560 and
# 1536 columns four waves per unit, eight in the smallest FP32 calls
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_every_kernel_gives_a_column_the_same_bits(rr, cols, prec):
    c, cot = cols
    full = _run(rr, c, cot, np.arange(c["ncol"]), prec)
    for lo, hi in ((40, 41), (1, 22), (22, 87), (87, 1622), (1000, 2536), (1008, 3567), (3, 2563)):
        part = _run(rr, c, cot, np.arange(lo, hi), prec)
        for k in full:
            assert np.array_equal(part[k], full[k][..., lo:hi]), (prec, lo, hi, k)


@pytest.mark.parametrize("n", [65, 700, 3001])
def test_nan_column_stays_alone(rr, cols, n):
    c, cot = cols
    good = _run(rr, c, cot, np.arange(n), "mixed")
    bad = subset(c, np.arange(c["ncol"]))
    bad["tlay"][7, 44] = np.nan
    got = _run(rr, bad, cot, np.arange(n), "mixed")
    keep = np.arange(n) != 44
    assert np.isnan(got["tlay"][:, 44]).any()
    for k in good:
        assert np.array_equal(got[k][..., keep], good[k][..., keep]), k
