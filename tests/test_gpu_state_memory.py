"""The generic step kernels with the walkers' state in LDS (up to 80 KiB a wave: 6 d rows of 512 bytes here while
sampling, 4 d while calibrating) and in HBM, for the catalogue and for device functors, against the specialised
kernel: bit for bit the same at the last width in LDS, the first in HBM, where only calibration stays in LDS, and
beyond."""
import numpy as np
import pytest

import device_functors as DF
from mcitest import COUPLING_INDEPENDENT, ESTIM_MJ, ESTIM_NOOP, KERNELS_GENERIC, OBS_X2, PDF_GAUSS_DIAG, RNG_MT, Chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [26, 27, 35, 60])
def test_state_in_lds_and_in_hbm(d):
    print("state memory", d, flush=True)
    a = 0.5 / np.random.default_rng(d).uniform(0.5, 2.0, d) ** 2
    out = []
    for name in ("specialised", "catalogue", "device"):
        c = Chain("mci", d, 70)
        c.setSeed(99)
        c.setRng(RNG_MT)
        c.setCoupling(COUPLING_INDEPENDENT)
        c.setNdecorrelationSteps(20)
        if name != "specialised":
            c.setKernelPath(KERNELS_GENERIC)
        if name == "device":
            c.addSamplingFunctionDevice("diag", DF.DIAG, d, a)
            c.addObservableDevice("xsq", DF.X2, d, (), 4, 1, True, ESTIM_MJ)
        else:
            c.addSamplingFunction(PDF_GAUSS_DIAG, a)
            c.addObservable(OBS_X2, (), 4, 1, True, ESTIM_MJ)
        first = c.integrate(4 * 32)
        out.append((*first, *c.integrate(4 * 16, False, False), c.getX(), c.getWalkerSteps(), *c.walkerAcceptance(), *c.walkerResults()))
    for other in out[1:]:
        for k, (f, g) in enumerate(zip(out[0], other)):
            assert np.array_equal(f, g), k


def test_a_run_too_large_for_the_card_is_an_error_once():
    """traces of 348 GB are refused, and the calls after that are not"""
    d, W = 16, 1024
    c = Chain("mci", d, W)
    c.setSeed(99)
    c.setRng(RNG_MT)
    c.setNdecorrelationSteps(20)
    c.addSamplingFunction(PDF_GAUSS_DIAG, np.full(d, 0.5))
    c.addObservable(OBS_X2, (), 1, 1, False, ESTIM_NOOP)
    print("traces of 348 GB", flush=True)
    with pytest.raises(RuntimeError):
        c.integrate(2_660_000, False, False)
    print("and of a few steps", flush=True)
    avg, _ = c.integrate(8, False, False)
    assert np.all(np.isfinite(avg))


@pytest.mark.parametrize("d,W", [(28, 65536), (28, 65537)])
def test_many_walkers_in_hbm(d, W):
    """a state in HBM with up to one wave a SIMD and with more, against the specialised kernel: bit for bit"""
    print("state in HBM", d, W, flush=True)
    out = []
    for generic in (False, True):
        c = Chain("mci", d, W)
        c.setSeed(98)
        c.setRng(RNG_MT)
        c.setCoupling(COUPLING_INDEPENDENT)
        c.setNfindMRT2Iterations(1)
        c.setNdecorrelationSteps(5)
        if generic:
            c.setKernelPath(KERNELS_GENERIC)
        c.addSamplingFunction(PDF_GAUSS_DIAG, np.full(d, 0.5))
        c.addObservable(OBS_X2, (), 4, 1, True, ESTIM_MJ)
        out.append((*c.integrate(4 * 4), c.getX(), *c.walkerAcceptance()))
    for k, (f, g) in enumerate(zip(*out)):
        assert np.array_equal(f, g), k
