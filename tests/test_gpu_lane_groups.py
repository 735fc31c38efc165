"""The kernels with a walker on a group of lanes (all-coordinate moves; single-coordinate moves on the
reference streams) against the generic kernel, at the edges of their forms: the smallest and largest dimensions of each (lanes, slots), walker counts that leave a
ragged last wave or call for two, four or eight lanes, odd step counts (a step pair cut, generator
outputs left over), and launches that continue the streams.  Every number is bit-identical."""
import numpy as np
import pytest

from mcitest import (ESTIM_MJ, ESTIM_NOOP, KERNELS_GENERIC, OBS_EXP_X2, OBS_X2, OBS_X2_SUM, PDF_GAUSS_DIAG, PDF_GAUSS_ISO, RNG_MT,
                     RNG_PHILOX, chain_setup, dptr)

pytestmark = pytest.mark.gpu

# native streams: two lanes for 17,000 walkers (where one does not hold the walker, or the card is not
# full), four for few, eight beyond 71 coordinates
NATIVE = [(1, 33), (3, 70), (4, 70), (7, 70), (8, 16), (15, 64), (16, 5), (23, 70), (24, 70), (36, 70), (39, 70), (40, 70), (55, 70),
          (56, 70), (71, 33), (72, 33), (79, 9), (80, 9), (88, 20), (2, 17000), (9, 17000), (11, 17000), (16, 17000), (17, 17000),
          (18, 33000), (35, 17000), (40, 17000)]
REFERENCE = [(1, 1), (2, 21), (4, 70), (5, 70), (8, 33), (9, 70), (12, 16), (13, 70), (16, 70), (17, 70), (24, 21), (25, 21), (32, 33),
             (33, 21), (48, 21), (49, 21), (51, 21), (63, 21), (64, 33), (65, 5)]
SINGLE = [(1, 5), (2, 21), (4, 70), (8, 33), (16, 70), (32, 16), (64, 21), (128, 5)]  # 128: one lane a walker
ALL_OBS = [OBS_X2, OBS_X2_SUM, OBS_EXP_X2]


@pytest.mark.parametrize("rng,d,W", [(RNG_PHILOX, *c) for c in NATIVE] + [(RNG_MT, *c) for c in REFERENCE])
def test_walker_on_a_group_of_lanes(rng, d, W):
    obs = [[OBS_X2], [OBS_X2_SUM], ALL_OBS, [OBS_X2, OBS_X2_SUM], [OBS_EXP_X2], [OBS_X2, OBS_EXP_X2]][d % 6]
    check(rng, d, W, 0, (3, 1, 0)[d % 3], obs)


@pytest.mark.parametrize("obs", [[OBS_X2], ALL_OBS], ids=["x2", "all"])
@pytest.mark.parametrize("blocksize", [0, 1, 3])
@pytest.mark.parametrize("d,W", SINGLE)
def test_single_coordinate_moves_on_a_group_of_lanes(d, W, blocksize, obs):
    check(RNG_MT, d, W, 1, blocksize, obs)


def check(rng, d, W, veclen, blocksize, obs):
    print("lane groups", rng, d, W, veclen, blocksize, obs, flush=True)
    est = ESTIM_NOOP if blocksize == 0 else ESTIM_MJ
    sig = np.random.default_rng(d).uniform(0.5, 2.0, d)
    pdf = (PDF_GAUSS_ISO, []) if d % 4 == 1 and veclen == 0 else (PDF_GAUSS_DIAG, 0.5 / sig ** 2)
    cfg = dict(ndim=d, seed=77 + d, ndecorr=37, move=(0, veclen, 1, None), pdfs=[pdf],
               obs=[(k, [], blocksize, 1, 0, est) for k in obs])
    n1 = 64 * max(blocksize, 1) if blocksize else 151
    out = {}
    for path in ("groups", "generic"):
        c = chain_setup("mci", cfg, nwalkers=W)
        c.setRng(rng)
        c.setCoupling(1)
        if path == "generic":
            c.setKernelPath(KERNELS_GENERIC)
        first = c.integrate(n1)
        data = [c.observableData(i, d if k == OBS_X2 else 1) for i, k in enumerate(obs)]
        second = c.integrate(16 * max(blocksize, 1), False, True)
        out[path] = (*first, *second, c.getX(), c.getWalkerSteps(), *c.walkerAcceptance(), *c.walkerResults(), *data)
    for k, (f, g) in enumerate(zip(out["groups"], out["generic"])):
        assert np.array_equal(f, g), k


# (outputs a step, coordinates, moves) and run lengths that end just before, at and after a part (52 outputs), a
# round (312) and two: the outputs left over go back to the state through element 0 and beyond
ENDS = [(3, 16, 1, (17, 18, 34, 35, 103, 104, 105, 208, 209)), (4, 3, 0, (12, 13, 14, 77, 78, 79, 156)),
        (13, 12, 0, (3, 4, 5, 23, 24, 25, 48)), (52, 51, 0, (1, 2, 5, 6, 7)), (65, 64, 0, (1, 2, 4, 5, 24, 25))]


@pytest.mark.parametrize("per,d,veclen,runs", ENDS)
def test_runs_that_end_at_the_edges_of_the_generator_parts(per, d, veclen, runs):
    """each run continues the streams of the one before, so a state put back wrongly shows in the next"""
    cfg = dict(ndim=d, seed=9 + d, ndecorr=0, nfind=0, move=(0, veclen, 1, None),
               pdfs=[(PDF_GAUSS_DIAG, 0.5 / np.random.default_rng(d).uniform(0.5, 2.0, d) ** 2)], obs=[(OBS_X2, [], 0, 1, 0, ESTIM_NOOP)])
    out = {}
    for path in ("groups", "generic"):
        c = chain_setup("mci", cfg, nwalkers=21)
        c.setRng(RNG_MT)
        c.setCoupling(1)
        c.setMRT2Step(0.7)
        if path == "generic":
            c.setKernelPath(KERNELS_GENERIC)
        out[path] = []
        for n in runs:
            print("generator parts", per, d, path, n, flush=True)
            out[path] += [*c.integrate(n, False, False), c.getX(), *c.walkerAcceptance()]
    for k, (f, g) in enumerate(zip(out["groups"], out["generic"])):
        assert np.array_equal(f, g), k


@pytest.mark.parametrize("d,W,ndecorr", [(16, 32769, 37), (16, 32769, 600), (64, 16385, 37), (32, 32768, 37), (64, 32800, 37)])
def test_launches_without_sums_on_either_form(d, W, ndecorr):
    """calibration and decorrelation of single-coordinate moves run on one lane or on four by their length and the
    walkers' number; each hands the generators on to the next, whichever it is, and an independent calibration leaves
    them at different places"""
    for coupling in (1, 0):
        print("without sums", d, W, ndecorr, coupling, flush=True)
        cfg = dict(ndim=d, seed=4, ndecorr=ndecorr, nfind=2 if coupling else -3, move=(0, 1, 1, None),
                   pdfs=[(PDF_GAUSS_DIAG, 0.5 / np.random.default_rng(d).uniform(0.5, 2.0, d) ** 2)], obs=[(OBS_X2, [], 8, 1, 0, ESTIM_MJ)])
        out = []
        for generic in (False, True):
            c = chain_setup("mci", cfg, nwalkers=W)
            c.setRng(RNG_MT)
            c.setCoupling(coupling)
            if generic:
                c.setKernelPath(KERNELS_GENERIC)
            first = c.integrate(16)
            out.append((*first, *c.integrate(16), c.getX(), c.getWalkerSteps(), *c.walkerAcceptance()))
        for k, (f, g) in enumerate(zip(*out)):
            assert np.array_equal(f, g), (coupling, k)


def test_launches_without_sums_do_not_pay_for_the_dimensions():
    """a decorrelation of 200 steps moves one coordinate a step and sums nothing: 64 dimensions take at most 1.7 times
    what two take (1.04 measured; 2.8 when every step selected among a lane's sixteen coordinates)"""
    took = []
    for d in (2, 64):
        c = chain_setup("mci", dict(ndim=d, seed=4, ndecorr=200, move=(0, 1, 1, None), pdfs=[(PDF_GAUSS_DIAG, np.full(d, 0.5))],
                                    obs=[(OBS_X2, [], 0, 1, 0, ESTIM_NOOP)]), nwalkers=65536)
        c.setRng(RNG_MT)
        c.setCoupling(1)
        best = np.inf
        for _ in range(5):
            print("decorrelation", d, flush=True)
            c.integrate(0, False, True)
            t = np.zeros(5)
            c.call("get_timings", dptr(t), 5)
            best = min(best, t[1])
        took.append(best)
    assert took[1] < 1.7 * took[0], took


def phase(c, i, calls):
    """the shortest of some calls' phases (milliseconds)"""
    best = np.inf
    for _ in range(calls):
        c.integrate(256)
        t = np.zeros(5)
        c.call("get_timings", dptr(t), 5)
        best = min(best, t[i])
    return best


def test_a_lane_of_eighteen_slots_keeps_them_in_registers():
    """three observables of a walker in sixty dimensions cost their sums, at most twice one observable's launch (1.1
    times is measured; eleven times with the walker's arrays in scratch memory)"""
    took = []
    for obs in ([OBS_X2], ALL_OBS):
        print("slots", obs, flush=True)
        c = chain_setup("mci", dict(ndim=60, seed=4, ndecorr=20, move=(0, 0, 1, None), pdfs=[(PDF_GAUSS_DIAG, np.full(60, 0.5))],
                                    obs=[(k, [], 1, 1, 0, ESTIM_MJ) for k in obs]), nwalkers=16384)
        c.setRng(RNG_PHILOX)
        c.setCoupling(1)
        took.append(phase(c, 2, 4))
    print("took", took, flush=True)
    assert took[1] < 2 * took[0], took


def test_traces_of_more_walkers_than_lanes_keep_two_waves_a_simd():
    """the sums that MJBlocker's mean would take are not kept where their registers would cost a wave: four waves a
    SIMD sample in less than 3.2 times one wave's time (2.1 measured; 3.9 with the sums)"""
    took = []
    for W in (65536, 262144):
        print("traces", W, flush=True)
        c = chain_setup("mci", dict(ndim=1, seed=4, ndecorr=20, move=(0, 0, 1, None), pdfs=[(PDF_GAUSS_DIAG, np.full(1, 0.5))],
                                    obs=[(OBS_X2, [], 1, 1, 0, ESTIM_MJ)]), nwalkers=W)
        c.setRng(RNG_PHILOX)
        c.setCoupling(1)
        took.append(phase(c, 2, 5))
    print("took", took, flush=True)
    assert took[1] < 3.2 * took[0], took


@pytest.mark.parametrize("d,W,block,obs,n", [
    (16, 16400, 1, [OBS_X2], 64), (16, 16400, 1, [OBS_X2], 128), (64, 16400, 8, ALL_OBS, 64), (64, 16400, 8, [OBS_X2_SUM], 128),
    (8, 32800, 8, [OBS_X2_SUM], 512), (16, 32800, 8, [OBS_X2_SUM], 512), (4, 32800, 1, [OBS_EXP_X2], 512)])
def test_launches_with_sums_on_either_form(d, W, block, obs, n):
    """... and so do the launches with observables, by what they sum and for how long"""
    print("with sums", d, W, block, obs, n, flush=True)
    cfg = dict(ndim=d, seed=4, ndecorr=7, nfind=1, move=(0, 1, 1, None), pdfs=[(PDF_GAUSS_DIAG, 0.5 / np.random.default_rng(d).uniform(0.5, 2.0, d) ** 2)],
               obs=[(k, [], block, 1, 0, ESTIM_MJ) for k in obs])
    out = []
    for generic in (False, True):
        c = chain_setup("mci", cfg, nwalkers=W)
        c.setRng(RNG_MT)
        c.setCoupling(1)
        if generic:
            c.setKernelPath(KERNELS_GENERIC)
        first = c.integrate(n)
        out.append((*first, *c.integrate(16 * block, False, False), c.getX(), *c.walkerAcceptance(), *c.walkerResults()))
    for k, (f, g) in enumerate(zip(*out)):
        assert np.array_equal(f, g), k


def test_sums_of_many_walkers_do_not_pay_for_the_dimensions():
    """|x|^2 alone, blocks of 16: 64 dimensions take at most 2.5 times what one takes (1.8 measured; 3.9 on groups of
    lanes, whose sum is over every coordinate, in order, each step)"""
    took = []
    for d in (1, 64):
        print("sums", d, flush=True)
        c = chain_setup("mci", dict(ndim=d, seed=4, ndecorr=20, move=(0, 1, 1, None), pdfs=[(PDF_GAUSS_DIAG, np.full(d, 0.5))],
                                    obs=[(OBS_X2_SUM, [], 16, 1, 0, ESTIM_MJ)]), nwalkers=65536)
        c.setRng(RNG_MT)
        c.setCoupling(1)
        took.append(phase(c, 2, 5))
    print("took", took, flush=True)
    assert took[1] < 2.5 * took[0], took
