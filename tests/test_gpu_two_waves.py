"""The single-coordinate native chain with a producer and a chain wave per 64 walkers (up to 16,384 walkers)
against the generic kernel: decisions, positions, counters and
step sizes bit for bit, block means (dwell-time sums) to rounding.  Blocks that cut the ring's eight and the
straight runs of four and two, runs that end inside them, ragged walker counts,
both sides of the rule, odd counters, and launches that continue the streams."""
import numpy as np
import pytest

from mcitest import (COUPLING_INDEPENDENT, ESTIM_NOOP, ESTIM_UNCORR, KERNELS_GENERIC, OBS_EXP_X2, OBS_X2, OBS_X2_SUM, PDF_GAUSS_DIAG, RNG_PHILOX, chain_setup, dptr)

pytestmark = pytest.mark.gpu
SETS = [[OBS_X2], [OBS_X2_SUM], [OBS_X2, OBS_X2_SUM], [OBS_EXP_X2], [OBS_X2, OBS_X2_SUM, OBS_EXP_X2]]


@pytest.mark.parametrize("d,W,block", [
    (1, 1, 1), (2, 63, 8), (3, 64, 13), (5, 65, 20), (8, 130, 3), (16, 70, 160), (17, 33, 5), (64, 21, 9), (6, 100, 0),
    (16, 16384, 12), (4, 300, 256), (8, 129, 259), (2, 65, 12), (7, 16385, 24), (5, 9999, 10), (128, 70, 4), (143, 70, 4), (144, 70, 4)])
def test_two_waves_run_the_generic_chain(d, W, block):
    obs = SETS[(d + W) % 5]
    print("two waves", d, W, block, obs, flush=True)
    sig = np.random.default_rng(d).uniform(0.5, 2.0, d)
    cfg = dict(ndim=d, seed=31 + d, ndecorr=37, move=(0, 1, 1, None), pdfs=[(PDF_GAUSS_DIAG, 0.5 / sig ** 2)],
               obs=[(k, [], block, 1, 0, ESTIM_UNCORR if block else ESTIM_NOOP) for k in obs])
    n1, n2 = (5 * block, 3 * block) if block else (151, 42)
    out = {}
    for path in ("waves", "generic"):
        c = chain_setup("mci", cfg, nwalkers=W)
        c.setRng(RNG_PHILOX)
        c.setCoupling(1 if W < 1000 else 0)
        if path == "generic":
            c.setKernelPath(KERNELS_GENERIC)
        c.integrate(n1)
        exact = [c.getX(), c.getWalkerSteps(), *c.walkerAcceptance()]
        data = [c.observableData(i, d if k == OBS_X2 else 1) for i, k in enumerate(obs)]
        c.integrate(n2, False, True)
        exact += [c.getX(), *c.walkerAcceptance()]
        data += [c.walkerResults()[0]]
        out[path] = exact, data
    for k, (f, g) in enumerate(zip(out["waves"][0], out["generic"][0])):
        assert np.array_equal(f, g), k
    # a block mean is a sum of at most B + (accepted moves) <= 2 B positive and negative terms no larger than
    # its coordinate's largest x^2 in the block: 2^-53 times their number times that, far below 1e-12 here
    for f, g in zip(out["waves"][1], out["generic"][1]):
        assert np.allclose(f, g, rtol=1e-10, atol=1e-12)


def test_groups_without_a_walker_left_end_at_once():
    """Independent calibration enqueues as many iterations as the last one took; those after the last walker has
    left its loop hold no walker and take no steps.  64 iterations from a step far too small (doubled about 50
    times, then five more), then from the step that they found (five to a dozen hold a walker): the rest of an
    idle iteration (its compaction and bookkeeping) is about a tenth of one with walkers, so the whole is below
    half; with idle iterations that run, the two take the same time."""
    d, W = 128, 70
    cfg = dict(ndim=d, seed=5, ndecorr=0, nfind=-64, move=(0, 1, 1, None), pdfs=[(PDF_GAUSS_DIAG, np.full(d, 0.5))],
               obs=[(OBS_X2, [], 0, 1, 0, ESTIM_NOOP)])
    c = chain_setup("mci", cfg, nwalkers=W)
    c.setRng(RNG_PHILOX)
    c.setCoupling(COUPLING_INDEPENDENT)
    took = []
    for small in (True, True, False):  # the first loads the kernels and finds the number of iterations
        print("calibration from", "a small step" if small else "the step found", flush=True)
        if small:
            c.setMRT2Step(1e-15)
        c.integrate(0, True, False)
        t = np.zeros(5)
        c.call("get_timings", dptr(t), 5)
        took.append(t[0])
    assert took[2] < 0.5 * took[1], took


def test_short_blocks_cost_their_sums():
    """Ending a block reads the d coordinates without waiting for each: 1,024 blocks of four steps at d = 100 take
    at most five times what 64 blocks of 64 take (3.1 are measured; 7.0 with one read at a time)."""
    d, took = 100, []
    for block in (4, 64):
        cfg = dict(ndim=d, seed=5, ndecorr=100, move=(0, 1, 1, None), pdfs=[(PDF_GAUSS_DIAG, np.full(d, 0.5))],
                   obs=[(OBS_X2_SUM, [], block, 1, 0, ESTIM_UNCORR)])
        c = chain_setup("mci", cfg, nwalkers=4000)
        c.setRng(RNG_PHILOX)
        c.setCoupling(1)
        best = np.inf
        for _ in range(4):
            print("blocks of", block, flush=True)
            c.integrate(4096)
            t = np.zeros(5)
            c.call("get_timings", dptr(t), 5)
            best = min(best, t[2])
        took.append(best)
    assert took[0] < 5 * took[1], took
