"""Which lists are spread over many workgroups (spread_pays, spread_rest in periodsearch_amd/csrc/ps_device.hip):
where the form gains, and not where it costs more than it gives -- one pass (nothing to spread), few passes
to many fits, and fits that may stop early past a round or in several pieces.  The results are the same bits
in either form (test_gpu_spread.py)."""
import ctypes as C

import numpy as np
import pytest

from periodsearch_amd import FIT_DTYPE, PS_KERNEL_JFREE, Batch, PeriodSearch, lib, synth
from tests.test_gpu_orbits import problem

pytestmark = pytest.mark.gpu


def passes(lmax, nrows, npass, stop=2):
    """One lightcurve of 64 points and calibrated points to fill npass passes of 128."""
    text = problem(lmax, lmax, nrows, 1, 64, 128 * npass - 67)
    lines = text.split("\n")
    lines[10] = str(stop)
    return "\n".join(lines)


def spread(ps):
    fn = lib().ps_test_spread
    fn.argtypes, fn.restype = [C.c_void_p], C.c_int
    return fn(ps._handle())


def prepared(text):
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    return ps


@pytest.mark.parametrize("lmax,nrows,npass,stop,expect", [
    # {fits: spread}; "r": a round of the resident workgroups (two to a CU)
    (2, 4, 1, 2, {"10": 0, "250": 0, "r+20": 0}),
    (2, 4, 2, 2, {"10": 0}),
    (6, 6, 2, 2, {"10": 10, "200": 0}),
    (6, 6, 4, 2, {"10": 10, "100": 100, "200": 0, "280": 0, "r+10": 10, "r+200": 0}),
    (6, 8, 10, 2, {"10": 10, "200": 200, "280": 280, "300": 0, "r": 0}),
    (6, 6, 10, 0.5, {"10": 10, "200": 200, "r+20": 0}),  # may stop early
    (3, 4, 40, 0.5, {"200": 200, "280": 0}),               # 280 fits are two pieces
    (3, 4, 40, 2, {"280": 280}),
])
def test_fits(lmax, nrows, npass, stop, expect):
    ps = prepared(passes(lmax, nrows, npass, stop))
    try:
        info = ps.info()
        slots = info["slots"]
        assert slots == 512, "the numbers are for two workgroups on each of 256 CUs"
        for what, want in expect.items():
            n = sum(slots if w == "r" else int(w) for w in what.split("+"))
            ps.fit_batch(ps.freq(1 + np.arange(n) // 10), 1 + np.arange(n) % 10, info["conw_r0"])
            assert spread(ps) == want, (what, spread(ps))
    finally:
        ps.close()


@pytest.mark.parametrize("lmax,nrows,npass,expect", [
    (2, 4, 1, {1: 0, 200: 0}), (3, 6, 2, {1: 0}), (3, 6, 6, {1: 1, 200: 0}), (6, 6, 3, {1: 1}),
    (6, 6, 4, {10: 10, 200: 0}), (6, 8, 20, {16: 16, 200: 200, 300: 0})])
def test_evaluations(lmax, nrows, npass, expect):
    ps = prepared(passes(lmax, nrows, npass))
    try:
        info = ps.info()
        a = np.zeros(info["ma"])
        nc = info["ncoef"]
        a[:nc], a[nc] = ps.geometry()["cg_first"], 1.0
        a[nc + 2] = 2 * np.pi * 24 * ps.freq(1)
        a[nc + 3:] = 0.5, 0.1, -0.5, -2.0, 1.0
        for n, want in expect.items():
            ps.eval(np.tile(a, (n, 1)), info["conw_r0"])
            assert spread(ps) == want, (n, spread(ps))
    finally:
        ps.close()


def test_the_shapes_compared_bit_for_bit_are_spread():
    """The short lists of test_gpu_spread.py that stand for the spread form are in it."""
    for spec in (synth.config1(stop_condition=5), synth.config0(stop_condition=0.01, n_iter_min=3)):
        ps = prepared(synth.generate(spec)[0])
        try:
            info = ps.info()
            n = info["slots"]
            freq, pole = ps.freq(1 + np.arange(n) // 10 % info["nmax"]), 1 + np.arange(n) % 10
            full = ps.fit_batch(freq, pole, info["conw_r0"])
            assert spread(ps) == 0
            for m in (1, 10, 100):
                got = ps.fit_batch(freq[:m], pole[:m], info["conw_r0"])
                assert spread(ps) == m
                for k in FIT_DTYPE.names:
                    assert np.array_equal(got[k], full[k][:m], equal_nan=True), (m, k)
        finally:
            ps.close()


def test_fits_of_no_iteration_evaluate_nothing():
    """Stop 1 with a minimum of 0: the driver's loop (period_search_BOINC.cpp:868-872) does not run."""
    text, _ = synth.generate(synth.config1(stop_condition=1, n_iter_min=0))
    ps = prepared(text)
    try:
        conw = ps.info()["conw_r0"]
        freq, pole = ps.freq(np.full(10, 2)), np.arange(1, 11)
        with Batch([ps]) as b:
            lists = ps.fit_batch(freq, pole, conw), b.run([conw], np.zeros(10), freq, pole)
        for got in lists:
            for k in ("niter", "nsolve_fail", "chisq", "dev", "dark"):
                assert (got[k] == 0).all(), (k, got[k])
    finally:
        ps.close()


@pytest.mark.parametrize("off,expect", [(0.0, 10), (4e-15, 0)])
def test_only_rounding_passes_for_symmetry(off, expect):
    """A mesh whose normals are off the symmetry by more than rounding is not folded (by tiles nothing is spread)."""
    ps = PeriodSearch.from_text(passes(6, 6, 10))
    g = ps._geo.contents
    np.ctypeslib.as_array(g.nor, (g.nfac * 3,))[0] += off
    ps.prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    try:
        ps.fit_batch(ps.freq(np.full(10, 2)), np.arange(1, 11), ps.info()["conw_r0"])
        assert spread(ps) == expect
    finally:
        ps.close()
