"""Fits and evaluations spread over many workgroups (periodsearch_amd/csrc/ps_spread.h) against the
one-workgroup form of the same kernels, bit for bit: the same fits as a full round of the resident
workgroups (which one workgroup each runs) and as short lists (which are spread), the last fits past a full
round, fixed and convergence stops, a damped system singular at every step, lists in several pieces, and
batches of uneven problems.  The per-fit body is period_search_BOINC.cpp:817-921 with mrqmin.c."""
import numpy as np
import pytest

from periodsearch_amd import FIT_DTYPE, PS_KERNEL_JFREE, Batch, PeriodSearch, synth

pytestmark = pytest.mark.gpu

SPECS = {
    "one_pass": synth.config0(n_dense=2, dense_points=30, stop_condition=7),
    "production": synth.config1(stop_condition=5),
    "convergence": synth.config0(stop_condition=0.01, n_iter_min=3),
    "lambert": synth.config0(seed=25, fit_lmax=5, cl_free=True, n_dense=4, dense_points=30, stop_condition=20),
    "singular": synth.config0(phase=(0.0, 0.1, -0.5), stop_condition=40),
}


def same(a, b, what):
    for k in FIT_DTYPE.names:
        assert np.array_equal(a[k], b[k], equal_nan=True), (what, k)


@pytest.mark.parametrize("name", list(SPECS))
def test_short_lists_match_a_full_round(name):
    text, _ = synth.generate(SPECS[name])
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    try:
        info = ps.info()
        slots, conw = info["slots"], info["conw_r0"]
        n = 1 + np.arange(slots) // 10 % info["nmax"]
        freq, pole = ps.freq(n), 1 + np.arange(slots) % 10
        full = ps.fit_batch(freq, pole, conw)
        for m in (1, 10, 100, slots // 2 + 1):
            same(ps.fit_batch(freq[:m], pole[:m], conw), full[:m], m)
        more = ps.fit_batch(np.append(freq, freq[:21]), np.append(pole, pole[:21]), conw)
        same(more, np.append(full, full[:21]), "past a round")
    finally:
        ps.close()


def test_lists_in_several_pieces():
    text, _ = synth.generate(synth.config3(stop_condition=2))
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    try:
        info = ps.info()
        slots, conw = info["slots"], info["conw_r0"]
        freq, pole = ps.freq(1 + np.arange(slots) // 10), 1 + np.arange(slots) % 10
        full = ps.fit_batch(freq, pole, conw)
        m = slots // 2
        same(ps.fit_batch(freq[:m], pole[:m], conw), full[:m], m)
    finally:
        ps.close()


@pytest.mark.parametrize("name", ["production", "lambert"])
def test_evaluations_match_a_full_round(name):
    text, _ = synth.generate(SPECS[name])
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    try:
        info = ps.info()
        vecs = synth.config2_vectors(ps, info["slots"])
        full = ps.eval(vecs, info["conw_r0"])
        for m in (1, 33, info["slots"] // 2 + 1):
            got = ps.eval(vecs[:m], info["conw_r0"])
            for k in ("alpha", "beta", "chisq"):
                assert np.array_equal(got[k], full[k][:m]), (m, k)
    finally:
        ps.close()


def test_small_batch_of_uneven_problems_matches_single_fits():
    specs = [SPECS["production"], SPECS["one_pass"], SPECS["lambert"], SPECS["convergence"],
             synth.config3(n_sparse=900, stop_condition=4)]
    searches = [PeriodSearch.from_text(synth.generate(s)[0]).prepare(device=0) for s in specs]
    try:
        conw = np.array([s.info()["conw_r0"] for s in searches])
        prob = np.repeat(np.arange(len(searches)), 10)
        freq = np.concatenate([s.freq(np.full(10, 2)) for s in searches])
        pole = np.tile(np.arange(1, 11), len(searches))
        with Batch(searches) as b:
            got = b.run(conw, prob, freq, pole)
            same(b.run(conw, prob, freq, pole), got, "again")
        for i, s in enumerate(searches):
            sel = prob == i
            same(got[sel], s.fit_batch(freq[sel], pole[sel], conw[i]), i)
    finally:
        for s in searches:
            s.close()
