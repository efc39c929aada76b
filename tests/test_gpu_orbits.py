"""Phase B of the J-free kernels by symmetry orbits of the facets (periodsearch_amd/csrc/ps_orbit.h): one
evaluation per parameter vector against the oracle's mrqcof and bright (mrqcof.c:16-148, bright.c:14-126) at
the sizes where the form can go wrong -- every degree and an order below the degree, the smallest and the
largest mesh, odd orbit counts, more orbits than one piece of the correction, passes of one point group
and of two, lightcurves that end on and beside a group's edge -- and with parameters fixed or the Lambert
weight free, which moves the row's columns; and the tile form, which a mesh without the symmetry keeps.

Tolerances: those of test_gpu_parity.py (normal equations 1e-11 of the matrix's size, chi2 1e-12, model
values 1e-13, Jacobian entries 1e-12 of the row's largest)."""
import numpy as np
import pytest

from periodsearch_amd import PS_KERNEL_JFREE, PS_KERNEL_LEGACY, PeriodSearch, synth
from tests import oracle_binding as ob

pytestmark = pytest.mark.gpu


def problem(lmax, mmax, nrows, dense, points, sparse, cl_free=False, fixed=()):
    text, _ = synth.generate(synth.config0(seed=77, fit_lmax=lmax, fit_nrows=nrows, n_dense=dense, dense_points=points,
                                           n_sparse=sparse, cl_free=cl_free))
    lines = text.split("\n")
    lines[4] = f"{lmax} {mmax}"
    for row in fixed:  # 0: the period, 6-8: the phase function
        f = lines[row].split()
        f[3 if row == 0 else 1] = "0"
        lines[row] = " ".join(f[:4 if row == 0 else 2])
    return "\n".join(lines)


def vectors(orc, n=3):
    rng = np.random.default_rng(5)
    out = []
    for pole in range(1, n + 1):
        a = orc.init_params(orc.freq(1), 3 * pole - 2)
        a[:orc.ncoef] += rng.normal(0, 0.05, orc.ncoef) / np.maximum(1, np.abs(np.arange(orc.ncoef)))
        out.append(a)
    return np.array(out)


CASES = [
    # lmax, mmax, nrows, dense, points, sparse
    (1, 1, 1, 2, 30, 0),       # one orbit: the second half of the orbits is empty
    (2, 1, 2, 1, 63, 1),       # one group, exactly full
    (3, 3, 3, 1, 64, 0),       # the convexity rows start the second group
    (3, 0, 6, 1, 65, 20),
    (4, 2, 5, 2, 64, 0),       # an odd number of orbits
    (4, 4, 4, 1, 128, 0),      # a lightcurve that fills a pass: the convexity rows alone in the next
    (5, 5, 7, 3, 41, 77),
    (6, 6, 6, 2, 50, 300),
    (6, 6, 8, 1, 127, 129),    # three pieces of the correction
    (6, 4, 1, 1, 20, 40),
]


@pytest.mark.parametrize("lmax,mmax,nrows,dense,points,sparse", CASES)
@pytest.mark.parametrize("cl_free,fixed", [(False, ()), (True, (0, 7)), (False, (0, 6, 7, 8))],
                         ids=["plain", "lambert", "fixed"])
def test_evaluations_match_oracle(lmax, mmax, nrows, dense, points, sparse, cl_free, fixed):
    text = problem(lmax, mmax, nrows, dense, points, sparse, cl_free, fixed)
    orc = ob.OracleCtx.from_text(text)
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    try:
        conw_r = ps.info()["conw_r0"]
        orc.set_conw(conw_r)
        vecs = vectors(orc)
        got = ps.eval(vecs, conw_r, raw=True)
        plain = ps.eval(vecs, conw_r)
        for k in ("alpha", "beta", "chisq"):
            assert np.array_equal(got[k], plain[k]), k
        arr = ps.input_arrays()
        n = len(arr["tim"])
        for v, a in enumerate(vecs):
            al, be, chi = orc.mrqcof(a)
            assert np.abs(got["alpha"][v] - al).max() <= 1e-11 * np.abs(al).max()
            assert np.abs(got["beta"][v] - be).max() <= 1e-11 * np.abs(be).max()
            assert abs(got["chisq"][v] - chi) <= 1e-12 * chi
            for p in sorted({0, n // 3, min(63, n - 1), min(64, n - 1), n - 1}):
                br, dy = orc.bright(a, arr["ee"][p], arr["ee0"][p], arr["tim"][p])
                assert abs(got["ymod"][v, p] - br) <= 1e-13 * abs(br), p
                assert np.abs(got["dyda"][v, p] - dy).max() <= 1e-12 * np.abs(dy).max(), p
    finally:
        ps.close()


@pytest.mark.parametrize("lmax,nrows", [(3, 6), (6, 8)])
def test_mesh_without_the_symmetry_keeps_the_tile_form(lmax, nrows):
    """A geometry the caller turned by a small angle: the J-free kernels agree with the
    materialised-Jacobian ones, which use no symmetry."""
    ps = PeriodSearch.from_text(problem(lmax, lmax, nrows, 3, 50, 40))
    g = ps._geo.contents
    nor = np.ctypeslib.as_array(g.nor, (g.nfac * 3,)).reshape(g.nfac, 3)
    c, s = np.cos(1e-3), np.sin(1e-3)
    nor[:] = nor @ np.array([[1, 0, 0], [0, c, -s], [0, s, c]]).T
    ps.prepare(device=0)
    try:
        conw_r = ps.info()["conw_r0"]
        orc = ob.OracleCtx.from_text(problem(lmax, lmax, nrows, 3, 50, 40))
        vecs = vectors(orc)
        got = {}
        for kernel in (PS_KERNEL_JFREE, PS_KERNEL_LEGACY):
            ps.set_kernel(kernel)
            got[kernel] = ps.eval(vecs, conw_r)
        a, b = got[PS_KERNEL_JFREE], got[PS_KERNEL_LEGACY]
        for k in ("alpha", "beta", "chisq"):
            assert np.abs(a[k] - b[k]).max() <= 1e-11 * np.abs(b[k]).max(), k
    finally:
        ps.close()
