"""Problems that the J-free kernels take by tiles (no symmetry orbits: a degree above 6, here the input line
"8 2"): fits and raw rows against the oracle (mrqmin.c, mrqcof.c:16-148, bright.c:14-126), the no-allocation
entry point, and batches that hold such problems beside problems with orbits.  Every fit of a batch equals
ps_fit_batch's bit for bit, in whichever form that takes it: short batches, whose fits with orbits are
spread, and long ones, which drain the queue.

Tolerances against the oracle: those of test_gpu_cholesky.py (1e-9 after three iterations) and
test_gpu_orbits.py (model values 1e-13, Jacobian entries 1e-12 of the row's largest)."""
import numpy as np
import pytest

from periodsearch_amd import FIT_DTYPE, PS_KERNEL_JFREE, Batch, PeriodSearch
from tests import oracle_binding as ob
from tests.test_gpu_orbits import problem, vectors
from tests.test_zz_no_alloc import noalloc

pytestmark = pytest.mark.gpu

STOP = 3


def text_of(lmax, mmax, *rest, **kw):
    lines = problem(lmax, mmax, *rest, **kw).split("\n")
    lines[10] = str(STOP)
    return "\n".join(lines)


def prepared(text):
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    return ps


def same(a, b, what):
    for k in FIT_DTYPE.names:
        assert np.array_equal(a[k], b[k], equal_nan=True), (what, k)


@pytest.mark.parametrize("lmax,mmax,nrows,dense,points,sparse,cl_free", [
    (8, 2, 6, 3, 50, 400, False), (8, 2, 5, 2, 64, 300, True), (7, 1, 8, 1, 127, 500, False)])
def test_tile_form_matches_oracle(lmax, mmax, nrows, dense, points, sparse, cl_free):
    text = text_of(lmax, mmax, nrows, dense, points, sparse, cl_free)
    orc = ob.OracleCtx.from_text(text)
    ps = prepared(text)
    try:
        conw = ps.info()["conw_r0"]
        orc.set_conw(conw)
        pole = np.array([1, 4, 8], np.int32)
        freq = ps.freq(np.array([1, 2, 3]))
        got = ps.fit_batch(freq, pole, conw)
        for i in range(3):
            ref = orc.fit(orc.freq(i + 1), int(pole[i]))
            assert got["niter"][i] == ref["niter"] == STOP and got["nsolve_fail"][i] == 0
            for k, rk in (("dev", "dev_new"), ("chisq", "chisq"), ("prd", "prd"), ("totarea", "totarea")):
                assert abs(got[k][i] - ref[rk]) <= 1e-9 * abs(ref[rk]), (i, k)
        same(noalloc(ps, freq, pole, conw), got, "noalloc")
        vecs = vectors(orc)
        raw = ps.eval(vecs, conw, raw=True)
        arr = ps.input_arrays()
        n = len(arr["tim"])
        for v, a in enumerate(vecs):
            for p in (0, n // 3, n - 1):
                br, dy = orc.bright(a, arr["ee"][p], arr["ee0"][p], arr["tim"][p])
                assert abs(raw["ymod"][v, p] - br) <= 1e-13 * abs(br), p
                assert np.abs(raw["dyda"][v, p] - dy).max() <= 1e-12 * np.abs(dy).max(), p
    finally:
        ps.close()


@pytest.mark.parametrize("reps", [1, 40])  # 70 fits, and more than the queue has workgroups
def test_batch_of_both_forms_matches_single_fits(reps):
    texts = [text_of(3, 3, 5, 3, 40, 300), text_of(8, 2, 4, 2, 50, 300), text_of(6, 6, 6, 2, 60, 200),
             text_of(8, 2, 4, 1, 50, 300, cl_free=True), text_of(4, 4, 4, 2, 30, 400, cl_free=True)]
    searches = [prepared(t) for t in texts]
    try:
        conw = np.array([s.info()["conw_r0"] for s in searches])
        prob = np.tile(np.repeat(np.arange(len(searches)), [10, 20, 10, 10, 20]), reps)
        pole = np.arange(len(prob)) % 10 + 1
        freq = np.array([searches[p].freq(1 + i % 7) for i, p in enumerate(prob)])
        with Batch(searches) as b:
            got = b.run(conw, prob, freq, pole)
            same(b.run(conw, prob, freq, pole), got, "the kept graph")
            few = np.flatnonzero(prob != 1)[:30]  # other counts, then the first ones again
            same(b.run(conw, prob[few], freq[few], pole[few]), got[few], "other counts")
            same(b.run(conw, prob, freq, pole), got, "again")
        for i, s in enumerate(searches):
            sel = prob == i
            same(got[sel], s.fit_batch(freq[sel], pole[sel], conw[i]), i)
    finally:
        for s in searches:
            s.close()
