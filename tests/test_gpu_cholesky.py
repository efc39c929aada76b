"""The damped solve of the J-free kernels (cholesky_solve, periodsearch_amd/csrc/ps_fit2.h) at the system
sizes on both sides of its panels of 16 columns: short fits against the oracle, whose solve is the
reference's full-pivot Gauss-Jordan (gauss_errc.c:9-73).  Tolerance 1e-9 relative, the FP64 parity bar.
(Systems that it hands to the elimination: test_gpu_solver.py, and two thirds of the solves of the
config0 scan fixture.)"""
import numpy as np
import pytest

from periodsearch_amd import PS_KERNEL_JFREE, PeriodSearch
from tests import oracle_binding as ob
from tests.test_gpu_orbits import problem

pytestmark = pytest.mark.gpu

FIXED = (0, 6, 7, 8)  # the period and the phase function


@pytest.mark.parametrize("mfit,lmax,mmax,cl_free,fixed", [
    (6, 1, 1, False, FIXED), (15, 3, 1, False, (0,)), (16, 3, 2, False, FIXED), (18, 3, 3, False, FIXED),
    (31, 4, 4, False, ()), (32, 4, 4, True, ()), (33, 5, 3, False, (6, 7, 8)), (47, 6, 4, True, FIXED[:3]),
    (48, 6, 4, False, (7,)), (49, 6, 4, False, ()), (55, 6, 6, False, ()), (56, 6, 6, True, ())])
def test_short_fits_match_oracle(mfit, lmax, mmax, cl_free, fixed):
    text = problem(lmax, mmax, 5, 4, 40, 400, cl_free, fixed)
    lines = text.split("\n")
    lines[10] = "3"  # iterations
    text = "\n".join(lines)
    orc = ob.OracleCtx.from_text(text)
    ps = PeriodSearch.from_text(text).prepare(device=0)
    ps.set_kernel(PS_KERNEL_JFREE)
    try:
        info = ps.info()
        assert info["mfit"] == mfit
        orc.set_conw(info["conw_r0"])
        pole = np.array([1, 4, 8])
        got = ps.fit_batch(ps.freq(np.array([1, 2, 3])), pole, info["conw_r0"])
        for i in range(3):
            ref = orc.fit(orc.freq(i + 1), int(pole[i]))
            assert got["niter"][i] == ref["niter"] == 3 and got["nsolve_fail"][i] == 0
            for k, rk in (("dev", "dev_new"), ("chisq", "chisq"), ("prd", "prd"), ("totarea", "totarea")):
                assert abs(got[k][i] - ref[rk]) <= 1e-9 * abs(ref[rk]), (i, k)
    finally:
        ps.close()
