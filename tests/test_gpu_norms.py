"""The norm reduction of a pass over few, many and a ragged number of
workgroup partials: max|F(0)| as a one-step solve reports it equals the
maximum over the F(0) that rism3d_residual returns.  Both come from the same
kernels in FP64, so the two maxima agree to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


# partials per quantity: 48, 108, 648, 13824 (more than three rounds of 4096)
@pytest.mark.parametrize("n", [(32, 32, 32), (48, 48, 48), (96, 64, 96), (192, 192, 192)])
def test_max_residual_over_partials(n, chi_w):
    print("case norms", n, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    s = {"N": n[0], "nx": n[0], "ny": n[1], "nz": n[2], "sx": 0.3 * n[0], "sy": 0.3 * n[1],
         "sz": 0.3 * n[2], "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": "KH", "norm-tol": 1e-12, "max-iter": 1}
    sol = S.solute(1, n=5)
    out = R.hnc3d_run_solute(sol, W, s, chi=chi_w)
    r = R.residual(sol, W, s, chi_w, np.zeros((3, n[2], n[1], n[0])))
    assert out["iterations"] == 1
    assert out["residual"] == np.max(np.abs(r))
