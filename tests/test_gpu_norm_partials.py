"""max|F(0)| as a one-step solve reports it equals the maximum over the F(0) of
rism3d_residual, to the bit, by the number of workgroup partials that the norm
reduction sums: on xy planes one per plane and site (3 x 32 = 96, 3 x 48 = 144), on
rows one per 64, 32, 16, 8 or 4 rows and site (N0 = 32, 48 to 64, 96 to 128, 192 to
256, 384): 48, 96, 1152 and 13824."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


@pytest.mark.parametrize("n,planes,partials", [
    ((32, 32, 32), 1, 96), ((48, 48, 48), 1, 144), ((32, 32, 32), 0, 48),
    ((48, 32, 32), 1, 96), ((96, 64, 96), 1, 1152), ((192, 192, 192), 1, 13824)])
def test_max_residual(n, planes, partials, chi_w, monkeypatch):
    print("case norm partials", n, planes, partials, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    monkeypatch.setenv("RISM3D_PLANES", str(planes))
    s = {"N": n[0], "nx": n[0], "ny": n[1], "nz": n[2], "sx": 0.3 * n[0], "sy": 0.3 * n[1],
         "sz": 0.3 * n[2], "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": "KH", "norm-tol": 1e-12, "max-iter": 1}
    rows = {32: 64, 48: 32, 96: 16, 192: 8}[n[0]]
    on_planes = planes and n[0] == n[1] and n[0] <= 64
    assert partials == 3 * (n[2] if on_planes else n[1] * n[2] // rows)
    sol = S.solute(1, n=5)
    R.profile_start()
    out = R.hnc3d_run_solute(sol, W, s, chi=chi_w)
    assert ("closure_r2c_xy<double>" in R.profile_read()) == bool(on_planes)
    r = R.residual(sol, W, s, chi_w, np.zeros((3, n[2], n[1], n[0])))
    assert out["iterations"] == 1
    assert out["residual"] == np.max(np.abs(r))
