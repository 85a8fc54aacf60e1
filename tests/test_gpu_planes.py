"""The FP64 chain on xy planes against the chain on rows.

A batch whose planes fill the chip runs on planes, one of its solutes alone
on rows (96 and 128 points per side), so both must reach the same root:
norm-tol 1e-10 leaves mu of these neutral solutes open by about 1e-9
kcal/mol (the change of mu with t is first order, of order rho P h^3 times
the residual), so they are compared to 1e-8."""
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


@pytest.mark.parametrize("N,B", [(96, 4), (128, 3)])
def test_batch_on_planes_equals_single_on_rows(N, B, chi_w):
    print(f"case planes fp64 {N}^3 batch {B}", flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    s = {"N": N, "L": 0.13 * N, "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": "KH", "norm-tol": 1e-10, "max-iter": 3000}
    sols = [S.solute(b, n=5, net=0) for b in range(B)]
    many = R.batch_solve(sols, W, s, chi_w)
    for b in (0, B - 1):
        one = R.hnc3d_run_solute(sols[b], W, s, chi=chi_w)
        d = abs(one["free-energy"] - many[b]["free-energy"])
        print(f"  solute {b} mu {one['free-energy']:.10f} |dmu| {d:.2e}", flush=True)
        assert one["status"] == "OK" and many[b]["status"] == "OK"
        assert d < 1e-8
