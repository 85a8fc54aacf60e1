"""The FP64 chain on xy planes against the chain on rows.

A batch whose planes fill the chip runs on planes, one of its solutes alone
on rows (96 and 128 points per side), so both must reach the same root:
norm-tol 1e-10 leaves mu of these neutral solutes open by about 1e-9
kcal/mol (the change of mu with t is first order, of order rho P h^3 times
the residual), so they are compared to 1e-8."""
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


@pytest.mark.parametrize("N,B", [(96, 2), (96, 4), (128, 3)])
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


@pytest.mark.parametrize("N,B", [(32, 1), (48, 4)])
def test_small_fp32_planes_reach_the_fp64_root(N, B, chi_w):
    """FP32 planes of 32 and 48 points (the last kx tile of 48 is half full):
    a mixed solve to an FP64-checked 1e-10 and the FP64 solve to 1e-10 share
    their root, compared as above."""
    print(f"case planes fp32 {N}^3 batch {B}", flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    s = {"N": N, "L": 0.15 * N, "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": "KH", "norm-tol": 1e-10, "max-iter": 3000}
    sols = [S.solute(b, n=3, net=0) for b in range(B)]
    a = R.batch_solve(sols, W, s, chi_w)
    b = R.batch_solve(sols, W, dict(s, precision="mixed", **{"mixed-tol": 1e-10,
                                                              "polish-iters": 0}), chi_w)
    for x, y in zip(a, b):
        assert x["status"] == "OK" and y["status"] == "OK"
        assert y["iterations-fp32"] > 0
        assert abs(x["free-energy"] - y["free-energy"]) < 1e-8
