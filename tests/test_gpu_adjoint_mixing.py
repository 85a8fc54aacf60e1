"""The adjoint extrapolates at every pass, whatever the forward solve does: its
passes with periodic mixing on (the default) and off (RISM3D_PULAY=1) differ only by
what the two roots differ by.  Periodic mixing would take about a third of the
passes; the bar is 0.8 to 1.25 of them.  Gradients of one root repeat to 1e-10 of
the largest of a kind, the two roots leave them open by some 1e-9; bar 1e-7."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_adjoint_passes(prec, chi_w, monkeypatch):
    print("case adjoint mixing", prec, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    s = {"N": 48, "L": 7.2, "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": "KH", "norm-tol": 1e-11, "mixed-tol": 1e-11, "polish-iters": 0,
         "max-iter": 3000, "precision": prec}
    n, d = {}, {}
    for period in ("1", "3"):
        monkeypatch.setenv("RISM3D_PULAY", period)
        out = R.hnc3d_run_solute(S.solute(5, n=6, net=0), W, s, chi=chi_w, adjoint=True)
        assert out["status"] == "OK"
        n[period], d[period] = out["adjoint-iterations"], out["free-energy-dsite"]
    print("  adjoint passes", n, flush=True)
    assert 0.8 * n["1"] <= n["3"] <= 1.25 * n["1"]
    for cols in ((0, 1, 2), (3,), (4,), (5,)):
        a, b = d["1"][:, cols], d["3"][:, cols]
        assert np.max(np.abs(a - b)) <= 1e-7 * np.max(np.abs(a))
