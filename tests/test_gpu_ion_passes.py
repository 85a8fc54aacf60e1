"""Ions with HNC in mixed precision.  Above max|F| = 1, where every pass
extrapolates, the residual history is FP8 with and without periodic mixing, so
the two iterations are the same up to there; only from there do they differ.  An
iteration that overflows begins again along the closures and counts all its
passes, about twice as many.  Periodic mixing may take half as many passes again
as an extrapolation at every pass (RISM3D_PULAY=1), no more."""
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


@pytest.mark.parametrize("device", ["0", "1"])
@pytest.mark.parametrize("ion,N,h,depth", [("F-", 48, 0.25, 8), ("F-", 64, 0.35, 8),
                                           ("Br-", 48, 0.35, 8), ("Br-", 64, 0.35, 16),
                                           ("Li+", 32, 0.35, 12), ("Li+", 64, 0.35, 12)])
def test_ions_do_not_overflow(ion, N, h, depth, device, chi_w, monkeypatch):
    print("case ion passes", ion, N, h, depth, device, flush=True)
    from bgy3d_amd import rism3d as R
    s = {"N": N, "L": h * N / 2, "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": "HNC", "norm-tol": 1e-7, "mixed-tol": 1e-7, "polish-iters": 0,
         "max-iter": 1500, "precision": "mixed", "diis-depth": depth}
    monkeypatch.setenv("RISM3D_DEVICE_MDIIS", device)
    n, mu = {}, {}
    for period in ("1", "3"):
        monkeypatch.setenv("RISM3D_PULAY", period)
        out = R.hnc3d_run_solute(ion + ", JC08, SPC/E", W, s, chi=chi_w)
        assert out["status"] == "OK"
        n[period], mu[period] = out["iterations"], out["free-energy"]
    print("  passes", n, flush=True)
    assert n["3"] <= 1.5 * n["1"]
