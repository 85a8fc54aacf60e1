"""Where plain steps overshoot.  Periodic mixing begins at a small max|F| and
ends with the first restart, so that an iteration that converges with an
extrapolation at every pass (RISM3D_PULAY=1) still does, in about as many passes:
ions with HNC and PSE-4 (an iteration that overflows begins again along the
closures and counts its passes twice), and steps so long that plain steps diverge
by themselves.  Twice the passes at most; the same root, to 1e-6 kcal/mol at
max|F| <= 1e-9."""
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"
SPACE = [("I-", 48, 0.35, "HNC", 8, 0.8), ("I-", 64, 0.25, "PSE4", 8, 0.5),
         ("Br-", 32, 0.30, "HNC", 12, 0.5), ("Na+", 32, 0.35, "HNC", 8, 0.5),
         ("Cl-", 32, 0.30, "PSE4", 5, 0.3),
         (2, 48, 0.30, "KH", 8, 3.0), (2, 48, 0.30, "KH", 8, 4.0), (7, 48, 0.30, "KH", 8, 2.5),
         ("Cl-", 48, 0.30, "KH", 8, 3.0)]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("who,N,h,closure,depth,step", SPACE)
def test_converges_as_with_an_extrapolation_each_pass(who, N, h, closure, depth, step, prec,
                                                      chi_w, monkeypatch):
    print("case pulay guard", who, N, h, closure, depth, step, prec, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    sol = who + ", JC08, SPC/E" if isinstance(who, str) else S.solute(who, n=4, net=0)
    s = {"N": N, "L": h * N / 2, "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536,
         "closure": closure, "norm-tol": 1e-9, "mixed-tol": 1e-9, "polish-iters": 0,
         "max-iter": 3000, "precision": prec, "diis-depth": depth, "diis-step": step}
    out = {}
    for period in ("1", "3"):
        monkeypatch.setenv("RISM3D_PULAY", period)
        out[period] = R.hnc3d_run_solute(sol, W, s, chi=chi_w)
    a, b = out["1"], out["3"]
    print("  passes", a["iterations"], b["iterations"], flush=True)
    assert a["status"] == "OK" and b["status"] == "OK"
    assert b["iterations"] <= 2 * a["iterations"]
    assert abs(a["free-energy"] - b["free-energy"]) < 1e-6
