"""Periodic Pulay mixing (several Gram rows from one reading of the residual
history, plain steps between the extrapolations) against an extrapolation at
every pass (RISM3D_PULAY=1): the same root.

Both stop at an FP64 max|F| <= 1e-10.  The solutes are neutral, and a
residual of 1e-10 leaves their mu open by some 1e-9 kcal/mol; bar 1e-8.  The
adjoint stops at 1e-11 (FP64) or 1e-10 (mixed) of max|dmu/dt|, so its gradients
agree to about 1e-8 of the largest of a kind; bar 1e-6."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


def _settings(N, **kw):
    return dict({"N": N, "L": 0.15 * N, "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0,
                 "nrad": 1536, "closure": "KH", "norm-tol": 1e-10, "mixed-tol": 1e-10,
                 "polish-iters": 0, "max-iter": 3000}, **kw)


# histories of 5, 8, 9, 10, 11 and 16 entries (kernels for 8, 10 and 16), the
# FP32 phase with BF16 and FP8 residuals and with the full FP32 u history
@pytest.mark.parametrize("depth,prec,env", [
    (5, "fp64", {}), (8, "fp64", {}), (9, "fp64", {}), (11, "fp64", {}), (16, "fp64", {}),
    (5, "mixed", {}), (8, "mixed", {}), (10, "mixed", {}), (16, "mixed", {}),
    (8, "mixed", {"RISM3D_R_FP8": "1"}), (10, "mixed", {"RISM3D_U_DIFF": "0"}),
    (8, "mixed", {"RISM3D_R_BF16": "0"})])
def test_periodic_reaches_the_root_of_every_pass(depth, prec, env, chi_w, monkeypatch):
    print("case pulay", depth, prec, env, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    sols = [S.solute(b, n=4, net=0) for b in range(3)]
    s = _settings(48, precision=prec, **{"diis-depth": depth})
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    got = {}
    for period in ("1", "3"):
        monkeypatch.setenv("RISM3D_PULAY", period)
        got[period] = R.batch_solve(sols, W, s, chi_w, want_g=True)
    for a, b in zip(got["1"], got["3"]):
        assert a["status"] == "OK" and b["status"] == "OK"
        assert abs(a["free-energy"] - b["free-energy"]) < 1e-8
        assert np.max(np.abs(a["GUV"] - b["GUV"])) < 1e-7


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_periodic_adjoint(prec, chi_w, monkeypatch):
    print("case pulay adjoint", prec, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    got = {}
    for period in ("1", "3"):
        monkeypatch.setenv("RISM3D_PULAY", period)
        out = R.hnc3d_run_solute(S.solute(5, n=4), W, _settings(32, precision=prec), chi=chi_w,
                                 adjoint=True)
        assert out["status"] == "OK"
        got[period] = out["free-energy-dsite"]
    a, b = got["1"], got["3"]
    for cols in ((0, 1, 2), (3,), (4,), (5,)):
        assert np.max(np.abs(a[:, cols] - b[:, cols])) <= 1e-6 * np.max(np.abs(a[:, cols]))
