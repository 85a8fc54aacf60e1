"""The autotuner's trials: passes one after the other, without the host's wait
that a pass of a solve ends with.  A trial pass therefore takes no longer than a
pass of a solve (Picard, which reads no history); 1.1 leaves room for the
launches one by one.  The median over three small grids, where a wait between
trial passes showed most (36 us instead of 28, against 31 of a solve's pass)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
W = "water, PR-SPC/E"


def _settings(n2, **kw):
    return dict({"N": 32, "nz": n2, "L": 4.8, "sx": 9.6, "sy": 9.6, "sz": 0.3 * n2,
                 "rho": 0.0333295, "beta": 1.6889, "rmax": 40.0, "nrad": 1536, "closure": "KH",
                 "lambda": 0.02, "norm-tol": 1e-12, "snes-solver": "picard"}, **kw)


def test_trials_run_back_to_back(chi_w, tmp_path, monkeypatch):
    print("case tuner trials", flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    f = tmp_path / "tune.txt"
    monkeypatch.setenv("RISM3D_TUNE_FILE", str(f))
    sol = S.solute(2, n=4, net=0)
    ratio = []
    for n2 in (32, 48, 64):
        def seconds(k):
            best = np.inf
            for _ in range(4):
                t0 = time.perf_counter()
                out = R.hnc3d_run_solute(sol, W, _settings(n2, **{"max-iter": k}), chi=chi_w)
                best = min(best, time.perf_counter() - t0)
                assert out["iterations"] == k
            return best
        per_pass = (seconds(600) - seconds(100)) / 500
        R.hnc3d_run_solute(sol, W, _settings(n2, tune=1, **{"max-iter": 2}), chi=chi_w)
        trial = [float(ln.split()[-1]) for ln in f.read_text().split("\n")
                 if ln.startswith(f"32x32x{n2},m3,B1,fp64 ")][-1]
        print(f"  32x32x{n2}: trial {1e3 * trial:.1f} us, pass {1e6 * per_pass:.1f} us", flush=True)
        ratio.append(1e-3 * trial / per_pass)
    assert sorted(ratio)[1] <= 1.1


CHILD = """
import json, os
import numpy as np
from bgy3d_amd import rism3d as R
from bgy3d_amd import synthetic as S
s = json.loads(os.environ["CASE"])
chi = np.load(os.environ["CHI"])
R.profile_start()
out = R.hnc3d_run_solute(S.solute(2, n=4, net=0), "%s", s, chi=chi)
print(json.dumps({"kernels": sorted(R.profile_read()), "mu": out["free-energy"]}))
""" % W


def test_file_without_fp64_planes(chi_w, tmp_path):
    """A file written when FP64 had no xy planes has 0 for them: the solve stays
    on planes.  In a process of its own, as a file is read at the first tuning."""
    print("case tuner file", flush=True)
    import json
    import os
    import subprocess
    import sys
    np.save(tmp_path / "chi.npy", chi_w)
    f = tmp_path / "tune.txt"
    f.write_text("32x32x32,m3,B1,fp64 0 2 0 0 0.0350\n")
    s = _settings(32, tune=1, **{"max-iter": 3})
    env = dict(os.environ, CASE=json.dumps(s), CHI=str(tmp_path / "chi.npy"),
               RISM3D_TUNE_FILE=str(f))
    p = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True,
                       timeout=100)
    assert p.returncode == 0, p.stderr
    got = json.loads(p.stdout.strip().split("\n")[-1])
    assert "closure_r2c_xy<double>" in got["kernels"], got
    assert f.read_text().count("fp64") == 1  # the entry was used, nothing timed
