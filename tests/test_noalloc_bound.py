"""Which problems rism3d_residual_noalloc admits: the fields, the spectra and
the whole k tables in both precisions have to fit its 96 MiB.  Six solvent sites
on 48 x 64 x 64 and on 48 x 32 x 128 points leave 1.7 MiB for the radial tables,
27 of them, so that 10260 radial points still fit and 10300 do not."""
import ctypes

import numpy as np
import pytest

GRIDS = [(48, 64, 64), (48, 32, 128)]
SOLVENT = [("X%d" % i, (0.4 * i, 0.0, 0.1 * i), 2.6 + 0.2 * i, 0.12, 0.2 * (-1) ** i)
           for i in range(6)]
SOLUTE = [("C", (0.4, -0.3, 0.2), 3.2, 0.15, 0.6), ("O", (-0.9, 0.6, -0.4), 3.0, 0.17, -0.8),
          ("H", (1.6, 0.3, 0.9), 1.0, 0.05, 0.2)]


def _problem(n, nrad):
    s = {"N": n[0], "L": 0.15 * n[0], **dict(zip(("nx", "ny", "nz"), n)),
         **{k: 0.3 * v for k, v in zip(("sx", "sy", "sz"), n)}, "rho": 0.02, "beta": 1.6889,
         "rmax": 60.0, "nrad": nrad, "closure": "KH"}
    k = (np.arange(nrad) + 0.5) * np.pi / 60.0
    chi = np.empty((6, 6, nrad))
    for i in range(6):
        for j in range(6):
            chi[i, j] = (i == j) + 0.1 * (-1.0) ** (i + j) * np.exp(-0.5 * k * k)
    t = 0.1 * np.random.default_rng(3).standard_normal((6, n[2], n[1], n[0]))
    return s, chi, t


def _status(n, nrad):
    from bgy3d_amd import rism3d as R
    lib = R.load()
    s, chi, t = _problem(n, nrad)
    pd, opt = R.problem_data(s), R.make_options(s)
    sv, su = R.make_sites(SOLVENT), R.make_sites(SOLUTE)
    r = np.empty_like(t)
    return lib.rism3d_residual_noalloc(ctypes.byref(pd), 6, sv, len(su), su, R._dptr(chi),
                                       ctypes.byref(opt), R._dptr(t), R._dptr(r))


@pytest.mark.parametrize("n", GRIDS)
def test_admitted_up_to_the_capacity(n):
    """Decided before any device work, so the same without a GPU (NO_DEVICE)."""
    from bgy3d_amd import rism3d as R
    for nrad in (2048, 10260):
        assert _status(n, nrad) in (R.OK, R.NO_DEVICE)
    assert _status(n, 10300) == R.NO_SCRATCH


@pytest.mark.gpu
@pytest.mark.parametrize("n", GRIDS)
def test_at_the_capacity_equals_residual(n):
    print("case noalloc at capacity", n, flush=True)
    from bgy3d_amd import rism3d as R
    s, chi, t = _problem(n, 10260)
    a = R.residual(SOLUTE, SOLVENT, s, chi, t, noalloc=True)
    b = R.residual(SOLUTE, SOLVENT, s, chi, t)
    assert np.all(np.isfinite(b)) and np.array_equal(a, b)
