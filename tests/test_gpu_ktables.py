"""The k tables are held for ky <= N1/2 and kz <= N2/2 and read at mirrored
rows and planes; a 3D susceptibility from outside is held whole.  The same
chi(|k|) both ways: as the 1D table, and tabulated here on the 3D k grid.

The two solves differ in the rounding of one interpolation and stop at an FP64
max|F| <= 1e-10 around a neutral solute: mu bar 1e-8, g bar 1e-7."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NRAD, RMAX = 512, 40.0


def _chi(m):
    """A smooth chi_ij(k), delta_ij at large k."""
    k = (np.arange(NRAD) + 0.5) * np.pi / RMAX
    out = np.zeros((m, m, NRAD))
    for i in range(m):
        for j in range(m):
            a = 0.5 + 0.1 * (i + j)
            out[i, j] = (i == j) + (-1.0) ** (i + j) * 0.3 / (1 + abs(i - j)) * \
                np.exp(-a * k * k) * np.cos(k * (1 + abs(i - j)))
    return out


def _table3(chi, N, L):
    """chi - delta on the half-complex grid, interpolated as the 1D lookup does
    (central differences, one-sided at the ends of the index range)."""
    m = chi.shape[0]
    dk = [2 * np.pi / v for v in L]
    kx = np.arange(N[0] // 2 + 1) * dk[0]
    ky, kz = (np.fft.fftfreq(n, 1.0 / n) * d for n, d in ((N[1], dk[1]), (N[2], dk[2])))
    k = np.sqrt(kx[None, None, :] ** 2 + ky[None, :, None] ** 2 + kz[:, None, None] ** 2)
    x = k / (np.pi / RMAX) - 0.5
    i = np.clip((x + 0.5).astype(int), 0, NRAD - 1)
    ip = np.where(i < NRAD - 2, i + 1, i)
    im = np.where(i > 1, i - 1, i)
    out = []
    for a in range(m):
        for b in range(a + 1):
            tab = chi[a, b] - (a == b)
            out.append(tab[i] + (tab[ip] - tab[im]) / (ip - im) * (x - i))
    return np.stack(out)


# 2 and 4 sites: the LDS form of the z pass; 3 and 5: the register forms; xy
# planes (N0 = N1) and rows; a Nyquist column in blocks of its own and in a tile
@pytest.mark.parametrize("m,N,prec", [
    (2, (48, 32, 64), "fp64"), (4, (32, 32, 48), "mixed"),
    (3, (32, 48, 64), "fp64"), (3, (64, 64, 32), "fp64"), (3, (64, 48, 32), "mixed"),
    (3, (96, 32, 48), "mixed"), (5, (64, 64, 48), "mixed"), (5, (48, 64, 32), "fp64")])
def test_mirrored_tables_against_whole(m, N, prec):
    print("case ktables", m, N, prec, flush=True)
    from bgy3d_amd import rism3d as R
    from bgy3d_amd import synthetic as S
    L = [0.3 * n for n in N]
    solvent = [("X%d" % i, (0.4 * i, 0.0, 0.1 * i), 2.6 + 0.2 * i, 0.12,
                0.2 * (-1) ** i if i < m // 2 * 2 else 0.0) for i in range(m)]
    s = {"N": max(N), "L": max(L) / 2, **dict(zip(("nx", "ny", "nz"), N)),
         **dict(zip(("sx", "sy", "sz"), L)), "rho": 0.02, "beta": 1.6889, "rmax": RMAX,
         "nrad": NRAD, "closure": "KH", "norm-tol": 1e-10, "mixed-tol": 1e-10, "polish-iters": 0,
         "max-iter": 1000, "precision": prec, "no-renorm": True}
    chi = _chi(m)
    sol = S.solute(2, n=4, net=0)
    a = R.hnc3d_run_solute(sol, solvent, s, chi=chi)
    b = R.hnc3d_run_solute(sol, solvent, s, chi3d=_table3(chi, N, L))
    assert a["status"] == "OK" and b["status"] == "OK"
    assert abs(a["free-energy"] - b["free-energy"]) < 1e-8
    assert np.max(np.abs(a["GUV"] - b["GUV"])) < 1e-7
