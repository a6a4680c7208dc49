"""The analysis passes at the edges of their launch shapes: spectrum rows
shorter and longer than a wave and truncated shell counts, diagnostics of
partial tiles and chunks, drop lists around the sizes the context keeps.

Tolerances: FP64 sums of N terms in another order than numpy's, 1e-12
relative as in test_gpu_spectra.py; FP32 transforms 1e-6 of the total."""
import numpy as np
import pytest

from test_gpu_drops import _compare
from test_gpu_spectra import _numpy_spectrum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [(8, 0), (12, 0), (96, 1), (128, 0), (192, 1)])
def test_spectrum_rows(n, prec):
    from mhit36_mixedp_amd import Solver
    print(f"[analysis] spectrum n={n} prec={prec}", flush=True)
    rng = np.random.default_rng(n)
    vel = [rng.standard_normal((n, n, n)) + 0.25 for _ in range(3)]     # a mean: the k = 0 shell
    with Solver(nx=n, poisson_precision=prec) as s:
        s.set_velocity(*vel)
        E = s.energy_spectrum()
        ref = _numpy_spectrum(*vel)
        assert E.shape == ref.shape
        assert np.max(np.abs(E - ref)) < (1e-12 if prec == 0 else 1e-6) * ref.sum()
        assert np.array_equal(E, s.energy_spectrum())                   # a fixed summation order
        few = np.full(4, np.nan)                                        # fewer bins than shells
        import ctypes
        rc = s.lib.mhit_energy_spectrum(s._h, 3, few.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), None)
        assert rc == 0 and np.array_equal(few[:3], E[:3]) and np.isnan(few[3])


@pytest.mark.parametrize("n", [8, 12, 24, 96, 256])
def test_diagnostics_tiles(n):
    from mhit36_mixedp_amd import Solver
    print(f"[analysis] diag n={n}", flush=True)
    rng = np.random.default_rng(n)
    u, v, w = (rng.standard_normal((n, n, n)) for _ in range(3))
    phi = rng.uniform(0, 1, (n, n, n))
    mu, dx = 0.01, 2 * np.pi / n
    mass = phi.sum() * dx ** 3
    with Solver(nx=n, phiflag=1, mu=mu, rho=1.0) as s:
        s.set_velocity(u, v, w)
        s.upload_field(5, phi)
        d = s.diag()
        phi[0, 0, n - 1] = np.nan
        s.upload_field(5, phi)
        assert s.diag()["nan_count"] == 1
    c = lambda f, ax: (np.roll(f, -1, ax) - np.roll(f, 1, ax)) * 0.5 / dx
    g = [[c(f, ax) for ax in (2, 1, 0)] for f in (u, v, w)]
    ss = sum(g[a][a] ** 2 for a in range(3)) + sum(0.5 * (g[a][b] + g[b][a]) ** 2
                                                   for a, b in ((0, 1), (0, 2), (1, 2)))
    div = sum(np.roll(f, -1, ax) - f for f, ax in ((u, 2), (v, 1), (w, 0))) / dx
    assert d["ke"] == pytest.approx(0.5 * np.mean(u * u + v * v + w * w), rel=1e-12)
    assert d["dissipation"] == pytest.approx(2 * mu * ss.mean(), rel=1e-12)
    assert d["maxdiv"] == pytest.approx(np.abs(div).max(), rel=1e-13)
    assert d["nan_count"] == 0
    assert d["phi_mass"] == pytest.approx(mass, rel=1e-12)


@pytest.mark.parametrize("n,step", [(64, 4), (64, 6), (96, 4)])     # 4096, 1331 and 13824 drops
def test_many_drops(oracle_mod, n, step):
    from mhit36_mixedp_amd import Solver
    print(f"[analysis] drops n={n} every {step}", flush=True)
    phi = np.zeros((n, n, n))
    phi[:n - 2:step, :n - 2:step, :n - 2:step] = 1.0
    rng = np.random.default_rng(n)
    u, v, w = (rng.standard_normal((n, n, n)) for _ in range(3))
    with Solver(nx=n, phiflag=1) as s:
        s.upload_field(5, phi)
        s.set_velocity(u, v, w)
        for _ in range(2):
            _compare(s.drop_stats(), oracle_mod.drop_stats(phi, u, v, w))


@pytest.mark.parametrize("conn", [6, 26])
@pytest.mark.parametrize("n,density", [(8, 0.4), (12, 0.35), (32, 0.9), (64, 0.31), (128, 0.32)])
def test_runs_across_waves(oracle_mod, n, density, conn):
    """Masked runs that start and end in different waves and rows, at n below,
    at and above a wave's 64 cells, near the site-percolation threshold."""
    from mhit36_mixedp_amd import Solver
    print(f"[analysis] runs n={n} density={density} conn={conn}", flush=True)
    rng = np.random.default_rng(n)
    phi = rng.uniform(0, 1, (n, n, n))
    phi[n // 2, n // 3, :] = 0.0              # a whole periodic row
    u, v, w = (rng.standard_normal((n, n, n)) for _ in range(3))
    with Solver(nx=n, phiflag=1) as s:
        s.upload_field(5, 1.0 - phi)
        s.set_velocity(u, v, w)
        _compare(s.drop_stats(threshold=1.0 - density, connectivity=conn),
                 oracle_mod.drop_stats(1.0 - phi, u, v, w, threshold=1.0 - density, connectivity=conn))
