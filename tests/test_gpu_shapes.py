"""The size-based launch shapes of the marching passes, and chunks that do
not divide the grid, give the bits of any other shape."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(n, prec, **shape):
    from mhit36_mixedp_amd import Solver
    with Solver(nx=n, phiflag=1, sigma=0.5, dt=2e-4, poisson_precision=prec) as s:
        if shape:
            s.set_tuning(**shape)
        s.init_random_velocity(5, kmax=min(4.0, n / 4), urms=1.0)
        s.init_drops(1, 1.2, 5)
        s.step(3)
        return [s.download_field(f) for f in range(1, 10)]


@pytest.mark.parametrize("n,prec,shape", [
    (8, 1, dict(ns_mz=3, ac_mz=5)),
    (12, 0, dict(ns_mz=12, ac_mz=7)),
    (32, 1, dict(ns_my=16, ac_my=16, ns_mz=32, ac_mz=32)),
    (48, 0, dict(ns_mz=5, ac_mz=11)),
    (64, 1, dict(ns_my=16, ac_my=16, ns_mz=13, ac_mz=31)),
    (96, 0, dict(ns_my=8, ac_my=8, ns_mz=25, ac_mz=17)),
    (128, 1, dict(ac_my=16, ns_mz=37, ac_mz=128)),
    (192, 0, dict(ac_my=16, ns_mz=24, ac_mz=24)),
])
def test_default_shapes_against_others(n, prec, shape):
    print(f"[shapes] n={n} prec={prec} {shape}", flush=True)
    for f, (a, b) in enumerate(zip(_run(n, prec), _run(n, prec, **shape)), start=1):
        assert np.array_equal(a, b), f
