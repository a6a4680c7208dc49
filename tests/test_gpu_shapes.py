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


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n", [8, 12, 24, 48, 64, 96, 128, 192, 256])
def test_correction_mean_and_max(n, prec):
    """The means that a step removes and its signed maximum, over tiles that
    overhang the grid, one and two levels of partial sums: the removed mean
    is the initial one (every term of the step sums to zero over the box up
    to rounding), the downloaded velocity has zero mean (sums of n^3 terms of
    order one in FP64) and its maximum is the reported one to the last bit."""
    from mhit36_mixedp_amd import Solver
    print(f"[shapes] correction n={n} prec={prec}", flush=True)
    rng = np.random.default_rng(n)
    with Solver(nx=n, poisson_precision=prec, dt=1e-4, mu=0.01) as s:
        start = [rng.standard_normal((n, n, n)) + m for m in (0.5, -0.25, 0.125)]
        s.set_velocity(*start)
        s.step(1)
        vel = s.velocity()
        d = s.scalars()
        for v, v0, m in zip(vel, start, ("umean", "vmean", "wmean")):
            assert abs(v.mean()) < 1e-13
            assert abs(d[m] - v0.mean()) < 1e-12
        assert d["gumax"] == max(v.max() for v in vel)


@pytest.mark.parametrize("boxes", [7, 8, 9])
def test_batched_correction_of_128(boxes):
    """Batches of 128^3 below, at and above the size from which the
    correction sweeps flat rows: the bits of each box stepped alone."""
    from mhit36_mixedp_amd import Ensemble, Solver, default_params
    print(f"[shapes] {boxes} x 128^3", flush=True)
    p = [default_params(nx=128, phiflag=0, poisson_precision=1, dt=2e-4, mu=0.006) for _ in range(boxes)]
    with Ensemble(p) as ens:
        for b, box in enumerate(ens.boxes):
            box.init_random_velocity(3 + b, kmax=4.0, urms=1.0)
        ens.step(3)
        for b in (0, boxes // 2, boxes - 1):
            with Solver(p[b]) as s:
                s.init_random_velocity(3 + b, kmax=4.0, urms=1.0)
                s.step(3)
                assert s.scalars() == ens.boxes[b].scalars(), b
                for f in range(1, 4):
                    assert np.array_equal(s.download_field(f), ens.boxes[b].download_field(f)), (b, f)
