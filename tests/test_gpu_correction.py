"""The correction of large boxes: its summation order with the FP32 Poisson,
bit by bit, and the shapes that only 384^3 takes."""
import numpy as np
import pytest

from test_gpu_shapes import _run

pytestmark = pytest.mark.gpu


def _mean_in_order(q, planes):
    """Mean of q[z][y][x] in the documented order: planes of a chunk bottom
    up per column, the 64 columns of a wave as a butterfly, the 8 rows of a
    tile first to last, tiles by 1024 interleaved runs, the runs as a tree."""
    n = q.shape[0]
    tiles = []
    for z0 in range(0, n, planes):
        s = np.zeros((n, n))
        for z in range(z0, min(z0 + planes, n)):
            s = s + q[z]
        s = s.reshape(n, n // 64, 64)
        for off in (32, 16, 8, 4, 2, 1):
            s = s[..., :off] + s[..., off:2 * off]
        s = s.reshape(n // 8, 8, n // 64)
        t = s[:, 0]
        for r in range(1, 8):
            t = t + s[:, r]
        tiles.append(t.reshape(-1))
    tiles = np.concatenate(tiles)
    runs = np.zeros(1024)
    for b in range(0, tiles.size, 1024):
        part = tiles[b:b + 1024]
        runs[:part.size] = runs[:part.size] + part
    for off in (512, 256, 128, 64, 32, 16, 8, 4, 2, 1):
        runs = runs[:off] + runs[off:2 * off]
    return float(runs[0]) / n / n / n


# 1024, 3456 and 16384 tiles; a component that does not vary along its own
# axis, alone and without viscosity and forcing, is left as it is by a step,
# so the corrected velocity is known exactly
@pytest.mark.parametrize("n,planes,comp", [(256, 32, 0), (256, 32, 1), (256, 32, 2), (384, 32, 0), (384, 32, 1),
                                           (384, 32, 2), (512, 16, 1)])
def test_mean_is_summed_in_the_fixed_order(n, planes, comp):
    from mhit36_mixedp_amd import Solver
    print(f"[correction] order n={n} component {comp}", flush=True)
    rng = np.random.default_rng(n + comp)
    shape = [n, n, n]
    shape[2 - comp] = 1
    q = np.ascontiguousarray(np.broadcast_to(rng.standard_normal(shape) + 0.375, (n, n, n)))
    with Solver(nx=n, poisson_precision=1, dt=1e-4, mu=0.0, f1=0.0, f2=0.0, f3=0.0) as s:
        s.upload_field(comp + 1, q)
        s.step(1)
        d = s.scalars()
        left = s.download_field(comp + 1)
    mean = _mean_in_order(q, planes)
    assert d[("umean", "vmean", "wmean")[comp]] == mean
    assert np.array_equal(left, q - mean)
    assert d["gumax"] == max(q.max() - mean, 0.0)


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32"])
def test_correction_mean_and_max_384(prec):
    """As at the sizes of test_gpu_shapes.py, with its bounds: the removed
    mean is the initial one, what is left has zero mean, and its maximum is
    the reported one to the last bit."""
    from mhit36_mixedp_amd import Solver
    n = 384
    print(f"[correction] mean and maximum n={n} prec={prec}", flush=True)
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


def test_chunks_that_do_not_divide_384():
    """55 planes by default (the last chunk has 54) against 48 and 96."""
    print("[correction] chunks at 384^3", flush=True)
    for f, (a, b) in enumerate(zip(_run(384, 1), _run(384, 1, ns_mz=96, ac_mz=48)), start=1):
        assert np.array_equal(a, b), f
