"""Re-ordering in the middle of a run at the production size: moved tracers,
a nonzero velocity history and the graph of the swapped columns.  A tracer's
path does not depend on its place in the columns, so a run that re-orders
every five steps and one that never does give the same bits tracer by
tracer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_reorder_mid_run_at_full_size():
    from mhit36_mixedp_amd import Solver
    n, ntr = 512, 4_194_304
    print(f"[tracer re-order] n={n} tracers={ntr}, 12 steps", flush=True)
    out = {}
    with Solver(nx=n, phiflag=0, partflag=1, poisson_precision=1, dt=1e-3, mu=0.002) as s:
        for every in (5, 0):
            s.init_random_velocity(2024, kmax=8.0, urms=1.0)
            s.set_ab2_state(1.0, 0.0, 1.0)
            s.init_tracers_uniform(ntr, 2024)
            s.set_tuning(sort_every=every)
            s.step(1)
            first = s.download_tracers()["tag"]
            s.step(11)                      # every 5: again before steps 6 and 11
            out[every] = s.download_tracers()
            moved = not np.array_equal(first, out[every]["tag"])
            assert moved == (every == 5)    # tracers changed cells, and the order followed
        assert s.scalars()["cou"] > 0.1
    a, b = out[5], out[0]
    order_a, order_b = np.argsort(a["tag"]), np.argsort(b["tag"])
    for k in a:
        assert np.array_equal(a[k][order_a], b[k][order_b]), k
