"""The z chunks of the fused passes that a context reports or is given are
the ones that its launches take."""
import pytest

pytestmark = pytest.mark.gpu


def _pass_ms(s, steps=20):
    s.step(2)
    s.profile_enable()
    s.step(steps)
    rows = {r["stage"]: r["ms"] / r["calls"] for r in s.profile()}
    s.profile_enable(False)
    return rows["ns_ab2"], rows["acdi"]


@pytest.mark.parametrize("n", [48, 64])
def test_a_set_chunk_is_launched(n):
    """A whole column per workgroup leaves all but a few CUs idle (6 or 8
    tiles) and marches n planes instead of the default 2: more than ten times
    the time of the pass (a plane takes as long either way), of which a factor
    of two is asked for."""
    from mhit36_mixedp_amd import Solver
    print(f"[chunks] n={n}", flush=True)
    with Solver(nx=n, phiflag=1, sigma=0.5, dt=2e-4, poisson_precision=1) as s:
        s.init_random_velocity(5, kmax=4.0, urms=1.0)
        s.init_drops(1, 0.8, 5)
        short = _pass_ms(s)
        s.set_tuning(ns_mz=n, ac_mz=n)
        whole = _pass_ms(s)
        print(short, whole, flush=True)
        assert whole[0] > 2.0 * short[0] and whole[1] > 2.0 * short[1]
        assert s.tuning()["ns_mz"] == n and s.tuning()["ac_mz"] == n


def test_ensemble_reports_the_chunks_it_launches():
    """16 boxes each of 64^3, 96^3 and 128^3, every other one with drops: each
    launch (the boxes of one size and phase flag) reports a chunk with which it
    has a workgroup for nearly every CU by itself.  The CU count is taken from
    a 128^3 box alone, whose NS launch is one workgroup per CU (256)."""
    from mhit36_mixedp_amd import Ensemble, Solver, default_params
    print("[chunks] ensemble of 48", flush=True)
    sizes = [64] * 16 + [96] * 16 + [128] * 16
    cols = {8: 64, 16: 64, 32: 32, 10: 96}
    with Solver(nx=128) as s:
        t = s.tuning()
        cus = -(-128 // cols[t["ns_my"]]) * -(-128 // t["ns_my"]) * -(-128 // t["ns_mz"])
    with Ensemble([default_params(nx=n, phiflag=i % 2, sigma=0.5, dt=2e-4, poisson_precision=1)
                   for i, n in enumerate(sizes)]) as ens:
        for n in (64, 96, 128):
            for phase in (0, 1):
                group = [b.tuning() for b in ens.boxes if b.n == n and b.params.phiflag == phase]
                for mz, my in (("ns_mz", "ns_my"), ("ac_mz", "ac_my")):
                    t = group[0]
                    tiles = -(-n // cols[t[my]]) * -(-n // t[my]) * len(group)
                    print(n, phase, mz, t[mz], tiles * -(-n // t[mz]), flush=True)
                    assert all(g[mz] == t[mz] for g in group)
                    assert t[mz] == 1 or tiles * -(-n // t[mz]) >= 0.8 * cus


@pytest.mark.parametrize("n,prec", [(128, 1), (192, 0)])
def test_both_passes_share_a_shape_above_64(n, prec):
    """Above 64^3 the ACDI pass has the tiles and chunks of the NS pass by
    default, and the bits of 64 x 8 tiles."""
    import numpy as np
    from mhit36_mixedp_amd import Solver
    print(f"[chunks] shared shape n={n}", flush=True)
    phi = []
    for shape in ({}, dict(ac_my=8, ac_mz=19)):
        with Solver(nx=n, phiflag=1, sigma=0.5, dt=2e-4, poisson_precision=prec) as s:
            t = s.tuning()
            assert t["ac_my"] == t["ns_my"] == 16 and t["ac_mz"] == t["ns_mz"]
            if shape:
                s.set_tuning(**shape)
            s.init_random_velocity(5, kmax=4.0, urms=1.0)
            s.init_drops(1, 1.2, 5)
            s.step(3)
            phi.append((s.download_field(5), s.download_field(9)))
    for a, b in zip(*phi):
        assert np.array_equal(a, b)
