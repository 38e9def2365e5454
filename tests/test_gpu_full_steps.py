"""1D simulations without branch-free steps (no diffusion at all, or steps too wide):
kernels of their own, in tail launches, throughput launches and batches, with caps
inside and at the ends of cycles."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu

NONE = dict(K0_cm2s=0.0, T_min=0.05, r_inj=3.0)


def integers(s):
    return (s.n_particles, s.n_events, s.n_outside, s.total_steps, s.n_nan, s.n_step_cap, list(s.count))


# 64 lanes to a particle, 2, 1 and a throughput launch
@pytest.mark.parametrize("n", (1, 700, 20_000, 65_536, 70_001))
@pytest.mark.parametrize("max_steps", (1, 7, 8, 43, 2500))
def test_without_diffusion(engine, oracle, n, max_steps):
    p = abi.make_params(abi.MODEL_1D_BP, N=n, seed=5, first=3, max_steps=max_steps, **NONE)
    s = engine.run_plain(p)[0]
    rc, o, _, _ = oracle.run(p)
    assert rc == 0 and integers(s) == integers(o) and s.n_step_cap == n
    assert bytes(engine.run_plain_noalloc(p)) == bytes(s)


@pytest.mark.parametrize("max_steps", (3, 4, 400))
def test_wide_steps(engine, max_steps):
    """V dt = 1.6 AU, in launches of every kind and both counts of lanes."""
    kw = dict(seed=3, dt=6e5, K0_cm2s=5e22, max_steps=max_steps)
    whole = engine.run_plain(abi.make_params(abi.MODEL_1D_FP, N=200_000, **kw))[0]
    parts = [engine.run_plain(abi.make_params(abi.MODEL_1D_FP, N=n, first=at, **kw))[0]
             for at, n in ((0, 500), (500, 39_500), (40_000, 160_000))]
    from geliosphere_amd.engine import merge_spectra
    rc, merged = merge_spectra(parts)
    assert rc == 0 and bytes(merged) == bytes(whole)


def test_batches_of_both_kinds(engine):
    sims = []
    for i, n in enumerate((30_000, 45_000, 1, 0, 500, 66_000)):
        sims.append(abi.make_params(abi.MODEL_1D_BP, N=n, seed=20 + i, max_steps=300 + i, **NONE))
        sims.append(abi.make_params(abi.MODEL_1D_BP, N=n // 2, seed=40 + i, max_steps=3000, r_inj=60.0))
        sims.append(abi.make_params(abi.MODEL_1D_FP, N=n, seed=60 + i, dt=6e5 if i % 2 else 500.0))
    outs = engine.run_batch(sims)
    for p, o in zip(sims, outs):
        assert bytes(o) == bytes(engine.run_plain(p)[0]), (p.model, p.n_particles, p.K0)


def test_no_cycle_is_computed_twice(engine):
    """A step without diffusion against a branch-free one: 1.3 times as long (2.5 when
    the branch-free steps were taken as well and thrown away)."""
    def best(**kw):
        ms = []
        for k in range(4):
            engine.run_plain(abi.make_params(abi.MODEL_1D_BP, N=1_000_000, seed=k, max_steps=4000, **kw))
            ms.append(engine.last_stats().kernel_ms)
        return min(ms)
    with_k, without = best(r_inj=3.0, T_min=0.05), best(**NONE)
    assert without < 1.9 * with_k, (without, with_k)


def test_launches_of_changing_size(engine):
    """Chunks that are cut to fit a small event region and grow again: a launch
    without a hand-on after one with."""
    p = abi.make_params(abi.MODEL_1D_FP, N=200_000, seed=3, dt=6e5, K0_cm2s=5e22)
    whole = engine.run_plain(p)[0]
    assert whole.n_events > 1000
    engine.set_plain_limits(max_events=300)
    try:
        assert bytes(engine.run_plain(p)[0]) == bytes(whole)
    finally:
        engine.set_plain_limits()


def test_batches_of_more_groups_than_streams(engine):
    """Six groups: four models, and both 1D models without branch-free steps; in
    throughput launches (70,000 particles) and in tail launches."""
    for n in (35_000, 300):
        sims = []
        for i in range(2):
            sims.append(abi.make_params(abi.MODEL_1D_BP, N=n, seed=20 + i, max_steps=300 + i, **NONE))
            sims.append(abi.make_params(abi.MODEL_1D_FP, N=n, seed=40 + i, dt=6e5))
            for m in (abi.MODEL_1D_FP, abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP, abi.MODEL_2D_GELIOSPHERE):
                sims.append(abi.make_params(m, N=n + i, seed=60 + 10 * m + i, dt=500.0, r_inj=80.0, T_min=0.3))
        want = [bytes(engine.run_plain_noalloc(p)) for p in sims]
        for _ in range(3):   # the captured graph again
            assert [bytes(o) for o in engine.run_batch(sims)] == want
