"""The tail launches (few particles, several lanes to a particle) and the
hand-on from the throughput launch, against gs_run_plain_noalloc, which runs
every particle in the throughput kernel from start to end: identical spectra,
bit for bit, at the edges of the particle counts where lanes per particle and
launches change."""
import pytest

from geliosphere_amd import abi

pytestmark = pytest.mark.gpu

MODELS = (abi.MODEL_1D_FP, abi.MODEL_1D_BP, abi.MODEL_2D_SOLARPROP, abi.MODEL_2D_GELIOSPHERE)
# 1 wave holds 64 particles, 65,536 lanes are one wave per SIMD: 64 lanes per
# particle up to 1024 particles, one lane above 32,768, a throughput launch
# first above 65,536
COUNTS = (1, 63, 1024, 1025, 32_769, 65_536, 65_537, 300_001)


def params(model, n, **over):
    kw = dict(N=n, seed=41 + n, r_inj=60.0, T_min=0.3, dt=500.0, first=7)
    kw.update(over)
    return abi.make_params(model, **kw)


@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("n", COUNTS)
def test_tail_equals_throughput_kernel(engine, model, n):
    p = params(model, n)
    print("tail vs throughput:", abi.MODEL_NAMES[model], n, flush=True)
    got, _, _ = engine.run_plain(p)
    assert bytes(got) == bytes(engine.run_plain_noalloc(p))
    assert got.n_particles == n


@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("max_steps", (1, 6, 8, 2051))
def test_step_cap_inside_a_cycle(engine, model, max_steps):
    """Caps that are and are not whole cycles, in both kernels."""
    p = params(model, 3000, r_inj=1.0, T_min=0.01, max_steps=max_steps)
    got, _, _ = engine.run_plain(p)
    ref = engine.run_plain_noalloc(p)
    assert bytes(got) == bytes(ref)
    assert got.n_step_cap > 0 and got.total_steps <= 3000 * max_steps


@pytest.mark.parametrize("model", MODELS)
@pytest.mark.parametrize("n", (500, 3000, 6000, 10_000, 20_000))   # 64, 16, 8, 4 and 2 lanes to a particle
@pytest.mark.parametrize("max_steps", (15, 33, 64, 1031))
def test_step_cap_between_two_tests(engine, model, n, max_steps):
    """Caps inside and at the ends of the cycles that are tested together."""
    p = params(model, n, r_inj=1.0, T_min=0.01, max_steps=max_steps)
    got, _, _ = engine.run_plain(p)
    assert bytes(got) == bytes(engine.run_plain_noalloc(p))
    assert got.n_step_cap > 0 and got.total_steps <= n * max_steps


@pytest.mark.parametrize("model", MODELS[1:])
def test_particles_that_end_at_once(engine, model):
    p = params(model, 500, r_inj=150.0)
    got, _, _ = engine.run_plain(p)
    assert bytes(got) == bytes(engine.run_plain_noalloc(p))
    assert got.n_particles == 500 and got.total_steps == 0


def test_batches_of_changing_counts(engine):
    """The same simulations with other particle counts: launches move between
    tail and throughput, and the slices of the shared buffers move with them."""
    for counts in ((900, 200_000, 5_000, 70_000), (150_000, 1_000, 90_000, 2_000), (1, 2, 3, 4)):
        sims = [params(m, n, seed=5 + i) for i, (m, n) in enumerate(zip(MODELS, counts))]
        outs = engine.run_batch(sims)
        for p, o in zip(sims, outs):
            assert bytes(o) == bytes(engine.run_plain(p)[0]), (abi.MODEL_NAMES[p.model], p.n_particles)
